"""The fused module of a plan compiles at the limits of a workgroup's LDS: the
most rows and the widest layers, long chunks (two points per workgroup where
they fit) and short ones, one and several outputs, a single hidden layer, and a
narrow layer beside a wide one."""
import pytest

from cpde_amd import hip, workloads as W


@pytest.mark.parametrize('variables,order,neurons,width', [
    (3, 5, [3, 256, 1], 8192),             # one hidden layer: no product
    (3, 5, [3, 224, 8], 8192),
    (3, 5, [3, 208, 208, 8], 8192),        # 56 rows: one point
    (3, 5, [3, 208, 208, 1], 8192),        # and two, just below 160 KB
    (2, 6, [2, 80, 256, 1], 8192),         # 28 rows, two points
    (2, 6, [2, 128, 240, 1], 8192),
    (2, 6, [2, 128, 256, 8], 1000),
])
def test_modules_at_the_lds_limit_compile(tmp_path, monkeypatch, variables, order, neurons, width):
    monkeypatch.setenv('CPDE_JIT_CACHE', str(tmp_path))
    hip.jit_prepare(W.full_schema(variables, order), neurons, width)
