"""Variants that the autotuner times: the vector-ALU kernel and the matrix-core
kernel at every degree, no variant twice."""
import pytest

from piclas_amd import autotune, stage


@pytest.mark.parametrize("N", range(1, 8))
def test_shape_function(N):
    c = autotune.candidates(N)
    assert {(x["use_graph"], x["sf_kernel"]) for x in c} == {(g, k) for g in (False, True) for k in (1, 2)}
    assert len({tuple(sorted(x.items())) for x in c}) == len(c)
    assert any(x["sf_persistent"] for x in c) == (N == 3)
    assert not any(x["sf_kernel"] == 1 and (x["sf_persistent"] or x["sf_shared_loads"]) for x in c)


def test_other_depositions():
    assert [x["use_graph"] for x in autotune.candidates(2, stage.DEPO_CVWM)] == [False, True]
