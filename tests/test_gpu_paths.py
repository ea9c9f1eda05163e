"""Kernel variants at the sizes where their tiles end, against the FP64 oracle."""
import numpy as np
import pytest

from conftest import say
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [2, 3, 15, 16, 17, 63, 64, 65, 131])
@pytest.mark.parametrize("n", [65, 700])
def test_weighted_values_bitwise(ctx, n, t):
    """Edge weights and the FP64 recheck over series whose runs of 16 (bulk) and
    64 (short lists) time points end early, at odd lengths and aligned ones."""
    from pagani_amd import synth
    x = synth.bold(31 + t, n, t, 5)
    z64, _ = O.zscore(x)
    thr = 0.9 if t < 10 else 0.3
    for prec in (0, 1):
        say(f"weighted values n={n} t={t} prec={prec}")
        info = ctx.corr_build(x, n, t, thr, weighted=True, prec=prec)
        row, col, val = ctx.corr_csr(n, info.nnz, True)
        orow, ocol, oval = O.corr_csr_r(z64, thr, True)
        np.testing.assert_array_equal(row, orow)
        np.testing.assert_array_equal(col, ocol)
        np.testing.assert_array_equal(val.view(np.uint32), oval.view(np.uint32))
