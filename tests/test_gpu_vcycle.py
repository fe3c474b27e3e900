"""The V-cycle's launch forms on the GPU against the oracle's cycle: a level in
two launches (tiles with halos), the coarse end in one workgroup per slot, and
the kernels of one sweep each, at box sizes around the tiles' and the
workgroup's edges."""
import numpy as np
import pytest

import formoniq_amd as fa
from oracle import oracle as o

from _common import both

pytestmark = pytest.mark.gpu

# (d, n, k, relative, sweeps): two-launch levels from 13^3 and 46^2 vertices on (in 3D
# up to 256 workgroups: 16^3 with 10 slots and 24^3 with 5 have more), partial last
# tiles, odd grids whose coarse box overhangs, a whole cycle in one launch (the largest and
# one smaller; 1D below, at and beyond the 2,048 vertices of one workgroup), 4D (no tiles), one
# and three sweeps (no tiles; the iterates change buffers)
CASES = [(1, 300, 0, True, 2), (1, 900, 0, True, 2), (1, 2046, 0, True, 2), (1, 2047, 0, True, 2),
         (1, 2048, 0, True, 2), (1, 5000, 0, True, 2), (2, 44, 1, False, 2), (2, 45, 1, True, 2), (2, 66, 0, True, 2),
         (2, 97, 1, False, 2), (3, 11, 1, False, 2), (3, 12, 1, True, 2), (3, 13, 2, True, 2), (3, 15, 1, False, 2),
         (3, 16, 2, False, 2), (3, 24, 1, False, 2),
         (3, 17, 0, True, 2), (3, 26, 0, True, 2), (4, 4, 1, False, 2), (2, 50, 1, False, 3), (3, 12, 1, False, 1),
         (3, 13, 1, True, 3)]


@pytest.mark.parametrize("d,n,k,rel,sweeps", CASES)
def test_cycle_forms_match_the_oracle(d, n, k, rel, sweeps):
    """One block application (m = 1) in FP64 to 1e-10 of its largest entry and in
    FP32 to 1e-5, the bounds of the other application tests (sums of at most 31
    terms in another order). In 1D the FP32 result is held against A = hdif_gram(0)
    instead: each residual of a cycle is rounded to 2^-24 of |A||x| a term, and the
    coarse correction of its smooth part amplifies that by up to the condition of
    D^-1 A (4 n^2 / pi^2), which A takes back: |A e| <= 31 2^-24 max(|A||z|), below
    5e-5 of the largest |A z| on these grids (measured: 0.9 to 1.2 of the 31, 11
    with 300 cells, whose coarsest level of 149 unknowns has the largest dense
    inverse; a cycle off by half leaves 0.5)."""
    ocx, oL, gcx, geo, cells, coords = both(d, n, 0.05, seed=n)
    gc = fa.WhitneyComplex(geo, relative=rel)
    opts = dict(preconditioner=fa.PC_MULTIGRID, cheb_degree=1, mg_sweeps=sweeps)
    prob = fa.Problem(gc, k, fa.solve_opts(precision=fa.FP64, **opts))
    prob.assemble()
    ns, nu, nh = prob.sizes
    oc = o.WhitneyComplex(ocx, oL, relative=rel)
    r = np.sin(np.arange(ns + nu + nh) * 0.7 + 0.3)
    want = o.hx_block_preconditioner(oc, coords, k, n, nh, sweeps=sweeps, cheb_m=1)(r)
    scale = np.abs(want).max()
    got = prob.apply_preconditioner(r, precision=fa.FP64)
    assert np.abs(got - want).max() <= 1e-10 * scale, np.abs(got - want).max() / scale
    got32 = fa.Problem(gc, k, fa.solve_opts(**opts)).apply_preconditioner(r, precision=fa.FP64_PC32)
    if d == 1:
        A = oc.hdif_gram(k).to_scipy().tocsr()
        z = want[:nu]
        bound = 31 * 2.0**-24 * (abs(A) @ np.abs(z)).max()
        assert bound <= 5e-5 * np.abs(A @ z).max()
        assert np.abs(A @ (got32[:nu] - z)).max() <= bound
        assert np.abs(got32 - want).max() <= 1e-2 * scale
    else:
        assert np.abs(got32 - want).max() <= 1e-5 * scale, np.abs(got32 - want).max() / scale
    again = prob.apply_preconditioner(r, precision=fa.FP64)
    np.testing.assert_array_equal(again, got)
