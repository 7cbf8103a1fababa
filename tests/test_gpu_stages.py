"""The fused integrator stages (tile kernels, nb = 2 and 4) against the separate
stage kernels the deterministic row kernel runs with, over band windows of every
width, k counts on both sides of a block of whole k points, and the terms of the
right-hand side.

Tolerance: the two paths differ in the order of FP64 sums of the scattering term
only, 1e-12 of the largest element of the result over a few steps."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from helpers import FS, random_energies, random_P, random_pairs, random_rho  # noqa: E402

from denmat_dynm_development_amd import _lib, scatt  # noqa: E402

pytestmark = pytest.mark.gpu


def _op(nb, nbd, nk, kernel, terms, seed):
    rng = np.random.default_rng(seed)
    b0 = (nbd - nb) // 2
    edm = random_energies(nk, nbd, rng)
    e = np.ascontiguousarray(edm[:, b0:b0 + nb])
    k1, k2 = random_pairs(nk, 3, rng, diag=True)
    P1, P2 = random_P(len(k1), nb, rng)
    op = scatt.ScatteringOperator(nk, nb, k1, k2, e, nk_full=nk)
    op.upload_P(P1, P2)
    if nbd != nb:
        op.set_window(nbd, b0, edm)
    f = rng.uniform(0.1, 0.4, (nk, nbd))
    schrod = "schrodinger" in terms
    op.set_flags(expt=not schrod and "noexpt" not in terms, schrodinger=schrod, kernel=kernel)
    if "H" in terms:
        op.set_coherent(1e-4 * random_rho(nk, nbd, rng))
    if "eq" in terms:
        op.compute_ddmdt_eq(np.ascontiguousarray(f[:, b0:b0 + nb]))
    if "linear" in terms:
        op.set_Lsc(np.ascontiguousarray(f[:, b0:b0 + nb]))
    if "semi" in terms:
        op.set_semiclassical(True)
    if "relax" in terms:
        op.set_phenom_relax(300 * FS, 0, nbd, f)
    op.set_observable(random_rho(nk, nbd, rng), f, 0, nbd, 1.0 / nk)
    return op, random_rho(nk, nbd, rng)


CASES = [(nb, nbd, terms) for nb, nbd, terms in [
    (2, 2, ()), (2, 2, ("H", "eq")), (2, 2, ("schrodinger",)), (2, 2, ("noexpt", "eq", "H")), (2, 2, ("linear",)),
    (2, 3, ("H",)), (2, 4, ("H", "relax")), (2, 5, ("schrodinger", "H")), (2, 6, ("H", "eq")), (2, 7, ("semi", "H")),
    (2, 8, ("H", "relax", "eq")), (4, 4, ()), (4, 4, ("H", "eq")), (4, 4, ("linear", "H")), (4, 5, ("H",)),
    (4, 6, ("semi", "relax")), (4, 8, ("schrodinger", "H"))]]


@pytest.mark.parametrize("nb,nbd,terms", CASES)
@pytest.mark.parametrize("edge", [-1, 0, 1])
def test_fused_stages_match_the_separate_ones(nb, nbd, terms, edge):
    torch = pytest.importorskip("torch")
    torch.cuda.set_device(0)
    nk = max(4, 2 * (256 // nbd ** 2) + edge)  # two blocks of whole k points, one less or one more
    print(f"case stages nb={nb} nbd={nbd} nk={nk} {terms}", flush=True)
    t = 31 * FS
    got = {}
    for kernel in (_lib.DMD_KERNEL_TILES, _lib.DMD_KERNEL_ROWS):
        op, rho = _op(nb, nbd, nk, kernel, terms, 100 * nbd + nb)
        with op:
            y, obs = op.integrate_rk4(rho, t, FS, 3, 1)
            z, t1, h, st = op.rkf45_apply(rho, t, t + 2 * FS, FS, hmax=FS, eps_abs=1e-3)
            r = op.compute_rhs(t, rho)
            u = op.integrate_euler(rho, t, FS, 2)
            d = op.evolve_driver(t, rho, np.eye(nbd).reshape(-1) - rho)
        got[kernel] = (y, obs, z, r, u, d), (t1, h, st["steps"], st["rejected"])
    (a, sa), (b, sb) = got.values()
    assert sa[0] == sb[0] and sa[2:] == sb[2:]
    for x, w in zip(a, b):
        s = np.abs(w).max()
        assert s > 0 and np.abs(x - w).max() <= 1e-12 * s


def test_adjoint_of_more_components_than_one_pass():
    """Nine components (one pass over the cotangent sums takes eight): the same
    handle nine times gives nine times the derivative it gives alone."""
    torch = pytest.importorskip("torch")
    torch.cuda.set_device(0)
    rng = np.random.default_rng(3)
    nk, nb = 70, 2
    e = random_energies(nk, nb, rng)
    k1, k2 = random_pairs(nk, 6, rng, diag=True)
    P1, P2 = random_P(len(k1), nb, rng)
    rho, f = random_rho(nk, nb, rng), rng.uniform(0.1, 0.4, (nk, nb))
    with scatt.ScatteringOperator(nk, nb, k1, k2, e) as op, scatt.ScatteringOperator(nk, nb, k1, k2, e) as c:
        c.upload_P(P1, P2)
        op.combine_P([c], [1.0])
        op.set_observable(random_rho(nk, nb, rng), f, 0, nb, 1.0 / nk)
        dobs = rng.normal(size=6)
        one, g1 = op.adjoint_rk4(rho, 0.0, FS, 5, 1, 2, dobs, [c])
        nine, g9 = op.adjoint_rk4(rho, 0.0, FS, 5, 1, 2, dobs, [c] * 9)
    assert np.abs(nine - one[0]).max() <= 1e-12 * abs(one[0])
    assert np.abs(g9 - g1).max() <= 1e-12 * np.abs(g1).max()


@pytest.mark.parametrize("nk,partners", [(3, 1), (65, 20), (512, 3), (513, 9), (1100, 2), (1537, 24)])
def test_tile_vjp_matches_the_row_kernels(nk, partners):
    """The tile VJP, its chunks from a few pairs to several iterations of every
    wavefront and its rows on both sides of a tile's edge, diagonal pairs included,
    against the gather and scatter of the general path: FP64 sums in another order,
    1e-12 of the largest element."""
    torch = pytest.importorskip("torch")
    torch.cuda.set_device(0)
    rng = np.random.default_rng(nk)
    e = random_energies(nk, 2, rng)
    k1, k2 = random_pairs(nk, partners, rng, diag=True)
    P1, P2 = random_P(len(k1), 2, rng)
    rho = random_rho(nk, 2, rng)
    v = rng.normal(size=(nk, 4)) + 1j * rng.normal(size=(nk, 4))
    got = []
    for kernel in (_lib.DMD_KERNEL_TILES, _lib.DMD_KERNEL_ROWS):
        with scatt.ScatteringOperator(nk, 2, k1, k2, e) as op:
            op.upload_P(P1, P2)
            op.set_flags(expt=True, schrodinger=False, kernel=kernel)
            got.append(op.vjp(31 * FS, rho, v))
    assert np.abs(got[1]).max() > 0
    assert np.abs(got[0] - got[1]).max() <= 1e-12 * np.abs(got[1]).max()
