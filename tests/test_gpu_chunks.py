"""The tile kernels' work split: pieces of the row-block tiles whose sizes fall
on and beside the units the split rounds to, against the CPU oracle.

Tolerance: FP64 sums of at most a few thousand terms per row, 1e-12 of the
result's norm as in the other parity tests."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from helpers import FS, random_energies, random_P, random_rho, rel_err  # noqa: E402

from denmat_dynm_development_amd import _lib, scatt  # noqa: E402
from oracle import oracle  # noqa: E402

pytestmark = pytest.mark.gpu


def _rows(nk, counts, rng):
    """Stored pairs with counts[k] partners k' >= k of row k (all of them past the end)."""
    k1, k2 = [], []
    for k, c in enumerate(counts):
        q = np.sort(rng.permutation(np.arange(k, nk))[:c])
        k1.append(np.full(len(q), k))
        k2.append(q)
    return np.concatenate(k1).astype(np.uint64), np.concatenate(k2).astype(np.uint64)


@pytest.mark.parametrize("nb,nk,counts", [
    (2, 700, [1] + [0] * 699),                       # one pair in all
    (2, 700, [255] + [0] * 400 + [257] + [0] * 298),  # one short piece in each of two tiles
    (2, 700, [64] * 700),                            # many pieces of the shortest length
    (2, 1500, [90] * 1500),                          # six tiles, more pieces than CUs
    (4, 70, [15] + [0] * 31 + [17] + [0] * 37),
    (4, 70, [64] * 70),
    (4, 300, [130] * 300),                           # panels of 4160 pairs and fewer
])
def test_tile_pieces_match_the_oracle(torch_cuda, nb, nk, counts):
    torch = torch_cuda
    rng = np.random.default_rng(nk + nb)
    k1, k2 = _rows(nk, counts, rng)
    e = random_energies(nk, nb, rng)
    P1, P2 = random_P(len(k1), nb, rng)
    rho = random_rho(nk, nb, rng)
    t = 23 * FS
    ref = oracle.evolve(k1, k2, P1, P2, e, rho, t=t, prefac=2 * np.pi / nk)
    with scatt.ScatteringOperator(nk, nb, k1, k2, e, nk_full=nk) as op:
        op.upload_P(P1, P2)
        for r1 in (None, np.eye(nb).reshape(-1) - rho):
            got = op.eval(t, torch.from_numpy(rho).cuda(), None if r1 is None else torch.from_numpy(r1).cuda())
            assert rel_err(got.cpu().numpy(), ref) < 1e-12
        P1b, P2b = op.download_P()
        assert np.array_equal(P1b, P1) and np.array_equal(P2b, P2)


@pytest.mark.parametrize("prec", [_lib.DMD_PREC_C64, _lib.DMD_PREC_BF16])
@pytest.mark.parametrize("nk,counts", [
    (70, [1] + [0] * 69),
    (70, [5] + [0] * 31 + [21] + [0] * 37),  # waves with no pair, one and two
    (40, [17] * 20 + [1] * 20),
    (70, [64] * 70),
    (300, [130] * 300),
])
def test_reduced_panels_are_exact_on_dyadic_data(torch_cuda, prec, nk, counts):
    """P of small integers and a state of eighths: every product and partial sum of
    the FP32 contraction is exact, so the result is the FP64 one but for the FP64
    epilogue's roundings (1e-13 of the largest element)."""
    torch = torch_cuda
    nb = 4
    rng = np.random.default_rng(nk + len(set(counts)))
    k1, k2 = _rows(nk, counts, rng)
    shape = (len(k1), 16, 16)
    P1, P2 = (rng.integers(-4, 5, shape) + 1j * rng.integers(-4, 5, shape) for _ in range(2))
    h = rng.integers(-4, 5, (nk, nb, nb)) / 16 + 1j * rng.integers(-4, 5, (nk, nb, nb)) / 16
    rho = np.ascontiguousarray((h + h.conj().transpose(0, 2, 1)).reshape(nk, 16))
    e = random_energies(nk, nb, rng)
    out = []
    for q in (_lib.DMD_PREC_FP64, prec):
        with scatt.ScatteringOperator(nk, nb, k1, k2, e, nk_full=nk, precision=q) as op:
            op.upload_P(P1, P2)
            if q != _lib.DMD_PREC_FP64:
                op.set_split(None)
            out.append(op.eval(0.0, torch.from_numpy(rho).cuda()).cpu().numpy())
    assert np.abs(out[0]).max() > 0
    assert np.abs(out[1] - out[0]).max() <= 1e-13 * np.abs(out[0]).max()


@pytest.fixture
def torch_cuda():
    torch = pytest.importorskip("torch")
    torch.cuda.set_device(0)
    return torch
