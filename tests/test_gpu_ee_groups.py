"""The e-e P of pairs grouped by q = k1 - k2 (nb <= 2, Lindblad form, no
exchange) against the per-pair kernel (DMD_EE_FORMS) on the same inputs, at
group sizes on both sides of a full group and one, two and three tiles of k3,
and against the CPU oracle on a small mesh.

Tolerance: both sides sum the same terms in FP64 in another order, up to 1200
k3 with 16 terms each; 1e-13 of the largest element, as between the per-form
passes, is some hundred roundings."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from helpers import random_energies  # noqa: E402

pytestmark = pytest.mark.gpu
R = np.array([[0.0, 5.34145, 5.34145], [5.34145, 0.0, 5.34145], [5.34145, 5.34145, 0.0]])


def _inputs(nb, km, drop, rng):
    g = np.stack(np.meshgrid(*[np.arange(n) for n in km], indexing="ij"), -1).reshape(-1, 3)
    g = g[np.sort(rng.permutation(len(g))[drop:])]  # k points missing from the mesh
    nk = len(g)
    e = random_energies(nk, nb, rng)
    f = 1 / (np.exp((e - 0.4 * e.max()) / 9.5e-4) + 1)
    nw = 3
    U = (rng.normal(size=(nk, nw, nb)) + 1j * rng.normal(size=(nk, nw, nb))) / 2
    A = rng.normal(size=(nk, nb, nb)) + 1j * rng.normal(size=(nk, nb, nb))
    dm = f[:, :, None] * np.eye(nb) + 0.05 * (A + A.conj().transpose(0, 2, 1)) / 2
    return g, g / np.array(km, float), e, f, U, dm.reshape(nk, nb * nb)


def _pairs_of_q(g, km, per_q, rng):
    """Stored pairs (i <= j in list order) with per_q[i] pairs of the i-th difference met."""
    nk = len(g)
    i, j = np.triu_indices(nk)
    d = (g[i] - g[j]) % np.array(km)
    code = (d[:, 0] * km[1] + d[:, 1]) * km[2] + d[:, 2]
    keep = []
    for n, c in zip(per_q, rng.permutation(np.unique(code))):
        keep.append(np.flatnonzero(code == c)[:n])
    k = np.sort(np.concatenate(keep))
    return i[k].astype(np.uint64), j[k].astype(np.uint64)


def _model(scatt, nw, km):
    return scatt.eimp_model("debye", 3e-6, 9.5e-4, abs(np.linalg.det(R)), scatt.reciprocal_metric(R), nw,
                            n_ionized=1.0, epsilon_background=3.0, degauss=4e-4, ethr=1.2e-3, kmesh=km, nk_full=36.0)


@pytest.mark.parametrize("nb", [1, 2])
@pytest.mark.parametrize("km,drop,per_q", [
    ((4, 4, 3), 3, [1, 2, 3, 4, 5, 7, 8, 9, 16, 17] + [40] * 30),  # every group size; one tile, k4 missing for some k3
    ((8, 8, 8), 0, [8, 30] + [128] * 32),  # 512 k3: the tile exactly
    ((9, 8, 8), 63, [11, 12] + [90] * 42),  # 513 k3: one past it
    ((11, 11, 10), 0, [40, 3, 25] + [390] * 30),  # three tiles
    ((4, 4, 3), 0, [5, 6, 6]),  # fewer than six pairs per q: the per-pair kernel
])
def test_grouped_matches_per_pair(monkeypatch, nb, km, drop, per_q):
    torch = pytest.importorskip("torch")
    torch.cuda.set_device(0)
    from denmat_dynm_development_amd import scatt
    print(f"case ee groups nb={nb} mesh={km} per_q={per_q}", flush=True)
    rng = np.random.default_rng(sum(per_q) + nb)
    g, kv, e, f, U, dm = _inputs(nb, km, drop, rng)
    k1, k2 = _pairs_of_q(g, km, per_q, rng)
    assert len(per_q) == 3 or len(k1) >= 6 * len(g)  # else the per-pair kernel on both sides
    nk, m, out = len(g), _model(scatt, U.shape[1], km), {}
    for forms in (None, "2"):
        if forms:
            monkeypatch.setenv("DMD_EE_FORMS", forms)
        else:
            monkeypatch.delenv("DMD_EE_FORMS", raising=False)
        with scatt.ScatteringOperator(nk, nb, k1, k2, e) as op:
            got = []
            op.add_ee_model(k1, k2, U, kv, f, m, add=False)
            got.append(op.download_P())
            op.add_ee_model_state(k1, k2, U, kv, f, m, dm=dm, add=False)
            got.append(op.download_P())
            op.add_ee_dP(k1, k2, U, kv, f, m, dm, add=False)
            got.append(op.download_P())
            out[forms] = got
    for (a1, a2), (b1, b2) in zip(out[None], out["2"]):
        for a, b in ((a1, b1), (a2, b2)):
            s = np.abs(b).max()
            assert s > 0 and np.abs(a - b).max() <= 1e-13 * s


@pytest.mark.parametrize("nb", [1, 2])
def test_grouped_matches_the_oracle(nb):
    torch = pytest.importorskip("torch")
    torch.cuda.set_device(0)
    from denmat_dynm_development_amd import scatt
    from oracle import oracle
    rng, km = np.random.default_rng(5 + nb), (4, 4, 3)
    g, kv, e, f, U, dm = _inputs(nb, km, 3, rng)
    i, j = np.triu_indices(len(g))
    k1, k2 = i.astype(np.uint64), j.astype(np.uint64)  # every pair, k = k' among them
    m = _model(scatt, U.shape[1], km)
    d = m.as_dict()
    vq = np.array([oracle.eimp_vq(d, oracle.eimp_q2(d["GGT"], kv[a], kv[b])) for a, b in zip(i, j)])
    dm1 = np.eye(nb).reshape(-1) - dm
    R1, R2 = oracle.ee_model_P(k1, k2, U, kv, e, f, vq, km, 4e-4, 1.2e-3, 36.0, True, dm=dm, dm1=dm1)
    with scatt.ScatteringOperator(len(g), nb, k1, k2, e) as op:
        op.add_ee_model_state(k1, k2, U, kv, f, m, dm=dm, scale=0.7, add=False)
        A1, A2 = op.download_P()
    for a, r in ((A1, R1), (A2, R2)):
        s = np.abs(r).max()
        assert s > 0 and np.abs(a - 0.7 * r).max() <= 1e-12 * s
