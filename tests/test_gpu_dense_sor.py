"""The dense-matrix dipole solve against the pass-by-pass one, on the same
inputs (PIMD_SOR_DENSE = 2 and 0), at the edges of its forms: 21/22, 42/43 and
64/65 dipole sites (rows held per lane group; one block per bead or a launch
per iteration), odd and even iteration caps, boxes whose |kz| range falls into
each bucket of the weight table, and the mixed form.

Both evaluate the same sums in FP64, so energies, gradients and dipoles agree
to rounding: a dipole field sums some 1e3 terms (1e-13 relative), and the
forces are linear in the dipoles.
"""
import numpy as np
import pytest

from helpers import max_abs, rel_err

pytestmark = pytest.mark.gpu

CASES = [
    # model, waters, beads, box aspect, eps, maxiter
    (3, 21, 2, (1, 1, 1), 1e-6, 15), (3, 22, 2, (1, 1, 1), 1e-8, 15),
    (3, 42, 1, (1, 1, 1), 1e-6, 4), (3, 43, 3, (1, 1, 1.6), 1e-6, 15),
    (3, 64, 2, (1, 1, 1), 1e-6, 3), (3, 65, 2, (1, 1, 1), 1e-6, 15),
    (3, 67, 1, (1, 1, 1), 1e-6, 5), (3, 100, 2, (1, 1, 1), 1e-6, 4),
    (2, 7, 2, (1, 1, 1), 1e-4, 15), (2, 21, 3, (1, 1, 1), 1e-6, 15),
    (2, 22, 2, (1, 1, 1), 1e-8, 15), (2, 45, 2, (1, 1.2, 1), 1e-6, 5),
]


def _forces(monkeypatch, dense, p, R, Rc):
    from pimd_amd.ttm import TTMForceField
    monkeypatch.setenv("PIMD_SOR_DENSE", str(dense))
    ff = TTMForceField(p)
    r = ff.full_bead_forces(R, Rc)
    ff.close()
    return r


@pytest.mark.parametrize("model,N,P,aspect,eps,maxiter", CASES)
@pytest.mark.parametrize("mixed", [0, 1])
def test_dense_solve_matches_passes(monkeypatch, model, N, P, aspect, eps, maxiter, mixed):
    from pimd_amd.params import TTMParams
    from pimd_amd.systems import ring_polymer, spaced_water_box
    print("case", model, N, P, aspect, eps, maxiter, mixed, flush=True)
    cen, L = spaced_water_box(N, seed=5, tries=30)
    box = tuple(L * a for a in aspect)
    R, _ = ring_polymer(cen, P, seed=6)
    p = TTMParams(pot_model=model, nwaters=N, nbeads=P, box=box, eps_ewald=eps,
                  polar_maxiter=maxiter).resolved()
    ref = _forces(monkeypatch, 0, p, R, R.mean(0))
    p.precision = mixed
    got = _forces(monkeypatch, 2, p, R, R.mean(0))
    if not mixed:
        assert np.array_equal(got["iters"], ref["iters"])
        assert rel_err(got["Upott"], ref["Upott"]) < 1e-11
        assert max_abs(got["dRRt"], ref["dRRt"]) < 1e-9
        assert max_abs(got["dip_momEt"], ref["dip_momEt"]) < 1e-10
        assert max_abs(got["virt"], ref["virt"]) < 1e-7
    else:
        # the mixed form's pair passes are FP32, its dense solve FP64: forces
        # within the form's 1e-5 of FP64
        d = got["dRRt"] - ref["dRRt"]
        assert np.sqrt(np.mean(d * d)) < 1e-5 * np.sqrt(np.mean(ref["dRRt"] ** 2))
