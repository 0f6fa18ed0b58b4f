"""The reciprocal-space passes at the edges of their tiles: 16 kz-columns and 8
|kz| to a structure-factor product, chunks of 8 sites, 16-site tiles, one or
two to a group of a field block, one round of tasks and several.  Molecule counts that
leave one site, a full tile and one more; boxes of unequal axes, whose |kz|
reach from 4 past 16; every model; the dipole passes forced where the dense
solve would take them.  Against the oracle at the bounds of
test_gpu_forces.py; the mixed form's forces and virials within its 1e-5 of
FP64.  The molecules are moved off the lattice sites by up to 0.05 A: two
centroids exactly half a box apart have a minimum image that rounding decides."""
import numpy as np
import pytest

from test_gpu_forces import _oracle_forces, check_against

pytestmark = pytest.mark.gpu

CASES = [
    # model, waters, beads, box aspect, eps
    (3, 2, 1, (1, 1, 1), 1e-8), (3, 11, 2, (1, 1, 3), 1e-8), (3, 16, 3, (1, 1, 1), 1e-4),
    (3, 33, 2, (1.5, 1, 1), 1e-6), (3, 33, 1, (1, 1, 5), 1e-10), (3, 86, 2, (1, 1, 1), 1e-10),
    (2, 2, 1, (1, 1, 1), 1e-6), (2, 11, 2, (1, 2, 1), 1e-8), (2, 43, 2, (1, 1, 2), 1e-8),
    (4, 11, 2, (1, 1, 4), 1e-8), (5, 43, 3, (1, 1, 1), 1e-6),
    # beads enough for two tiles to a site group
    (3, 33, 48, (1, 1, 1.5), 1e-6), (2, 17, 64, (1, 1, 1), 1e-6), (4, 22, 64, (1, 1, 1), 1e-6),
]


@pytest.mark.parametrize("model,N,P,aspect,eps", CASES)
def test_reciprocal_passes(monkeypatch, model, N, P, aspect, eps):
    from pimd_amd.params import TTMParams
    from pimd_amd.systems import ring_polymer, spaced_water_box
    from pimd_amd.ttm import TTMForceField
    print("case", model, N, P, aspect, eps, flush=True)
    monkeypatch.setenv("PIMD_SOR_DENSE", "0")
    cen, L = spaced_water_box(N, seed=7, tries=30)
    shift = np.random.default_rng(9).uniform(-0.05, 0.05, (N, 1, 3))
    cen = (np.reshape(cen, (N, 3, 3)) + shift).reshape(3 * N, 3)
    R, _ = ring_polymer(cen, P, seed=8)
    p = TTMParams(pot_model=model, nwaters=N, nbeads=P, box=tuple(L * a for a in aspect),
                  eps_ewald=eps).resolved()
    ff = TTMForceField(p)
    r = ff.full_bead_forces(R, R.mean(0))
    ff.close()
    ref = _oracle_forces(p, R, R.mean(0), list(range(P)))
    check_against(r, ref, p, "recip")
    if model > 3:
        return
    p.precision = 1
    ff = TTMForceField(p)
    m = ff.full_bead_forces(R, R.mean(0))
    ff.close()
    d = m["dRRt"] - r["dRRt"]
    assert np.sqrt(np.mean(d * d)) < 1e-5 * np.sqrt(np.mean(r["dRRt"] ** 2))
    # the centroid virial may pass through zero: by the virial's size
    size = np.max(np.abs(r["virt_cm"]))
    assert np.max(np.abs(m["virt_cm"] - r["virt_cm"])) < 1e-5 * size
    assert np.max(np.abs(m["virialct"] - r["virialct"])) < 1e-5 * size
