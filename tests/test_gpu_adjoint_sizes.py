"""The adjoint sweep at the edges of its kernels: odd molecule counts (remainders
of the 8 x 8 tiles, of the 16 lanes per site and of the 4 sites per wave group)
against the tangent sweeps, configurations cut into slices, the pass-by-pass
dipole solve against the dense one, and systems too large for the dense one
against the forward model.  The bars against the tangents are those of
test_gpu_ttm_adjoint.py."""
import numpy as np
import pytest

from test_gpu_ttm_adjoint import _compare

pytestmark = pytest.mark.gpu


def _setup(model, N, P, **kw):
    from pimd_amd.params import TTMParams
    from pimd_amd.systems import ring_polymer, spaced_water_box
    from pimd_amd.ttm import TTMForceField
    cen, L = spaced_water_box(N, seed=N, tries=30)
    R, _ = ring_polymer(cen, max(P, 2), seed=N + 1)
    p = TTMParams(pot_model=model, nwaters=N, nbeads=P, box=(L, L, L), polar_eps=1e-12,
                  polar_maxiter=100, **kw).resolved()
    rng = np.random.default_rng(N)
    return TTMForceField(p), R[:P], rng.standard_normal(P), rng.standard_normal((P, 3 * N, 3))


@pytest.mark.parametrize("model,N,P", [(3, 9, 3), (3, 17, 2), (3, 33, 1), (2, 7, 3), (2, 11, 2)])
def test_adjoint_odd_sizes_match_tangents(model, N, P):
    print("case", model, N, P, flush=True)
    ff, R, ew, gw = _setup(model, N, P, eps_ewald=1e-8)
    ga = ff.ttm_adjoint(R, ew, gw, 101)[0]
    gt = np.concatenate([ff.ttm_param_grad(R, ew, gw)[0], ff.dms_coef_grad(R, ew, gw)[0],
                         [ff.gamma_m_grad(R, ew, gw)[0]]])
    _compare("loss gradient", ga, gt, model)
    ff.close()


def test_adjoint_in_slices(monkeypatch):
    """32 H2O: 147 KB of matrix per configuration, 7 per MB; nine of them in two
    slices give the same bits as in one."""
    ff, R, ew, gw = _setup(3, 32, 9)
    one = ff.ttm_adjoint(R, ew, gw)
    monkeypatch.setenv("PIMD_ADJ_MAT_MB", "1")
    two = ff.ttm_adjoint(R, ew, gw)
    for a, b in zip(one, two):
        assert np.array_equal(a, b)
    ff.close()


def test_adjoint_dipoles_beyond_lds():
    """700 TTM3-F waters (2100 dipole components, solved pass by pass): the energy against the force
    call's, and dE/d polarM against its central difference (h = 1e-6 relative:
    truncation 1e-12, rounding 1e-13 / 1e-6 of the energy)."""
    ff, R, ew, gw = _setup(3, 700, 1)
    _, E, dE = ff.ttm_adjoint(R, ew, gw, 16)
    U = ff.full_bead_forces(R, R[0])["Upott"]
    assert abs(E[0] - U[0]) < 1e-11 * abs(U[0])
    th = ff.ttm_params()
    u = []
    for s in (1, -1):
        t = th.copy()
        t[7] *= 1 + s * 1e-6
        ff.set_ttm_params(t)
        u.append(ff.full_bead_forces(R, R[0])["Upott"][0])
    fd = (u[0] - u[1]) / (2e-6 * th[7])
    assert abs(fd - dE[0, 7]) < 1e-6 * abs(fd) + 1e-7 * abs(U[0]) / th[7]
    ff.close()


@pytest.mark.parametrize("model,N,P,maxiter", [(3, 2, 2, 100), (3, 13, 3, 100), (3, 65, 2, 4),
                                               (3, 66, 1, 5), (2, 7, 3, 100), (2, 22, 2, 3)])
def test_adjoint_passes_match_dense(monkeypatch, model, N, P, maxiter):
    """The pass-by-pass dipole solve against the dense one (PIMD_ADJ_DENSE = 0
    and by size) where four sites to a workgroup and 64 molecules to a wave
    leave remainders, stopped by convergence and after odd and even counts:
    the same sums in another order, 1e-11 of the largest derivative."""
    print("case", model, N, P, maxiter, flush=True)
    ff, R, ew, gw = _setup(model, N, P, eps_ewald=1e-6)
    ff.close()
    from pimd_amd.params import TTMParams
    from pimd_amd.ttm import TTMForceField
    ff = TTMForceField(TTMParams(**{**ff.params.__dict__, "polar_maxiter": maxiter}))
    dense = ff.ttm_adjoint(R, ew, gw, 100)
    monkeypatch.setenv("PIMD_ADJ_DENSE", "0")
    passes = ff.ttm_adjoint(R, ew, gw, 100)
    ff.close()
    for a, b in zip(dense, passes):
        assert np.max(np.abs(a - b)) <= 1e-11 * np.max(np.abs(a))


def test_adjoint_memory_grows_with_the_sites():
    """2000 TTM2.1-F waters: the dual dipole matrix alone would take 5.2 GB.
    The adjoint's device memory stays under 1 GB, its energy is the force
    call's and dE/d polarO the central difference."""
    import ctypes as C
    ff, R, ew, gw = _setup(2, 2000, 1, eps_ewald=1e-4)
    hip = C.CDLL("libamdhip64.so.7")
    free, total = C.c_size_t(), C.c_size_t()

    def free_bytes():
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    U = ff.full_bead_forces(R, R[0])["Upott"]
    before = free_bytes()
    _, E, dE = ff.ttm_adjoint(R, ew, gw, 16)
    assert before - free_bytes() < 1 << 30
    assert abs(E[0] - U[0]) < 1e-11 * abs(U[0])
    th = ff.ttm_params()
    u = []
    for s in (1, -1):
        t = th.copy()
        t[5] *= 1 + s * 1e-6
        ff.set_ttm_params(t)
        u.append(ff.full_bead_forces(R, R[0])["Upott"][0])
    fd = (u[0] - u[1]) / (2e-6 * th[5])
    assert abs(fd - dE[0, 5]) < 1e-6 * abs(fd) + 1e-7 * abs(U[0]) / th[5]
    ff.close()
