"""The line transforms and the x-line pass at the sizes where their plans
change: every radix of a stage, one- to four-stage lines, y-z planes of both
register budgets and the separate line passes, and every number of types of
the x-line pass (1 to 8, 9 beyond it, Mx = 4 without it)."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import field as F
from tests.conftest import rms_rel

pytestmark = pytest.mark.gpu


def _dev(a, dtype):
    return torch.as_tensor(np.ascontiguousarray(a)).to(dtype).cuda().contiguous()


@pytest.mark.parametrize("mesh", [(4, 4, 4), (6, 10, 6), (18, 10, 10), (30, 12, 16), (50, 54, 18), (90, 150, 20),
                                  (16, 162, 54), (8, 30, 250), (12, 90, 60), (24, 100, 100), (6, 144, 150),
                                  (6, 150, 200), (4, 750, 8), (480, 4, 6), (900, 6, 4), (4, 8, 1024),
                                  (4, 192, 192), (10, 240, 250),
                                  # several planes per CU (more than 256 of them): the register blocks and
                                  # wavefronts chosen for planes of 2 KB to 150 KB
                                  (150, 72, 256), (160, 200, 96), (150, 90, 72), (160, 54, 96), (270, 16, 18),
                                  (160, 162, 108)])
def test_line_plans_vs_numpy(hip, mesh):
    """r2c and c2r against numpy in FP64; an FP32 transform's error grows like
    sqrt(log G) ulp: 2e-6 of the spectrum's RMS, 2e-5 of the largest value back."""
    from hymd_amd.field import ParticleMesh
    rng = np.random.default_rng(sum(mesh))
    pm = ParticleMesh(mesh, (1.0, 1.0, 1.0), 2)
    x = rng.normal(size=(2,) + mesh).astype(np.float32)
    ref = np.fft.rfftn(x.astype(np.float64), axes=(1, 2, 3))
    X = pm.r2c(_dev(x, torch.float32)).cpu().numpy()
    assert np.sqrt(np.mean(np.abs(X - ref) ** 2)) / np.sqrt(np.mean(np.abs(ref) ** 2)) < 2e-6
    y = pm.c2r(_dev(ref.astype(np.complex64), torch.complex64)).cpu().numpy()
    np.testing.assert_allclose(y / np.prod(mesh), x, atol=2e-5 * np.abs(x).max())


@pytest.mark.parametrize("mesh", [(4, 6, 8), (6, 4, 6), (18, 10, 12), (16, 30, 20), (30, 16, 10), (128, 8, 6),
                                  (150, 6, 8), (96, 10, 16), (256, 6, 4), (64, 20, 18), (8, 100, 100), (4, 150, 160),
                                  (6, 192, 200), (160, 6, 8), (192, 6, 8), (216, 6, 8), (240, 6, 8)])
@pytest.mark.parametrize("T", [1, 2, 3, 4, 5, 6, 7, 8, 9])
def test_field_pass_matches_oracle(hip, mesh, T):
    """Force grids, densities, their spectra, potentials and energy of one
    update against the FP64 oracle (1e-5 and 1e-6 of each one's RMS), and the
    force grids of the update that returns nothing else."""
    from hymd_amd.field import ParticleMesh
    rng = np.random.default_rng(sum(mesh) + T)
    box = np.array(mesh) * 0.25
    n = 3000
    x = (rng.uniform(0, 1, (n, 3)) * box).astype(np.float32)
    types = rng.integers(0, T, n).astype(np.int32)
    A = rng.uniform(0.0, 1.0, (T, T))
    A = A + A.T + T * np.eye(T)
    b = rng.uniform(-1, 1, T)
    ham = F.Quadratic(A, b, 0.3)
    ref = F.update_field(x.astype(np.float64), types, T, mesh, box, 0.4, ham, compute_potential=True)
    pm = ParticleMesh(mesh, box, T)
    xd, td = _dev(x, torch.float32), _dev(types, torch.int32)
    only, fm = pm.create("real", batch=(T, 3)), pm.create("real", batch=(T, 3))
    phi, v, phif = pm.create("real", batch=T), pm.create("real", batch=T), pm.create("complex", batch=T)
    pm.field_update(xd, td, T, A, b, 0.3, [1.0] * T, 0.4, only)
    e = pm.field_update(xd, td, T, A, b, 0.3, [1.0] * T, 0.4, fm, phi=phi, phi_fourier=phif, v_ext=v,
                        want_energy=True)
    want = np.array([[ref["force_mesh"][t][d] for d in range(3)] for t in range(T)])
    assert rms_rel(only.cpu().numpy(), want) < 1e-5
    assert rms_rel(fm.cpu().numpy(), want) < 1e-5
    assert rms_rel(phi.cpu().numpy(), np.array(ref["phi"])) < 1e-6
    assert rms_rel(v.cpu().numpy(), np.array(ref["v_ext"])) < 1e-6
    assert rms_rel(phif.cpu().numpy(), np.array(ref["phi_fourier"])) < 1e-6
    assert e == pytest.approx(F.field_energy(ref["phi"], ham, mesh, box), rel=1e-6)


# lines enough (4160) for the widths that small meshes halve: 8 lines of 384 to
# 512 threads, 4 lines, and one line of one and of two types
@pytest.mark.parametrize("mesh,T", [((180, 64, 128), 4), ((200, 64, 128), 3), ((240, 64, 128), 2), ((256, 64, 128), 4),
                                    ((160, 64, 128), 5), ((144, 64, 128), 4), ((100, 64, 128), 8), ((900, 10, 8), 1),
                                    ((720, 10, 8), 2)])
def test_field_pass_at_full_width(hip, mesh, T):
    test_field_pass_matches_oracle(hip, mesh, T)


@pytest.mark.parametrize("mesh", [(6, 10, 8), (90, 12, 10), (160, 8, 6), (180, 64, 128), (216, 10, 8), (240, 64, 128),
                                  (256, 8, 10), (900, 6, 8)])
def test_pme_pass_matches_oracle(hip, mesh):
    """Field, potential and energy of the PME solve against the FP64 oracle at
    the x edges where its x-line pass changes (1e-6 of each one's RMS; an FP32
    transform's error is 2e-7 there)."""
    from hymd_amd.field import ParticleMesh
    rng = np.random.default_rng(sum(mesh))
    box = np.array(mesh) * 0.25
    n = 3000
    x = (rng.uniform(0, 1, (n, 3)) * box).astype(np.float32)
    q = np.where(np.arange(n) % 2, 1.0, -1.0)
    ref = F.update_field_force_q(x.astype(np.float64), q, mesh, box, 0.4, 138.9, 45.0)
    pm = ParticleMesh(mesh, box, 1)
    f, ef = torch.empty((n, 3), dtype=torch.float32, device="cuda"), pm.create("real", batch=3)
    psi, rho = pm.create("real"), pm.create("real")
    e = pm.pme(_dev(x, torch.float32), _dev(q, torch.float32), 0.4, 138.9 / 45.0, 0.0, f, phi_q=rho, psi=psi,
               elec_field=ef, want_energy=True)
    assert rms_rel(psi.cpu().numpy(), ref["psi"]) < 1e-6
    for d in range(3):
        assert rms_rel(ef[d].cpu().numpy(), ref["elec_field"][d]) < 1e-6
    assert rms_rel(f.cpu().numpy(), ref["forces"]) < 1e-6
    assert e == pytest.approx(F.field_q_energy(ref["phi_q"], ref["psi"], 0.0, mesh, box), rel=1e-6)


def test_edges_refused(hip):
    from hymd_amd._lib import HymdError
    from hymd_amd.field import ParticleMesh
    for mesh in ((250, 8, 8), (8, 486, 8), (500, 8, 8), (8, 960, 8), (8, 14, 8)):
        with pytest.raises(HymdError):
            ParticleMesh(mesh, (1.0, 1.0, 1.0), 1)


# either side of the 2^20 particles from which the keys are ranked per
# workgroup, with its shared table (ordered) and without (unordered)
@pytest.mark.parametrize("n", [(1 << 20), (1 << 20) + 1, (1 << 20) + 1027])
@pytest.mark.parametrize("ordered", [False, True])
def test_binning_of_large_inputs(hip, n, ordered):
    """Painted grids of the sorted path equal the scatter paint's bit for bit,
    one crowded row among them; and with weights, nine in ten of them and all of
    8192 successive particles zero (those are not binned: whole wavefronts
    and workgroups of them, and such that start with one)."""
    from hymd_amd.field import ParticleMesh
    mesh, box, T = (18, 20, 16), (4.5, 5.0, 4.0), 2
    rng = np.random.default_rng(n + ordered)
    x = rng.uniform(0, 1, (n, 3)) * np.array(box)
    x[: n // 8, :2] = 0.3
    if ordered:
        c = (x / 0.25).astype(np.int64)
        x = x[np.lexsort((c[:, 2], c[:, 1], c[:, 0]))]
    types = rng.integers(0, T, n).astype(np.int32)
    pm = ParticleMesh(mesh, box, T)
    xd, td = _dev(x, torch.float32), _dev(types, torch.int32)
    grid = pm.paint_fixed(xd, td, T)
    scat = torch.zeros((T,) + mesh, dtype=torch.int64, device="cuda")
    pm.paint_fixed(xd, td, T, out=scat, accumulate=True)
    assert torch.equal(grid.to(torch.int64), scat)
    w = rng.uniform(-1.0, 1.0, n) * (rng.random(n) < 0.1)
    w[5000: 5000 + 8192] = 0.0
    wd = _dev(w, torch.float32)
    scat = torch.zeros((1,) + mesh, dtype=torch.int64, device="cuda")
    pm.paint_fixed(xd, None, 1, weights=wd, out=scat, accumulate=True)
    assert torch.equal(pm.paint_fixed(xd, None, 1, weights=wd), scat)


@pytest.mark.parametrize("ordered", [False, True])
def test_batch_of_many_particles(hip, ordered):
    """A batch of more than 2^20 particles (keys ranked per workgroup), replicas
    that end within a wavefront or a workgroup and an empty one: moments and
    forces of each equal those of the replica alone, bit for bit."""
    from hymd_amd.batch import ReplicaBatch
    from hymd_amd.field import ParticleMesh
    counts = np.array([400001, 350003, 0, 63, 300007, 90001])
    meshes = np.array([[32, 24, 20], [24, 24, 24], [16, 16, 16], [16, 16, 16], [32, 24, 20], [20, 16, 18]])
    boxes = meshes * 0.4
    rng = np.random.default_rng(7 + ordered)
    xs, ts = [], []
    for c, m, L in zip(counts, meshes, boxes):
        x = rng.uniform(0, 1, (c, 3)) * L
        if ordered:
            cell = (x / 0.4).astype(np.int64)
            x = x[np.lexsort((cell[:, 2], cell[:, 1], cell[:, 0]))]
        xs.append(_dev(x, torch.float32))
        ts.append(_dev(rng.integers(0, 2, c), torch.int32))
    b = ReplicaBatch(meshes, boxes, counts, 2)
    R, kappa, sigma = len(counts), np.full(len(counts), 0.05), np.full(len(counts), 0.5)
    chi = np.zeros((R, 2, 2))
    chi[:, 0, 1] = chi[:, 1, 0] = 20.0
    x, t = torch.cat(xs), torch.cat(ts)
    got = b.moments(x, t, sigma)
    forces = b.energy_forces_and_gradients(x, t, chi, kappa, sigma)[4]
    rho0 = counts / np.prod(boxes, axis=1)
    A = b.coupling(chi, kappa, rho0)
    first = np.concatenate([[0], np.cumsum(counts)])
    for r in np.flatnonzero(counts):
        pm = ParticleMesh(tuple(int(v) for v in meshes[r]), boxes[r], 2)
        grids, P, phi0 = _moment_grids(pm, xs[r], ts[r], 2, A[r], np.zeros(2), float(sigma[r]))
        np.testing.assert_array_equal(got[r][0], P)
        np.testing.assert_array_equal(got[r][2], phi0)
        f = torch.empty_like(xs[r])
        pm.readout_forces(xs[r], ts[r], 2, grids, f)
        assert torch.equal(forces[first[r]: first[r + 1]], f)
    b.close()


# no iteration, one, several; a mesh whose x lines have no x-line pass (Mx = 4)
@pytest.mark.parametrize("mesh,crit,conv", [((12, 10, 8), 2.0, "max_diff"), ((12, 10, 8), 0.99, "max_diff"),
                                            ((12, 10, 8), 1e-7, "max_diff"), ((4, 12, 10), 1e-6, "max_diff"),
                                            ((4, 12, 10), 1e-4, "csum"), ((30, 16, 18), 1e-9, "euclidean_norm")])
def test_dielectric_iteration_counts(hip, mesh, crit, conv):
    """The variable-dielectric loop, whose host looks at an iteration when the
    next is enqueued: iterations (to within one, the criterion being met to
    FP32 rounding), potential and polarisation (1e-4 and 1e-3 of their RMS)
    against the FP64 oracle."""
    from hymd_amd import config as C
    from hymd_amd import field as HF
    from oracle import gpe as OG
    rng = np.random.default_rng(3)
    L, T, n = np.array(mesh) * 0.4, 2, 3000
    x = (rng.uniform(0, 1, (n, 3)) * L).astype(np.float32)
    types = (x[:, 2] > 0.5 * L[2]).astype(np.int32)
    q = np.zeros(n, dtype=np.float32)
    q[:200], q[200:400] = 1.0, -1.0
    cfg = C.Config(n_steps=1, time_step=0.03, mesh_size=mesh, sigma=0.6, kappa=0.05, box_size=L, n_types=T,
                   coulombtype="PIC_Spectral_GPE", dielectric_type=[20.0, 80.0], type_charges=[0.5, -0.5],
                   conv_crit=crit, convergence_type=conv)
    pm, fields, elec, coul = HF.initialize_pm(None, cfg)
    ref_phi = F.update_field(x.astype(np.float64), types, T, mesh, L, cfg.sigma,
                             F.Quadratic(np.eye(T), np.zeros(T), 0.0))["phi"]
    ph = _dev(np.array(ref_phi), torch.float32)
    phi_q, phi_q_f, psi, efield = elec
    eps, eps_f, eta, eta_f, pol, pol_prev, _, contrib, vbar, vbar_f, fme, fme_f = coul
    forces = torch.empty((n, 3), dtype=torch.float32, device="cuda")
    HF.update_field_force_q_GPE(None, [ph[t] for t in range(T)], _dev(types, torch.int32), _dev(q, torch.float32),
                                phi_q, phi_q_f, eps, eps_f, eta, eta_f, pol_prev, pol, efield, forces, contrib, psi,
                                vbar, vbar_f, fme, fme_f, None, None, None, pm, _dev(x, torch.float32), cfg)
    ref = OG.update_field_force_q_gpe(x.astype(np.float64), types, q.astype(np.float64), ref_phi, mesh, L, cfg.sigma,
                                      cfg.dielectric_type, cfg.type_charges, cfg.coulomb_constant,
                                      conv_crit=cfg.conv_crit, conv=conv, phi_eps=np.zeros(mesh),
                                      elec_field_contrib=np.zeros(mesh))
    assert abs(pm.gpe_iterations - ref["iterations"]) <= (1 if crit < 0.5 else 0)
    assert rms_rel(psi.cpu().numpy(), ref["psi"]) < 1e-4
    if ref["iterations"]:
        assert rms_rel(pol.cpu().numpy(), ref["phi_pol"]) < 1e-3
    assert rms_rel(forces.cpu().numpy(), ref["forces"]) < 1e-4


@pytest.mark.parametrize("bad", [-1, 40])
@pytest.mark.parametrize("energies", [False, True])
@pytest.mark.parametrize("term", ["bonds", "angles", "dihedrals"])
def test_bonded_index_out_of_range(hip, bad, energies, term):
    """The stateless kernels find a bad index while the forces are enqueued:
    the call is refused, forces, dipoles, transfer matrices and energies stay as
    they were, the next call works."""
    from hymd_amd import _lib
    n, m = 40, 37
    real = torch.float32
    x = torch.rand((n, 3), generator=torch.Generator().manual_seed(3), dtype=real).cuda()
    idx = [torch.arange(m, device="cuda", dtype=torch.int32) + j for j in range(4)]
    par = [torch.full((m,), v, device="cuda", dtype=torch.float64) for v in (0.1, 1.0)]
    coeff = torch.rand((m, 6, 5), generator=torch.Generator().manual_seed(4), dtype=real).cuda()
    dtype, last = torch.ones(m, device="cuda", dtype=torch.int32), torch.ones(m, device="cuda", dtype=torch.int32)
    box = (ctypes.c_double * 3)(2.0, 2.0, 2.0)
    e, pr, clamped = ctypes.c_double(-7.0), (ctypes.c_double * 3)(-7.0, -7.0, -7.0), ctypes.c_int64(-7)
    out = [torch.full(shape, 5.0, device="cuda", dtype=real) for shape in ((n, 3), (m, 4, 3), (m, 6, 3, 3))]

    def evaluate(members):
        p = [v.data_ptr() for v in members]
        energy = ctypes.byref(e) if energies else None
        if term == "dihedrals":
            _lib.call("hymd_cdf", out[0].data_ptr(), x.data_ptr(), out[1].data_ptr(), out[2].data_ptr(), n, box, *p,
                      coeff.data_ptr(), dtype.data_ptr(), last.data_ptr(), m, 1, _lib.HYMD_F32, energy,
                      ctypes.byref(clamped) if energies else None, None)
        else:
            _lib.call("hymd_cbf" if term == "bonds" else "hymd_caf", out[0].data_ptr(), x.data_ptr(), n, box, *p,
                      par[0].data_ptr(), par[1].data_ptr(), m, _lib.HYMD_F32, energy, pr if energies else None, None)

    members = idx[: {"bonds": 2, "angles": 3, "dihedrals": 4}[term]]
    wrong = [v.clone() for v in members]
    wrong[-1][7] = bad
    torch.cuda.synchronize()
    with pytest.raises(_lib.HymdError):
        evaluate(wrong)
    torch.cuda.synchronize()
    assert e.value == -7.0 and list(pr) == [-7.0] * 3 and clamped.value == -7
    assert all(bool((v == 5.0).all()) for v in out)
    evaluate(members)
    torch.cuda.synchronize()
    assert not bool((out[0] == 5.0).any()) and bool(torch.isfinite(out[0]).all())
    if term == "dihedrals":
        assert not bool((out[1] == 5.0).any()) and not bool((out[2] == 5.0).any())


@pytest.mark.parametrize("T", [1, 2, 3, 4, 5, 6, 7, 8])
def test_force_adjoint_of_every_type_count(hip, T):
    """dL/dA_ts of L = sum_i g_i . F_i is L at the unit coupling E_ts (the
    forces are linear in A); FP64 oracle forces, 1e-5 of the largest entry (FP32 spectra)."""
    from hymd_amd.autograd import field_adjoint
    from hymd_amd.field import ParticleMesh
    rng = np.random.default_rng(T)
    mesh, box, n, sigma = (12, 10, 16), np.array((3.0, 2.5, 4.0)), 700, 0.5
    x = (rng.uniform(0, 1, (n, 3)) * box).astype(np.float32)
    types = rng.integers(0, T, n).astype(np.int32)
    g = rng.normal(size=(n, 3)).astype(np.float32)
    pm = ParticleMesh(mesh, box, T)
    dA, _ = field_adjoint(pm, _dev(x, torch.float32), _dev(types, torch.int32), T, sigma, np.eye(T),
                          _dev(g, torch.float32))
    x64, ref = x.astype(np.float64), np.zeros((T, T))
    for t in range(T):
        for u in range(T):
            E = np.zeros((T, T))
            E[t, u] = 1.0
            out = F.update_field(x64, types, T, mesh, box, sigma, F.Quadratic(E, np.zeros(T), 0.0))
            ref[t, u] = np.sum(g * F.compute_field_force(x64, types, out["force_mesh"], mesh, box))
    np.testing.assert_allclose(dA, ref, rtol=0, atol=1e-5 * np.abs(ref).max())


@pytest.mark.parametrize("T", [1, 2, 3, 4, 5, 6, 7, 8])
def test_moments_of_every_type_count(hip, T):
    """Energy of one Hamiltonian from the spectral moments and from the field
    update (FP64 sums of FP32 spectra in another order: 1e-6)."""
    from hymd_amd.autograd import moments
    from hymd_amd.field import ParticleMesh
    rng = np.random.default_rng(T)
    mesh, box, n, sigma = (12, 10, 16), np.array((3.0, 2.5, 4.0)), 900, 0.5
    xd = _dev(rng.uniform(0, 1, (n, 3)) * box, torch.float32)
    td = _dev(rng.integers(0, T, n), torch.int32)
    A = rng.uniform(0, 1, (T, T)) + 2 * np.eye(T)
    A = A + A.T
    pm = ParticleMesh(mesh, box, T)
    e = pm.field_update(xd, td, T, A, np.zeros(T), 0.0, [1.0] * T, sigma, pm.create("real", batch=(T, 3)),
                        want_energy=True)
    P = np.asarray(moments(pm, xd, td, T, sigma)[0])
    assert 0.5 * np.prod(box) * np.sum(A * P) == pytest.approx(e, rel=1e-6)


def _moment_grids(pm, xd, td, T, A, b, sigma):
    """Force grids of the separate passes (hymd_field_moments), whose density
    spectra the handle then holds; (grids, moments P, phi~(0))."""
    from hymd_amd._lib import call, darr, dptr
    grids = pm.create("real", batch=(T, 3))
    nv = T * (T + 1) + T
    out = (ctypes.c_double * nv)()
    call("hymd_field_moments", pm.handle, dptr(xd, torch.float32), dptr(td, torch.int32), int(xd.shape[0]), T,
         darr([1.0] * T), sigma, out, darr(np.ravel(A)), darr(b), dptr(grids, torch.float32))
    m = np.array(out)
    P = np.zeros((T, T))
    P[np.triu_indices(T)] = m[: T * (T + 1) // 2]
    return grids, P + np.triu(P, 1).T, m[T * (T + 1):]


# one line per workgroup, two of eight types, two and four where the rows have
# 129 elements: the separate passes; three shapes of the fused pass for contrast
@pytest.mark.parametrize("mesh,T,separate", [((216, 12, 10), 8, True), ((240, 10, 8), 7, True),
                                             ((144, 12, 10), 8, True), ((192, 64, 256), 6, True),
                                             ((240, 64, 256), 4, True), ((240, 10, 8), 6, False),
                                             ((192, 60, 256), 6, False), ((144, 12, 10), 7, False)])
def test_held_spectra_route(hip, mesh, T, separate):
    """Force grids from held spectra: where the x-line pass would run too few
    lines per workgroup they come from the separate passes, bit for bit the
    moments' own grids; else from the fused pass, equal to FP32 rounding (1e-6
    of the RMS).  Both agree with the FP64 oracle."""
    from hymd_amd._lib import call, darr, dptr
    from hymd_amd.field import ParticleMesh
    rng = np.random.default_rng(sum(mesh) + T)
    box = np.array(mesh) * 0.25
    n, sigma = 3000, 0.4
    x = (rng.uniform(0, 1, (n, 3)) * box).astype(np.float32)
    types = rng.integers(0, T, n).astype(np.int32)
    A = rng.uniform(0.0, 1.0, (T, T))
    A = A + A.T + T * np.eye(T)
    b = rng.uniform(-1, 1, T)
    pm = ParticleMesh(mesh, box, T)
    grids, _, _ = _moment_grids(pm, _dev(x, torch.float32), _dev(types, torch.int32), T, A, b, sigma)
    held = pm.create("real", batch=(T, 3))
    call("hymd_field_forces_held", pm.handle, T, darr(np.ravel(A)), darr(b), sigma, dptr(held, torch.float32), None)
    assert torch.equal(held, grids) == separate
    assert rms_rel(held.cpu().numpy(), grids.cpu().numpy()) < 1e-6
    ref = F.update_field(x.astype(np.float64), types, T, mesh, box, sigma, F.Quadratic(A, b, 0.0))
    want = np.array([[ref["force_mesh"][t][d] for d in range(3)] for t in range(T)])
    assert rms_rel(held.cpu().numpy(), want) < 1e-5


# x edges with a fixed pass: 128, 160 and 256 points, a width that the general
# pass takes there and the fixed pass's own
@pytest.mark.parametrize("mesh,T,other,own", [((128, 20, 18), 2, 4, 16), ((128, 20, 18), 4, 4, 8),
                                              ((160, 18, 20), 3, 2, 4), ((256, 12, 10), 5, 2, 8),
                                              ((256, 12, 10), 6, 2, 8)])
def test_xline_width_takes_effect(hip, mesh, T, other, own):
    """The launch-shape knob: another width than the fixed x-line pass's runs
    the general one, whose radices round differently (1e-6 of the RMS, not the
    same bits), for the field update and for PME; the pass's own width and none
    give the same bits."""
    from hymd_amd import tune
    from hymd_amd.field import ParticleMesh
    rng = np.random.default_rng(sum(mesh) + T)
    box = np.array(mesh) * 0.25
    n = 3000
    x = _dev(rng.uniform(0, 1, (n, 3)) * box, torch.float32)
    types = _dev(rng.integers(0, T, n), torch.int32)
    q = _dev(np.where(np.arange(n) % 2, 1.0, -1.0), torch.float32)
    A = rng.uniform(0.0, 1.0, (T, T))
    A = A + A.T
    pm = ParticleMesh(mesh, box, T)

    def grids(width):
        tune.apply(pm, {"xline_width": width})
        fm, ef = pm.create("real", batch=(T, 3)), pm.create("real", batch=3)
        pm.field_update(x, types, T, A, np.zeros(T), 0.0, [1.0] * T, 0.4, fm)
        pm.pme(x, q, 0.4, 1.0, 0.0, torch.empty_like(x), elec_field=ef)
        return fm, ef

    default, same, changed = grids(0), grids(own), grids(other)
    assert torch.equal(same[0], default[0]) and not torch.equal(changed[0], default[0])
    assert not torch.equal(changed[1], default[1])
    for a, b in zip(changed, default):
        assert rms_rel(a.cpu().numpy(), b.cpu().numpy()) < 1e-6


@pytest.mark.parametrize("solver,axis", [("pme", 0), ("gpe", 0), ("gpe", 1), ("gpe", 2)])
def test_derivative_factor_in_fp64(hip, solver, axis):
    """The electric field of a charge density cos(2 k x) on eight points, whose
    transforms are exact (factors of 1 and i), in a box whose k rounds to FP32
    with a relative error of 5e-8 or more.  A field that multiplies by k in
    FP64 is off by its roundings alone, which differ in sign over the 64
    amplitudes (6e-8 at most each: 2e-8 bounds their mean); one that multiplies
    by the rounded k is off by 5e-8 in every one."""
    from hymd_amd._lib import call, darr, dptr
    from hymd_amd.field import ParticleMesh
    mesh = [8, 4, 4] if axis == 0 else [8, 8, 4] if axis == 1 else [8, 4, 8]
    L = next(v for v in 3.0 + np.arange(320) / 64.0  # node positions are exact
             if np.float32(2 * (2.0 * np.pi / v)) / (2 * (2.0 * np.pi / v)) - 1.0 > 5e-8)
    k = 2 * (2.0 * np.pi / L)
    box = np.full(3, 4.0)
    box[axis] = L
    pm = ParticleMesh(mesh, box, 1)
    node = np.stack(np.meshgrid(*[np.arange(m) for m in mesh], indexing="ij"), -1).reshape(-1, 3)
    x = _dev(node * (box / mesh), torch.float32)
    wave = np.array([1.0, 0.0, -1.0, 0.0, 1.0, 0.0, -1.0, 0.0])[node[:, axis]]
    odd = (node[:, axis] % 2 == 1).reshape(mesh)
    dv = np.prod(box) / np.prod(mesh)
    n = len(node)
    errs = []
    for s in np.linspace(1.0, 1.97, 64).astype(np.float32):
        q = _dev(s * wave, torch.float32)
        if solver == "pme":
            ef, f = pm.create("real", batch=3), torch.empty_like(x)
            pm.pme(x, q, 0.0, 1.0, 0.0, f, elec_field=ef)
            got = np.abs(ef[axis].cpu().numpy().astype(np.float64)[odd])
        else:
            one = pm.create("real", 1.0, batch=1)
            eps, contrib, dot, f = pm.create("real"), pm.create("real"), pm.create("real"), torch.empty_like(x)
            call("hymd_update_field_force_q_gpe", pm.handle, dptr(x, torch.float32),
                 dptr(torch.zeros(n, dtype=torch.int32, device="cuda"), torch.int32), dptr(q, torch.float32), n, 1,
                 dptr(one, torch.float32), darr([1.0]), darr([0.0]), 0.0, 1.0, 1e-6, 0.6, 0, 10,
                 dptr(eps, torch.float32), None, None, dptr(contrib, torch.float32), None,
                 dptr(dot, torch.float32), None, dptr(f, torch.float32), None, None, None)
            got = np.sqrt(dot.cpu().numpy().astype(np.float64)[odd])
        errs.append(np.mean(got) / (4.0 * np.pi * float(s) / (dv * k)) - 1.0)
    assert abs(np.mean(errs)) < 2e-8


def test_line_pass_scratch(hip):
    """An update that returns every grid of a mesh whose planes do not fit in
    LDS, five per type, here 4.4 GB of half spectra: device memory grows by 4 GB at
    most, and the grids, made in two goes, equal those of updates that make
    fewer and the transforms of the returned spectra."""
    from hymd_amd.field import ParticleMesh
    rng = np.random.default_rng(5)
    mesh, T, n = (600, 256, 256), 6, 20000
    box = np.array(mesh) * 0.25
    x = _dev(rng.uniform(0, 1, (n, 3)) * box, torch.float32)
    types = _dev(rng.integers(0, T, n), torch.int32)
    A = rng.uniform(0.0, 1.0, (T, T))
    A, b = A + A.T, rng.uniform(-1, 1, T)
    pm = ParticleMesh(mesh, box, T)
    fm, phi, v = pm.create("real", batch=(T, 3)), pm.create("real", batch=T), pm.create("real", batch=T)
    phif = pm.create("complex", batch=T)
    args = (x, types, T, A, b, 0.0, [1.0] * T, 0.4)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    pm.field_update(*args, fm, phi=phi, phi_fourier=phif, v_ext=v)
    torch.cuda.synchronize()
    assert before - torch.cuda.mem_get_info()[0] <= (4 << 30) + (16 << 20)

    def close(a, b):  # to FP32 rounding: an update that returns densities may take other x passes
        return all(float((p - q).norm()) < 1e-6 * float(q.norm()) for p, q in zip(a.flatten(0, -4), b.flatten(0, -4)))

    only, v2 = torch.empty_like(fm), torch.empty_like(v)
    pm.field_update(*args, only, v_ext=v2)
    assert close(fm, only) and close(v, v2)
    assert close(phi, pm.c2r(phif))
