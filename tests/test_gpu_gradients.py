"""GPU parity of the band-energy backward (``qe_python_amd.gradients``).

Bars: FP64 energy within 1e-12 relative of the oracle; FP64 gradients
(dE/dV, dE/dtau, dE/dpsi*) within 1e-10 relative (Frobenius) of the oracle
gradients and within 1e-6 of central finite differences of the device
energy (h = 1e-5 bohr for tau, exact linear / quadratic steps for V and psi);
FP32 (complex64) energy within 2e-6 and gradients within 2e-5 relative.
"""

import numpy as np
import pytest
import torch

from oracle.forces import band_energy_gradients
from qe_python_amd.synthetic import make_system

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(np.asarray(b)))


def setup(name, nb, seed=3):
    from qe_python_amd.gradients import BandEnergyModel
    s = make_system(name)
    rng = np.random.default_rng(seed)
    psi = s.trial[:, :nb] * 2.0
    f = rng.uniform(0.5, 2.0, nb)
    model = BandEnergyModel(s.basis, s.shape, s.projectors.beta_species, s.projectors.couplings)
    ref = band_energy_gradients(s.basis.indices, s.basis.kinetic, s.basis.vectors, s.shape,
                                s.real_potential, s.projectors.beta_species,
                                s.projectors.couplings, s.projectors.positions, psi, f)
    return s, psi, f, model, ref


def run(model, s, psi, f, precision="fp64", positions=None, potential=None):
    from qe_python_amd.gradients import band_energy
    p = torch.tensor(psi, device=DEV, requires_grad=True)
    v = torch.tensor(s.real_potential if potential is None else potential, device=DEV,
                     requires_grad=True)
    t = torch.tensor(s.projectors.positions if positions is None else positions, device=DEV,
                     requires_grad=True)
    e = band_energy(model, p, v, t, f, precision=precision)
    e.backward()
    return (float(e.detach()), v.grad.cpu().numpy(), t.grad.cpu().numpy(), p.grad.cpu().numpy())


@pytest.fixture(scope="module")
def small():
    return setup("small", 8)


def test_small_fp64_against_oracle(small):
    s, psi, f, model, (e, dv, dtau, gpsi) = small
    e_d, dv_d, dtau_d, gpsi_d = run(model, s, psi, f)
    assert e_d == pytest.approx(e, rel=1e-12)
    assert rel(dv_d, dv) < 1e-10
    assert rel(dtau_d, dtau) < 1e-10
    assert rel(gpsi_d, gpsi) < 1e-10


def test_small_fp32_against_oracle(small):
    s, psi, f, model, (e, dv, dtau, gpsi) = small
    e_d, dv_d, dtau_d, gpsi_d = run(model, s, psi, f, precision="fp32")
    assert e_d == pytest.approx(e, rel=2e-6)
    assert rel(dv_d, dv) < 2e-5
    assert rel(dtau_d, dtau) < 2e-5
    assert rel(gpsi_d, gpsi) < 2e-5


def test_small_device_gradients_against_central_differences(small):
    from qe_python_amd.gradients import band_energy
    s, psi, f, model, _ = small
    _, dv_d, dtau_d, gpsi_d = run(model, s, psi, f)

    def energy(positions=None, potential=None, p=None):
        with torch.no_grad():
            return float(band_energy(
                model, torch.tensor(psi if p is None else p, device=DEV),
                torch.tensor(s.real_potential if potential is None else potential, device=DEV),
                torch.tensor(s.projectors.positions if positions is None else positions,
                             device=DEV), f))

    h = 1e-4  # bohr; E is a smooth function of tau (truncation ~h^2)
    for a, c in [(0, 0), (1, 2)]:
        plus = s.projectors.positions.copy()
        minus = s.projectors.positions.copy()
        plus[a, c] += h
        minus[a, c] -= h
        fd = (energy(positions=plus) - energy(positions=minus)) / (2 * h)
        assert fd == pytest.approx(dtau_d[a, c], rel=1e-5, abs=1e-8)
    hv = 0.1  # E is linear in V: the central difference is exact
    for idx in [(0, 0, 0), (7, 20, 33)]:
        vp, vm = s.real_potential.copy(), s.real_potential.copy()
        vp[idx] += hv
        vm[idx] -= hv
        fd = (energy(potential=vp) - energy(potential=vm)) / (2 * hv)
        assert fd == pytest.approx(dv_d[idx], rel=1e-8, abs=1e-12)
    d = np.random.default_rng(9).standard_normal(psi.shape) * (1 + 1j)
    hp = 1e-2  # E is quadratic in psi: the central difference is exact
    fd = (energy(p=psi + hp * d) - energy(p=psi - hp * d)) / (2 * hp)
    assert fd == pytest.approx(float(np.real(np.vdot(gpsi_d, d))), rel=1e-6)


def test_medium_workload_backward_against_oracle():
    """The differentiation workload: 72^3 grid, 64 atoms, 128 occupied bands
    (f = 2), complex128 and complex64."""
    from qe_python_amd.gradients import BandEnergyModel
    s = make_system("medium")
    nb = 128
    psi = s.trial[:, :nb]
    f = np.full(nb, 2.0)
    model = BandEnergyModel(s.basis, s.shape, s.projectors.beta_species, s.projectors.couplings)
    e, dv, dtau, gpsi = band_energy_gradients(
        s.basis.indices, s.basis.kinetic, s.basis.vectors, s.shape, s.real_potential,
        s.projectors.beta_species, s.projectors.couplings, s.projectors.positions, psi, f)
    e_d, dv_d, dtau_d, gpsi_d = run(model, s, psi, f)
    assert e_d == pytest.approx(e, rel=1e-12)
    assert rel(dv_d, dv) < 1e-10 and rel(dtau_d, dtau) < 1e-10 and rel(gpsi_d, gpsi) < 1e-10
    e32, dv32, dtau32, gpsi32 = run(model, s, psi, f, precision="fp32")
    assert e32 == pytest.approx(e, rel=2e-6)
    assert rel(dv32, dv) < 2e-5 and rel(dtau32, dtau) < 2e-5 and rel(gpsi32, gpsi) < 2e-5


def test_medium_workload_central_differences():
    """The differentiation workload at its own size (72^3 grid, 64 atoms,
    128 bands, f = 2) against central differences of the FP64 device energy
    with the config's steps: h = 1e-5 bohr in tau (the three largest force
    components) and 1e-6 Ry in V(r) (E is linear in V, so that difference is
    exact up to rounding; it is taken along a seeded direction over the whole
    grid).  The complex128 gradient is held to 1e-6 and the complex64 one to
    1e-4 of each difference."""
    from qe_python_amd.gradients import BandEnergyModel, band_energy
    s = make_system("medium")
    nb = 128
    psi = s.trial[:, :nb]
    f = np.full(nb, 2.0)
    model = BandEnergyModel(s.basis, s.shape, s.projectors.beta_species, s.projectors.couplings)
    _, dv64, dtau64, _ = run(model, s, psi, f)
    _, dv32, dtau32, _ = run(model, s, psi, f, precision="fp32")
    p_dev = torch.tensor(psi, device=DEV)
    v0 = s.real_potential

    def energy(positions=None, potential=None):
        with torch.no_grad():
            return float(band_energy(
                model, p_dev, torch.tensor(v0 if potential is None else potential, device=DEV),
                torch.tensor(s.projectors.positions if positions is None else positions,
                             device=DEV), f))

    h = 1.0e-5
    flat = np.argsort(np.abs(dtau64).ravel())[::-1][:3]
    for a, c in zip(*np.unravel_index(flat, dtau64.shape)):
        plus = s.projectors.positions.copy()
        minus = s.projectors.positions.copy()
        plus[a, c] += h
        minus[a, c] -= h
        fd = (energy(positions=plus) - energy(positions=minus)) / (2 * h)
        print(f"tau[{a},{c}]: fd {fd:.10e} c128 {dtau64[a, c]:.10e} c64 {dtau32[a, c]:.10e}")
        assert dtau64[a, c] == pytest.approx(fd, rel=1e-6)
        assert dtau32[a, c] == pytest.approx(fd, rel=1e-4)
    # V(r): a step of 1e-6 Ry along a seeded direction over the whole grid
    # (a single grid point would move E by less than its FP64 rounding)
    hv = 0.5e-6
    d = np.random.default_rng(11).standard_normal(v0.shape)
    fd = (energy(potential=v0 + hv * d) - energy(potential=v0 - hv * d)) / (2 * hv)
    g64, g32 = float(np.sum(dv64 * d)), float(np.sum(dv32 * d))
    print(f"V along d: fd {fd:.10e} c128 {g64:.10e} c64 {g32:.10e}")
    assert g64 == pytest.approx(fd, rel=1e-6)
    assert g32 == pytest.approx(fd, rel=1e-4)


@pytest.mark.parametrize("dtype,tol", [(torch.complex128, 1e-12), (torch.complex64, 2e-5)])
@pytest.mark.parametrize("npw,nch,natom,nb", [
    (1, 1, 1, 1), (31, 1, 3, 2), (65, 8, 4, 15), (200, 11, 3, 17), (1030, 18, 8, 33),
    (777, 13, 5, 0)])
def test_position_gradient_at_tile_edges(dtype, tol, npw, nch, natom, nb):
    """qepw_position_gradient (one product over the bands) against the sums
    over dO_c = i B^H (q_c psi) in NumPy: one projector, either side of the 32
    projectors where the tile changes, ragged rows, bands and projectors."""
    from qe_python_amd import _native as nat
    from qe_python_amd import device as dv
    lib = nat.load()
    rng = np.random.default_rng(npw + nb)
    p = nch * natom

    def block(rows, cols):
        return rng.standard_normal((rows, cols)) + 1j * rng.standard_normal((rows, cols))
    psi, proj, coupled = block(npw, nb), block(npw, p), block(p, nb)
    q, f = rng.standard_normal((npw, 3)), rng.standard_normal(nb)
    dev = [torch.from_numpy(np.ascontiguousarray(x.T)).to(DEV).to(dtype)
           for x in (psi, proj, coupled)]
    # the operands as stored (rounded to the block's precision)
    psi, proj, coupled = (x.cpu().numpy().astype(complex).T for x in dev)
    qd, fd = torch.from_numpy(q).to(DEV), torch.from_numpy(f).to(DEV)
    off = torch.arange(0, p + 1, nch, dtype=torch.int32, device=DEV)
    out = torch.full((natom, 3), float("nan"), dtype=torch.float64, device=DEV)
    prec = dv.precision_code(dtype)
    need = lib.qepw_position_gradient_workspace(prec, npw, p, nb)
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)

    def call(size):
        return lib.qepw_position_gradient(
            prec, dev[0].data_ptr(), npw, nb, dev[1].data_ptr(), npw, p, dev[2].data_ptr(), p,
            fd.data_ptr(), qd.data_ptr(), npw, off.data_ptr(), natom, out.data_ptr(),
            ws.data_ptr(), size, dv.stream_handle(torch.device(DEV)))
    with pytest.raises(Exception):
        nat.check(call(need - 1), "short workspace")
    nat.check(call(need), "qepw_position_gradient")
    ref = np.empty((natom, 3))
    for c in range(3):
        d = 1j * proj.conj().T @ (q[:, c, None] * psi)
        t = 2.0 * ((d.conj() * coupled).real @ f)
        ref[:, c] = t.reshape(natom, nch).sum(1)
    # rounding grows with the terms, which may cancel in one force
    scale = max(np.linalg.norm(ref), 2.0 * np.sqrt(2.0 * npw * p * max(nb, 1)) / 10)
    assert np.linalg.norm(out.cpu().numpy() - ref) <= tol * scale


def test_argument_errors(small):
    from qe_python_amd.gradients import band_energy
    s, psi, f, model, _ = small
    p = torch.tensor(psi, device=DEV)
    v = torch.tensor(s.real_potential, device=DEV)
    t = torch.tensor(s.projectors.positions, device=DEV)
    with pytest.raises(ValueError):
        band_energy(model, p[:-1], v, t, f)
    with pytest.raises(ValueError):
        band_energy(model, p, v[:-1], t, f)
    with pytest.raises(ValueError):
        band_energy(model, p, v, t, f[:-1])


def test_position_gradient_checks_its_operands(small):
    """BandEnergyModel.position_gradient refuses operands of another dtype or
    smaller than the sizes that the kernel reads."""
    s, psi, f, model, _ = small
    nb, p = len(f), model.natom * model.nch
    good = {"psi": torch.ones((nb, model.npw), dtype=torch.complex128, device=DEV),
            "proj": torch.ones((p, model.npw), dtype=torch.complex128, device=DEV),
            "coupled": torch.ones((nb, p), dtype=torch.complex128, device=DEV),
            "weights": torch.ones(nb, dtype=torch.float64, device=DEV)}
    assert model.position_gradient(**good).shape == (model.natom, 3)
    bad = [("proj", good["proj"].to(torch.complex64)), ("coupled", good["coupled"].to(torch.complex64)),
           ("weights", good["weights"].float()), ("weights", good["weights"][1:]),
           ("psi", good["psi"][:, 1:]), ("proj", good["proj"][:, 1:]), ("proj", good["proj"][1:]),
           ("coupled", good["coupled"][1:]), ("coupled", good["coupled"][:, 1:])]
    for name, value in bad:
        with pytest.raises(ValueError):
            model.position_gradient(**{**good, name: value})


@pytest.mark.parametrize("dtype,tol", [(torch.complex128, 1e-12), (torch.complex64, 2e-5)])
def test_projector_forces_of_given_derivatives(small, dtype, tol):
    """qepw_projector_forces on the blocks dO_c = i B^H (q_c psi), made with
    BandEnergyModel.scale_rows, against position_gradient, which sums over the
    bands first (bars of the gradients above)."""
    from qe_python_amd import _native as nat
    from qe_python_amd import device as dv
    s, psi, f, model, _ = small
    lib = nat.load()
    nb, p = len(f), model.natom * model.nch
    x = torch.from_numpy(np.ascontiguousarray(psi[model.plan.perm].T)).to(DEV).to(dtype)
    proj = model.projectors(torch.tensor(s.projectors.positions, device=DEV), dtype)
    v = torch.zeros(model.shape[::-1], dtype=dv.real_dtype(dtype), device=DEV)
    _, _, coupled = model.apply(x, v, proj)
    w = torch.tensor(f, device=DEV)
    scaled, blocks = torch.empty_like(x), torch.empty((3, nb, p), dtype=dtype, device=DEV)
    for c in range(3):
        model.scale_rows(x, scaled, s=model.gk[:, c], sstride=3)
        dv.gemm(nat.OP_C, p, nb, model.npw, 1j, proj, scaled, 0.0, blocks[c], model.workspace)
    out = torch.full((model.natom, 3), float("nan"), dtype=torch.float64, device=DEV)
    nat.check(lib.qepw_projector_forces(
        dv.precision_code(dtype), blocks.data_ptr(), p, nb * p, coupled.data_ptr(),
        dv.ld_of(coupled), w.data_ptr(), nb, model.offsets.data_ptr(), model.natom,
        out.data_ptr(), dv.stream_handle(torch.device(DEV))), "qepw_projector_forces")
    assert rel(out.cpu(), model.position_gradient(x, proj, coupled, w).cpu()) < tol


@pytest.mark.parametrize("dtype,tol", [(torch.complex128, 1e-12), (torch.complex64, 2e-5)])
@pytest.mark.parametrize("npw,nch,natom,nb", [(12011, 29, 7, 97), (23847, 10, 25, 127)])
def test_position_gradient_on_large_tiles(dtype, tol, npw, nch, natom, nb):
    """qepw_position_gradient where the product runs on 64 x 64 tiles (the
    workspace holds two partial sums a tile row), with ragged rows, bands and
    projectors, against the sums over dO_c = i B^H (q_c psi) in NumPy."""
    from qe_python_amd import _native as nat
    from qe_python_amd import device as dv
    lib = nat.load()
    rng = np.random.default_rng(npw + nb)
    p = nch * natom

    def block(rows, cols):
        x = rng.standard_normal((cols, rows)) + 1j * rng.standard_normal((cols, rows))
        return torch.from_numpy(x).to(DEV).to(dtype)
    psi, proj, coupled = block(npw, nb), block(npw, p), block(p, nb)
    q, f = rng.standard_normal((npw, 3)), rng.standard_normal(nb)
    qd, fd = torch.from_numpy(q).to(DEV), torch.from_numpy(f).to(DEV)
    off = torch.arange(0, p + 1, nch, dtype=torch.int32, device=DEV)
    out = torch.full((natom, 3), float("nan"), dtype=torch.float64, device=DEV)
    prec, size = dv.precision_code(dtype), 16 if dtype == torch.complex128 else 8
    need = lib.qepw_position_gradient_workspace(prec, npw, p, nb)
    weighted = -(-p * nb * size // 256) * 256
    assert need == weighted + 3 * p * 2 * -(-npw // 64) * 8
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    nat.check(lib.qepw_position_gradient(
        prec, psi.data_ptr(), npw, nb, proj.data_ptr(), npw, p, coupled.data_ptr(), p,
        fd.data_ptr(), qd.data_ptr(), npw, off.data_ptr(), natom, out.data_ptr(),
        ws.data_ptr(), need, dv.stream_handle(torch.device(DEV))), "qepw_position_gradient")
    psi, proj, coupled = (x.cpu().numpy().astype(complex).T for x in (psi, proj, coupled))
    ref = np.empty((natom, 3))
    for c in range(3):
        d = 1j * proj.conj().T @ (q[:, c, None] * psi)
        ref[:, c] = (2.0 * ((d.conj() * coupled).real @ f)).reshape(natom, nch).sum(1)
    scale = max(np.linalg.norm(ref), 2.0 * np.sqrt(2.0 * npw * p * nb) / 10)
    assert np.linalg.norm(out.cpu().numpy() - ref) <= tol * scale
