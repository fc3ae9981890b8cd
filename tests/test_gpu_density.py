"""GPU parity of the SCF's density accumulation (``sum_band``):
``LocalPotentialWorkspace.accumulate_density`` (reference:
``qepy_pw/basis.py:1210-1282``, kernel ``_native_fft.pyx:2592-2648``, caller
``pw/scf.py:1382-1451``) against the oracle's restatement on the small and
medium workloads, accumulation into an existing grid, device in/out, the
reference's argument errors, and a Hamiltonian sharing the workspace's plan.
"""

import numpy as np
import pytest

from oracle.hpsi import OracleHamiltonian, accumulate_density, linear_slots
from qe_python_amd.synthetic import make_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,nb", [("small", 16), ("medium", 24), ("cell54", 16),
                                     ("cell64", 16)])
def test_density_matches_oracle(name, nb):
    from qe_python_amd.basis import LocalPotentialWorkspace
    s = make_system(name)
    rng = np.random.default_rng(41)
    coeff = s.trial[:, :nb]
    w = rng.uniform(0.1, 2.0, nb)
    ref = accumulate_density(coeff, w, linear_slots(s.basis.indices, s.shape), s.shape)
    ws = LocalPotentialWorkspace(s.basis.indices, s.shape)
    start = rng.standard_normal(s.shape)
    rho = start.copy()
    ws.accumulate_density(rho, coeff, w)
    np.testing.assert_allclose(rho - start, ref, rtol=0, atol=1e-12 * np.abs(ref).max())
    # the SCF's normalisation by the volume only rescales the weights
    rho2 = np.zeros(s.shape)
    ws.accumulate_density(rho2, coeff, w / 7.0)
    np.testing.assert_allclose(rho2, ref / 7.0, rtol=0, atol=1e-12 * np.abs(ref).max())


def test_density_device_tensors_and_errors():
    import torch

    from qe_python_amd.basis import LocalPotentialWorkspace
    from qe_python_amd.diagonalization import PlaneWaveHamiltonian
    s = make_system("small")
    ws = LocalPotentialWorkspace(s.basis, s.shape)
    coeff = s.trial[:, :5]
    w = np.linspace(0.5, 1.5, 5)
    ref = accumulate_density(coeff, w, linear_slots(s.basis.indices, s.shape), s.shape)
    rho = torch.zeros(s.shape, dtype=torch.float64, device="cuda")
    ws.accumulate_density(rho, torch.from_numpy(coeff).cuda(), w)
    np.testing.assert_allclose(rho.cpu().numpy(), ref, rtol=0, atol=1e-12 * np.abs(ref).max())
    with pytest.raises(ValueError, match="disagree"):
        ws.accumulate_density(np.zeros(s.shape), coeff, w[:4])
    with pytest.raises(ValueError, match="wrong local shape"):
        ws.accumulate_density(np.zeros((4, 4, 4)), coeff, w)
    # a Hamiltonian built on the workspace shares its plan and matches the oracle
    beta, coup, diag = s.packed_term()
    from qe_python_amd.diagonalization import PackedProjectorTerm
    ham = PlaneWaveHamiltonian(s.basis, s.potential_g, (PackedProjectorTerm(beta, coup, diag),),
                               local_workspace=ws, real_potential=s.real_potential)
    assert ham.plan is ws.plan
    from types import SimpleNamespace
    oh = OracleHamiltonian(s.basis.indices, s.basis.kinetic, s.shape, s.real_potential,
                           (SimpleNamespace(beta=beta, coupling=coup, diagonal=diag),),
                           potential_average=float(np.real(s.potential_g.flat[0])))
    got, want = ham.apply(coeff), oh.apply(coeff)
    assert np.linalg.norm(got - want) <= 1e-12 * np.linalg.norm(want)


def test_density_at_a_general_kpoint():
    """A k-point basis shifts the sphere (other sticks and active columns): the
    density of its bands against the oracle, and the SCF identity
    sum_r V(r) rho(r) / N = sum_b w_b <psi_b|V_loc psi_b> with the device
    Hamiltonian's local part."""
    from qe_python_amd.basis import LocalPotentialWorkspace
    s = make_system("medium", kpoint=np.array([0.21, 0.07, 0.33]))
    nb = 16
    rng = np.random.default_rng(43)
    coeff = s.trial[:, :nb]
    w = rng.uniform(0.1, 2.0, nb)
    ref = accumulate_density(coeff, w, linear_slots(s.basis.indices, s.shape), s.shape)
    ws = LocalPotentialWorkspace(s.basis.indices, s.shape)
    rho = np.zeros(s.shape)
    ws.accumulate_density(rho, coeff, w)
    np.testing.assert_allclose(rho, ref, rtol=0, atol=1e-12 * np.abs(ref).max())
    local = OracleHamiltonian(s.basis.indices, np.zeros(s.npw), s.shape, s.real_potential)
    expect = np.sum(w * np.real(np.einsum("gb,gb->b", coeff.conj(), local.apply(coeff))))
    got = np.sum(s.real_potential * rho) / rho.size
    assert abs(got - expect) <= 1e-11 * abs(expect)


@pytest.mark.parametrize("shape", [(128, 128, 20), (144, 150, 16)])
def test_density_on_split_stage_grids(shape):
    """Planes no workgroup can hold in FP64 (128 x 128 and 144 x 150) take
    the split plane stage in the density too: FP64 and FP32 against the
    oracle, and the V-rho identity sum_r V rho / N = sum_b w_b <psi_b|V psi_b>
    against the same grid's h_psi."""
    import torch

    from qe_python_amd.basis import LocalPotentialWorkspace, make_bases
    from qe_python_amd.diagonalization import PlaneWaveHamiltonian
    rng = np.random.default_rng(32)
    reciprocal = 2.0 * np.pi / 12.0 * np.eye(3)
    basis = make_bases(reciprocal, np.array([0.1, 0.3, 0.2]), 8.0)[0]
    nb = 5
    coeff = rng.standard_normal((len(basis), nb)) + 1j * rng.standard_normal((len(basis), nb))
    w = rng.uniform(0.2, 2.0, nb)
    ref = accumulate_density(coeff, w, linear_slots(basis.indices, shape), shape)
    ws = LocalPotentialWorkspace(basis.indices, shape)
    rho = np.zeros(shape)
    ws.accumulate_density(rho, coeff, w)
    np.testing.assert_allclose(rho, ref, rtol=0, atol=1e-12 * np.abs(ref).max())
    from qe_python_amd.diagonalization import _upload_block
    dev = torch.device("cuda", torch.cuda.current_device())
    psi32 = _upload_block(coeff, ws.plan.perm_device, ws.npw, dev, torch.complex64)
    out32 = torch.empty(shape[::-1], dtype=torch.float64, device=dev)
    ws._accumulate_device(psi32, torch.from_numpy(w).to(dev), out32)
    np.testing.assert_allclose(out32.permute(2, 1, 0).cpu().numpy(), ref, rtol=0,
                               atol=2e-6 * np.abs(ref).max())
    vr = rng.uniform(-1.0, 0.5, shape)
    ham = PlaneWaveHamiltonian(basis, np.zeros(shape, complex), (), real_potential=vr,
                               local_workspace=ws)
    hx = ham.apply(coeff) - coeff * np.asarray(basis.kinetic)[:, None]
    lhs = float(np.sum(vr * rho)) / np.prod(shape)
    rhs = float(np.sum(w * np.real(np.sum(coeff.conj() * hx, axis=0))))
    assert lhs == pytest.approx(rhs, rel=1e-11)


@pytest.mark.parametrize("shape,dense", [
    ((16, 16, 20), False), ((60, 60, 16), False), ((72, 72, 16), False), ((75, 75, 16), False),
    ((80, 80, 16), False), ((90, 90, 16), False), ((96, 96, 16), False), ((40, 40, 16), True),
    ((72, 72, 16), True), ((80, 80, 16), True), ((18, 16, 20), False), ((48, 60, 20), False),
    ((90, 108, 16), False), ((108, 120, 16), False), ((30, 128, 16), False),
    ((192, 50, 16), False), ((24, 30, 20), True)])
def test_density_of_any_two_lengths(shape, dense):
    """The density's plane kernels over square and rectangular planes, with and
    without exchange lines of their own, for spheres that reach the ends of the
    pruned slots and bases that fill the axes, with one band and a number that
    no slice count divides, against NumPy's FFT."""
    import torch

    from qe_python_amd import device as dv
    from qe_python_amd.basis import LocalPotentialWorkspace
    rng = np.random.default_rng(53)
    ax = [np.arange(-((n - 1) // 2), n // 2 + 1) if dense
          else np.arange(-((n + 1) // 4), (n - 1) // 4 + 1) for n in shape]
    m = np.stack(np.meshgrid(*ax, indexing="ij"), -1).reshape(-1, 3)
    if not dense:   # an ellipsoid reaching the ends of each axis
        half = np.array([len(a) / 2.0 for a in ax])
        mid = np.array([(a[0] + a[-1]) / 2.0 for a in ax])
        m = m[(((m - mid) / half) ** 2).sum(1) <= 1.0]
    m = m[rng.permutation(len(m))].astype(np.int32)
    ws = LocalPotentialWorkspace(m, shape)
    for nb in (1, 19):
        x = rng.standard_normal((len(m), nb)) + 1j * rng.standard_normal((len(m), nb))
        w = rng.uniform(0.1, 2.0, nb)
        ref = np.zeros(shape)
        for b in range(nb):
            grid = np.zeros(shape, complex)
            grid[tuple((m % np.array(shape)).T)] = x[:, b]
            ref += w[b] * np.abs(np.fft.ifftn(grid, norm="forward")) ** 2
        rho = np.zeros(shape)
        ws.accumulate_density(rho, x, w)
        np.testing.assert_allclose(rho, ref, rtol=0, atol=1e-12 * np.abs(ref).max())
        dev = torch.device("cuda", torch.cuda.current_device())
        from qe_python_amd.diagonalization import _upload_block
        psi32 = _upload_block(x, ws.plan.perm_device, ws.npw, dev, torch.complex64)
        out32 = torch.empty(shape[::-1], dtype=torch.float64, device=dev)
        ws._accumulate_device(psi32, torch.from_numpy(w).to(dev), out32)
        assert dv.real_dtype(psi32.dtype) == torch.float32
        np.testing.assert_allclose(out32.permute(2, 1, 0).cpu().numpy(), ref, rtol=0,
                                   atol=2e-6 * np.abs(ref).max())


@pytest.mark.parametrize("shape,dtype", [
    ((96, 128, 16), "complex128"), ((75, 108, 16), "complex128"), ((120, 128, 16), "complex128"),
    ((160, 120, 16), "complex64"), ((144, 144, 16), "complex64"), ((72, 75, 16), "complex64")])
def test_density_in_the_quoted_workspace(shape, dtype):
    """qepw_accumulate_density in exactly the bytes that
    qepw_accumulate_density_workspace quotes, where the plane stage and the
    density run on the same kernels and where they do not, against NumPy."""
    import torch

    from qe_python_amd import _native as nat
    from qe_python_amd import device as dv
    from qe_python_amd.basis import LocalPotentialWorkspace
    from qe_python_amd.diagonalization import _upload_block
    lib = nat.load()
    dev = torch.device("cuda", torch.cuda.current_device())
    torch_type = getattr(torch, dtype)
    rng = np.random.default_rng(59)
    ax = [np.arange(-((n + 1) // 4), (n - 1) // 4 + 1) for n in shape]
    m = np.stack(np.meshgrid(*ax, indexing="ij"), -1).reshape(-1, 3)
    half = np.array([len(a) / 2.0 for a in ax])
    mid = np.array([(a[0] + a[-1]) / 2.0 for a in ax])
    m = m[(((m - mid) / half) ** 2).sum(1) <= 1.0].astype(np.int32)
    plan = LocalPotentialWorkspace(m, shape).plan
    prec = dv.precision_code(torch_type)
    for nb in (1, 3):
        x = rng.standard_normal((len(m), nb)) + 1j * rng.standard_normal((len(m), nb))
        w = rng.uniform(0.1, 2.0, nb)
        psi = _upload_block(x, plan.perm_device, len(m), dev, torch_type)
        wd = torch.from_numpy(w).to(dev)
        out = torch.empty(shape[::-1], dtype=torch.float64, device=dev)
        need = lib.qepw_accumulate_density_workspace(plan.handle, prec, nb)
        ws = torch.empty(need, dtype=torch.uint8, device=dev)
        nat.check(lib.qepw_accumulate_density(
            plan.handle, prec, psi.data_ptr(), dv.ld_of(psi), nb, wd.data_ptr(), 1.0,
            out.data_ptr(), ws.data_ptr(), need, dv.stream_handle(dev)),
            "qepw_accumulate_density")
        ref = np.zeros(shape)
        for b in range(nb):
            grid = np.zeros(shape, complex)
            grid[tuple((m % np.array(shape)).T)] = x[:, b]
            ref += w[b] * np.abs(np.fft.ifftn(grid, norm="forward")) ** 2
        tol = 1e-12 if dtype == "complex128" else 2e-6
        np.testing.assert_allclose(out.permute(2, 1, 0).cpu().numpy(), ref, rtol=0,
                                   atol=tol * np.abs(ref).max())
