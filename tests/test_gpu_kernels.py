"""GPU parity of the GEMM and the bandwidth-bound Davidson kernels, called
through the C ABI, against NumPy and the oracle's restatements of the
reference formulas (``oracle.davidson``).

Tolerances: complex128 results within 1e-13 relative (GEMM: 1e-12 of the
product norm); complex64 GEMM within 2e-6 + 1e-7 sqrt(k) of the product
norm (FP32 accumulation over k terms).
"""

import numpy as np
import pytest
import torch

from oracle import davidson as odav

pytestmark = pytest.mark.gpu

DEV = "cuda"


def dev_block(a, dtype=torch.complex128):
    """(rows, cols) host -> (cols, rows) device column-major tensor."""
    return torch.from_numpy(np.ascontiguousarray(np.asarray(a).T)).to(DEV).to(dtype)


def host_block(t):
    return t.cpu().numpy().T


def rand(rng, *shape):
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


@pytest.mark.parametrize("prec", ["c128", "c64"])
@pytest.mark.parametrize("op", ["N", "C", "NB", "CB"])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (5, 7, 3), (64, 64, 16), (65, 130, 37),
                                   (256, 128, 23847), (17, 300, 4000), (2945, 8, 32),
                                   (384, 384, 384), (500, 130, 257), (3, 2, 0),
                                   # one output column: the matrix-vector kernels
                                   (23847, 1, 256), (256, 1, 23847), (300, 1, 5000),
                                   (1, 1, 3000), (70000, 1, 3), (7, 1, 0)])
def test_gemm_matches_numpy(prec, op, m, n, k):
    from qe_python_amd import _native as nat
    from qe_python_amd import device as dv
    rng = np.random.default_rng(m * 1000 + n * 10 + k)
    dtype = torch.complex128 if prec == "c128" else torch.complex64
    a = rand(rng, m, k) if op[0] == "N" else rand(rng, k, m)
    b = rand(rng, n, k) if op.endswith("B") else rand(rng, k, n)
    c = rand(rng, m, n)
    alpha, beta = 0.7 - 0.2j, -0.3 + 0.5j
    ta, tb, tc = dev_block(a, dtype), dev_block(b, dtype), dev_block(c, dtype)
    ws = dv.Workspace(torch.device(DEV))
    code = (nat.OP_N if op[0] == "N" else nat.OP_C) | (nat.OP_BC if op.endswith("B") else 0)
    dv.gemm(code, m, n, k, alpha, ta, tb, beta, tc, ws)
    opa = a if op[0] == "N" else a.conj().T
    b = b.conj().T if op.endswith("B") else b
    if prec == "c64":
        a32, b32, c32 = (x.astype(np.complex64).astype(np.complex128) for x in (opa, b, c))
        ref = alpha * (a32 @ b32) + beta * c32
        # FP32 accumulation over k terms: error grows like sqrt(k) * 2^-24
        tol = 2e-6 + 1e-7 * np.sqrt(k)
    else:
        ref = alpha * (opa @ b) + beta * c
        tol = 1e-12
    got = host_block(tc)
    scale = max(np.linalg.norm(ref), 1e-30)
    assert np.linalg.norm(got - ref) / scale < tol


@pytest.mark.parametrize("prec", ["c128", "c64"])
@pytest.mark.parametrize("op", ["N", "C", "NB", "CB"])
def test_every_gemm_tile_variant_matches_numpy(prec, op):
    """Each tile variant of the GEMM (forced through a tuning rule, with and
    without split K) on shapes that are not multiples of its tiles, against
    NumPy; the rules are cleared and the committed table restored after."""
    import ctypes

    from qe_python_amd import _native as nat
    from qe_python_amd import autotune
    from qe_python_amd import device as dv
    lib = nat.load()
    dtype = torch.complex128 if prec == "c128" else torch.complex64
    code = (nat.OP_N if op[0] == "N" else nat.OP_C) | (nat.OP_BC if op.endswith("B") else 0)
    ws = dv.Workspace(torch.device(DEV))
    try:
        for variant in range(lib.qepw_gemm_variant_count()):
            for m, n, k, splits in [(70, 130, 45, 1), (4100, 97, 33, 1), (200, 61, 3000, 7),
                                    (33, 129, 513, 3)]:
                rng = np.random.default_rng(variant * 100 + m + n + k)
                a = rand(rng, m, k) if op[0] == "N" else rand(rng, k, m)
                b = rand(rng, n, k) if op.endswith("B") else rand(rng, k, n)
                c = rand(rng, m, n)
                alpha, beta = 0.6 + 0.3j, -0.2 + 0.1j
                ta, tb, tc = dev_block(a, dtype), dev_block(b, dtype), dev_block(c, dtype)
                lib.qepw_gemm_clear_rules()
                rng_ = (ctypes.c_int64 * 6)(m, m, n, n, k, k)
                nat.check(lib.qepw_gemm_set_rule(dv.precision_code(dtype), code, rng_,
                                                 variant, splits), "set_rule")
                dv.forget_gemm_plans()
                plan = (ctypes.c_int64 * 4)()
                nat.check(lib.qepw_gemm_plan(dv.precision_code(dtype), code, m, n, k, plan),
                          "plan")
                assert plan[0] == variant
                dv.gemm(code, m, n, k, alpha, ta, tb, beta, tc, ws)
                opa = a if op[0] == "N" else a.conj().T
                bb = b.conj().T if op.endswith("B") else b
                ref = alpha * (opa @ bb) + beta * c
                tol = 1e-12 if prec == "c128" else 2e-6 + 1e-7 * np.sqrt(k)
                err = np.linalg.norm(host_block(tc) - ref) / np.linalg.norm(ref)
                assert err < tol, (variant, m, n, k, splits, err)
    finally:
        lib.qepw_gemm_clear_rules()
        autotune.load_table()


@pytest.mark.parametrize("prec", ["c128", "c64"])
@pytest.mark.parametrize("op", ["N", "C"])
def test_gemm_chosen_plans_at_tile_and_step_edges(prec, op):
    """The built-in tile and split at the edges of tiles (columns 2, 15..17,
    a row more than a tile) and of K steps (depths 1, 15, 17, a split's ragged
    end), against NumPy, with the partials inside the static scratch."""
    import ctypes

    from qe_python_amd import _native as nat
    from qe_python_amd import device as dv
    lib = nat.load()
    dtype = torch.complex128 if prec == "c128" else torch.complex64
    size = 16 if prec == "c128" else 8
    code = nat.OP_N if op == "N" else nat.OP_C
    ws = dv.Workspace(torch.device(DEV))
    for m, n, k in [(65, 2, 1), (33, 15, 15), (1, 16, 17), (129, 17, 2950), (64, 16, 4097),
                    (2951, 16, 31), (4097, 13, 257), (8, 8, 2950), (257, 40, 2049)]:
        rng = np.random.default_rng(m + n + k)
        a = rand(rng, m, k) if op == "N" else rand(rng, k, m)
        b = rand(rng, k, n)
        ta, tb = dev_block(a, dtype), dev_block(b, dtype)
        tc = dev_block(np.zeros((m, n), complex), dtype)
        plan = (ctypes.c_int64 * 4)()
        nat.check(lib.qepw_gemm_plan(dv.precision_code(dtype), code, m, n, k, plan), "plan")
        assert plan[1] == 1 or plan[1] * m * n * size <= lib.qepw_gemm_static_scratch_bytes()
        dv.gemm(code, m, n, k, 1.0, ta, tb, 0.0, tc, ws)
        ref = (a if op == "N" else a.conj().T) @ b
        tol = 1e-12 if prec == "c128" else 2e-6 + 1e-7 * np.sqrt(k)
        err = np.linalg.norm(host_block(tc) - ref) / np.linalg.norm(ref)
        assert err < tol, (m, n, k, list(plan), err)


@pytest.mark.parametrize("prec", ["c128", "c64"])
@pytest.mark.parametrize("op", ["N", "C", "NB", "CB"])
def test_one_column_products_at_their_edges(prec, op):
    """Matrix-vector products either side of 64 rows, 16 columns, and the
    limits where they are split (A b above 384 columns, A^H b above 8192 rows
    with fewer than 64 outputs and above 32768), against NumPy."""
    from qe_python_amd import _native as nat
    from qe_python_amd import device as dv
    dtype = torch.complex128 if prec == "c128" else torch.complex64
    code = (nat.OP_N if op[0] == "N" else nat.OP_C) | (nat.OP_BC if op.endswith("B") else 0)
    ws = dv.Workspace(torch.device(DEV))
    for m, k in [(1, 1), (63, 15), (64, 16), (65, 17), (1000, 256), (72, 72), (63, 8192),
                 (63, 8193), (64, 8193), (1, 9000), (100, 384), (100, 385), (64, 32769)]:
        rng = np.random.default_rng(m + k)
        a = rand(rng, m, k) if op[0] == "N" else rand(rng, k, m)
        b = rand(rng, 1, k) if op.endswith("B") else rand(rng, k, 1)
        c = rand(rng, m, 1)
        ta, tb = dev_block(a, dtype), dev_block(b, dtype)
        bb = b.conj().T if op.endswith("B") else b
        for alpha, beta in ((1.0, 0.0), (0.6 + 0.3j, -0.2 + 0.1j)):
            tc = dev_block(c, dtype)
            dv.gemm(code, m, 1, k, alpha, ta, tb, beta, tc, ws)
            ref = alpha * ((a if op[0] == "N" else a.conj().T) @ bb) + beta * c
            tol = 1e-12 if prec == "c128" else 2e-6 + 1e-7 * np.sqrt(k)
            err = np.linalg.norm(host_block(tc) - ref) / np.linalg.norm(ref)
            assert err < tol, (m, k, err)


def chunked_gemv(a, b, splits, threads):
    """a (rows, k), b (k) complex64 summed in FP32 as a split product does:
    chunks of K, in each the chains of ``threads`` threads and their tree sum;
    the chunks by four waves, and those in order."""
    f = np.float32
    k = len(b)
    chunk = -(-k // splits)
    total = [[np.zeros(len(a), f), np.zeros(len(a), f)] for _ in range(4)]
    for z in range(-(-k // chunk)):
        part = np.zeros((2, threads, len(a)), f)
        for g in range(z * chunk, min(k, (z + 1) * chunk), threads):
            top = min(g + threads, min(k, (z + 1) * chunk))
            x = a[:, g:top].T.astype(complex)
            y = b[g:top, None].astype(complex)
            re = (x.real * y.real - (x.imag * y.imag).astype(f).astype(float)).astype(f)
            im = (x.real * y.imag + (x.imag * y.real).astype(f).astype(float)).astype(f)
            part[0, :top - g] += re
            part[1, :top - g] += im
        h = threads // 2
        while h:
            part[:, :h] += part[:, h:2 * h]
            h //= 2
        for c in range(2):
            total[z % 4][c] += part[c, 0]
    return sum((t[0] for t in total[1:]), total[0][0]) + 1j * sum((t[1] for t in total[1:]),
                                                                  total[0][1]).astype(complex)


@pytest.mark.parametrize("op,m,k,splits,threads", [
    ("N", 2951, 16, 2, 1), ("N", 2951, 168, 21, 1), ("N", 2951, 256, 32, 1), ("N", 2951, 384, 48, 1),
    ("C", 64, 23847, 16, 256), ("C", 64, 10118, 10, 256)])
def test_one_column_products_round_like_split_ones(op, m, k, splits, threads):
    """Unsplit matrix-vector products in FP32 are no further from the exact sums
    than chunks of 8 columns or 1024 rows summed apart (5% for the spread of
    some 700 to 12 000 sums)."""
    from qe_python_amd import _native as nat
    from qe_python_amd import device as dv
    ws = dv.Workspace(torch.device(DEV))
    got = want = 0.0
    for seed in range(2 if op == "N" else 12):
        rng = np.random.default_rng(seed)
        a, b = rand(rng, m, k).astype(np.complex64), rand(rng, k, 1).astype(np.complex64)
        tc = dev_block(np.zeros((m, 1)), torch.complex64)
        dv.gemm(nat.OP_N if op == "N" else nat.OP_C, m, 1, k, 1.0,
                dev_block(a if op == "N" else a.conj().T, torch.complex64),
                dev_block(b, torch.complex64), 0.0, tc, ws)
        exact = (a.astype(complex) @ b.astype(complex))[:, 0]
        got += np.linalg.norm(host_block(tc)[:, 0] - exact) ** 2
        want += np.linalg.norm(chunked_gemv(a, b[:, 0], splits, threads) - exact) ** 2
    assert got <= 1.05 ** 2 * want, (got / want) ** 0.5


@pytest.mark.parametrize("op,m,k", [("C", (1 << 22) + 3, 2), ("N", (1 << 28) + 5, 1)])
def test_one_column_products_of_the_most_rows(op, m, k):
    """Outputs beyond 2^32 work-items of the workgroups of 1024 that short
    matrix-vector products run in (small integers: exact)."""
    from qe_python_amd import _native as nat
    from qe_python_amd import device as dv
    ramp = torch.arange(m, device=DEV) % 1000
    a = torch.stack([ramp - 3 * j for j in range(k)]).to(torch.complex64)   # (k, m)
    b = torch.arange(1, k + 1, device=DEV).to(torch.complex64)[None]
    ref = sum((j + 1) * (ramp - 3 * j) for j in range(k))
    c = torch.full((1, m), 7.0 + 0j, dtype=torch.complex64, device=DEV)
    if op == "C":
        a = a.T.contiguous()
    dv.gemm(nat.OP_C if op == "C" else nat.OP_N, m, 1, k, 1.0, a, b, 0.0, c,
            dv.Workspace(torch.device(DEV)))
    assert torch.equal(c[0].real.long(), ref) and not torch.any(c[0].imag)


def test_gemm_in_a_workspace_of_fixed_size():
    """A product whose planned partials exceed the static scratch runs in the
    Rayleigh-Ritz steps' workspace with fewer splits; less than 21 splits of
    320 x 320 (the choice that needs no search) is refused."""
    from qe_python_amd import _native as nat
    from qe_python_amd import device as dv
    lib = nat.load()
    m, k = 320, 24000
    rng = np.random.default_rng(3)
    a = rand(rng, k, m)
    ta = dev_block(a, torch.complex128)
    tc = dev_block(np.zeros((m, m), complex), torch.complex128)
    ws = torch.empty(max(lib.qepw_rr_workspace(m), lib.qepw_gemm_workspace(
        nat.C128, nat.OP_C, m, m, k)), dtype=torch.uint8, device=DEV)
    import ctypes
    one, zero = (ctypes.c_double * 2)(1.0, 0.0), (ctypes.c_double * 2)(0.0, 0.0)
    ref = a.conj().T @ a
    for size in (lib.qepw_gemm_workspace(nat.C128, nat.OP_C, m, m, k), 21 * m * m * 16):
        nat.check(lib.qepw_gemm(nat.C128, nat.OP_C, m, m, k, one, ta.data_ptr(), k,
                                ta.data_ptr(), k, zero, tc.data_ptr(), m, ws.data_ptr(), size,
                                dv.stream_handle(torch.device(DEV))), "qepw_gemm")
        err = np.linalg.norm(host_block(tc) - ref) / np.linalg.norm(ref)
        assert err < 1e-12, (size, err)
    with pytest.raises(Exception):
        nat.check(lib.qepw_gemm(nat.C128, nat.OP_C, m, m, k, one, ta.data_ptr(), k,
                                ta.data_ptr(), k, zero, tc.data_ptr(), m, ws.data_ptr(),
                                12 * m * m * 16, dv.stream_handle(torch.device(DEV))), "short")


@pytest.mark.parametrize("prec,m,n,k", [
    ("c64", 384, 160, 23847), ("c64", 384, 150, 35769), ("c64", 384, 192, 35769),
    ("c64", 512, 40, 23847), ("c128", 512, 96, 47692), ("c128", 128, 128, 23847)])
def test_gemm_rounds_like_short_chains(prec, m, n, k):
    """A^H B against exact sums (operands of 18 bits, for complex128 of two such
    halves, whose products add up exactly in float64).  A sum of c terms of
    random sign in one accumulator is about sqrt(c / 2) roundings off; chains of
    at most 256 columns, the sum of a split's chains and the sum of the splits
    (by four waves) make sqrt(256 / 2 + chunk / 256 / 2 + splits / 8)."""
    import ctypes

    from qe_python_amd import _native as nat
    from qe_python_amd import device as dv
    lib = nat.load()
    dtype = torch.complex128 if prec == "c128" else torch.complex64
    rng = np.random.default_rng(m + n)

    def halves(rows):
        x = rng.uniform(-1.0, 1.0, (k, rows))
        hi = np.round(x * 2.0 ** 17) / 2.0 ** 17
        lo = np.round((x - hi) * 2.0 ** 34) / 2.0 ** 34
        return hi, lo if prec == "c128" else np.zeros_like(lo)

    def dot(x, y):   # x^T y as a sum and what it lacks
        return x[0].T @ y[0], (x[0].T @ y[1] + x[1].T @ y[0]) + x[1].T @ y[1]
    ar, ai, br, bi = halves(m), halves(m), halves(n), halves(n)
    ta, tb = dev_block(sum(ar) + 1j * sum(ai), dtype), dev_block(sum(br) + 1j * sum(bi), dtype)
    tc = dev_block(np.zeros((m, n), complex), dtype)
    dv.gemm(nat.OP_C, m, n, k, 1.0, ta, tb, 0.0, tc, dv.Workspace(torch.device(DEV)))
    got = host_block(tc).astype(complex)
    (rr, rl), (ii, il), (ri, ril), (ir, irl) = dot(ar, br), dot(ai, bi), dot(ar, bi), dot(ai, br)
    err = np.hypot(np.linalg.norm((got.real - (rr + ii)) - (rl + il)),
                   np.linalg.norm((got.imag - (ri - ir)) - (ril - irl))) / np.linalg.norm(got)
    plan = (ctypes.c_int64 * 4)()
    nat.check(lib.qepw_gemm_plan(dv.precision_code(dtype), nat.OP_C, m, n, k, plan), "plan")
    chunk = k / plan[1]
    unit = 2.0 ** -53 if prec == "c128" else 2.0 ** -24
    bound = unit * np.sqrt(256 / 2 + chunk / 256 / 2 + plan[1] / 8)
    assert err < bound, (list(plan), err, bound)


@pytest.mark.parametrize("m,n,k", [(512, 192, 23847), (250, 384, 40001), (520, 1040, 5001),
                                   (64, 768, 23847)])
def test_gemm_bits_do_not_depend_on_the_workspace(m, n, k):
    """Products A^H B whose planned partials exceed the static scratch (FP64's):
    in the quoted workspace, in 32 MiB and in the static scratch they give the
    same bits (panels of rows or, one tile high, columns with the same plan)."""
    import ctypes

    from qe_python_amd import _native as nat
    from qe_python_amd import device as dv
    lib = nat.load()
    dtype, code = torch.complex128, nat.C128
    limit = int(lib.qepw_gemm_static_scratch_bytes())
    rng = np.random.default_rng(m + n)
    a, b, c = rand(rng, k, m), rand(rng, k, n), rand(rng, m, n)
    ta, tb = dev_block(a, dtype), dev_block(b, dtype)
    alpha, beta = (ctypes.c_double * 2)(0.5, -0.25), (ctypes.c_double * 2)(1.0, 0.5)
    need = int(lib.qepw_gemm_workspace(code, nat.OP_C, m, n, k))
    assert need > limit
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    out = []
    for size in (need, limit, None):
        tc = dev_block(c, dtype)
        head = (code, nat.OP_C, m, n, k, alpha, ta.data_ptr(), k, tb.data_ptr(), k, beta,
                tc.data_ptr(), m)
        stream = dv.stream_handle(torch.device(DEV))
        if size is None:
            nat.check(lib.qepw_gemm_static(*head, stream), "qepw_gemm_static")
        else:
            nat.check(lib.qepw_gemm(*head, ws.data_ptr(), size, stream), "qepw_gemm")
        out.append(host_block(tc))
    ref = (0.5 - 0.25j) * (a.conj().T @ b) + (1.0 + 0.5j) * c
    assert np.linalg.norm(out[0] - ref) / np.linalg.norm(ref) < 1e-12
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])


def test_gemm_unsplit_without_a_workspace():
    """A shallow product that the search splits still runs without a
    workspace."""
    import ctypes

    from qe_python_amd import _native as nat
    from qe_python_amd import device as dv
    lib = nat.load()
    m, n, k = 168, 96, 168
    assert int(lib.qepw_gemm_workspace(nat.C64, nat.OP_N, m, n, k)) > 0
    rng = np.random.default_rng(7)
    a, b = rand(rng, m, k), rand(rng, k, n)
    ta, tb = dev_block(a, torch.complex64), dev_block(b, torch.complex64)
    tc = dev_block(np.zeros((m, n), complex), torch.complex64)
    one, zero = (ctypes.c_double * 2)(1.0, 0.0), (ctypes.c_double * 2)(0.0, 0.0)
    nat.check(lib.qepw_gemm(nat.C64, nat.OP_N, m, n, k, one, ta.data_ptr(), m, tb.data_ptr(), k,
                            zero, tc.data_ptr(), m, None, 0,
                            dv.stream_handle(torch.device(DEV))), "qepw_gemm")
    err = np.linalg.norm(host_block(tc) - a @ b) / np.linalg.norm(a @ b)
    assert err < 2e-6 + 1e-7 * np.sqrt(k)


def test_gemm_split_k_is_deterministic():
    from qe_python_amd import _native as nat
    from qe_python_amd import device as dv
    rng = np.random.default_rng(5)
    a, b = rand(rng, 23847, 128), rand(rng, 23847, 160)
    ta, tb = dev_block(a), dev_block(b)
    ws = dv.Workspace(torch.device(DEV))
    outs = []
    for _ in range(2):
        tc = torch.empty((160, 128), dtype=torch.complex128, device=DEV)
        dv.gemm(nat.OP_C, 128, 160, 23847, 1.0, ta, tb, 0.0, tc, ws)
        outs.append(tc.cpu().numpy())
    assert np.array_equal(outs[0], outs[1])


def test_gemv_beta_zero_ignores_nan_output_and_is_deterministic():
    from qe_python_amd import _native as nat
    from qe_python_amd import device as dv
    rng = np.random.default_rng(10)
    a, b = rand(rng, 23847, 256), rand(rng, 23847, 1)
    ws = dv.Workspace(torch.device(DEV))
    outs = []
    for _ in range(2):
        tc = torch.full((1, 256), float("nan"), dtype=torch.complex128, device=DEV)
        dv.gemm(nat.OP_C, 256, 1, 23847, 1.0, dev_block(a), dev_block(b), 0.0, tc, ws)
        outs.append(host_block(tc))
    np.testing.assert_allclose(outs[0], a.conj().T @ b, rtol=1e-12, atol=1e-12)
    assert np.array_equal(outs[0], outs[1])


def test_gemm_beta_zero_ignores_nan_output():
    from qe_python_amd import _native as nat
    from qe_python_amd import device as dv
    rng = np.random.default_rng(9)
    a, b = rand(rng, 40, 20), rand(rng, 20, 10)
    tc = torch.full((10, 40), float("nan"), dtype=torch.complex128, device=DEV)
    dv.gemm(nat.OP_N, 40, 10, 20, 1.0, dev_block(a), dev_block(b), 0.0, tc,
            dv.Workspace(torch.device(DEV)))
    np.testing.assert_allclose(host_block(tc), a @ b, rtol=1e-13, atol=1e-13)


@pytest.fixture(scope="module")
def blocks():
    rng = np.random.default_rng(11)
    npw, nb = 3001, 9
    return rng, npw, nb, rand(rng, npw, nb), rand(rng, npw, nb)


def test_column_norms_and_inner_products(blocks):
    from qe_python_amd import device as dv
    rng, npw, nb, x, y = blocks
    sq = dv.column_squared_norms(dev_block(x), npw).cpu().numpy()
    np.testing.assert_allclose(sq, odav.column_squared_norms(x), rtol=1e-13)
    ip = dv.column_inner_products(dev_block(x), dev_block(y), npw).cpu().numpy()
    np.testing.assert_allclose(ip[0::2] + 1j * ip[1::2], np.einsum("gb,gb->b", x.conj(), y),
                               rtol=1e-13)
    sq32 = dv.column_squared_norms(dev_block(x, torch.complex64), npw).cpu().numpy()
    x32 = x.astype(np.complex64).astype(np.complex128)
    np.testing.assert_allclose(sq32, odav.column_squared_norms(x32), rtol=1e-13)


def test_subtract_energies_precondition_normalize_restart(blocks):
    from qe_python_amd import device as dv
    rng, npw, nb, x, r = blocks
    e = rng.uniform(-1, 1, nb)
    diag = rng.uniform(0, 20, npw)
    td = dev_block(r)
    dv.subtract_band_energies(td, dev_block(x), torch.from_numpy(e).to(DEV), npw)
    np.testing.assert_allclose(host_block(td), r - x * e[None, :], rtol=1e-14, atol=1e-14)

    cols = np.array([0, 3, 4, 8], dtype=np.int32)
    out = torch.empty((len(cols), npw), dtype=torch.complex128, device=DEV)
    dv.qe_precondition(dev_block(r), torch.from_numpy(cols).to(DEV),
                       torch.from_numpy(e[cols]).to(DEV), torch.from_numpy(diag).to(DEV),
                       out, npw)
    np.testing.assert_allclose(host_block(out), odav.qe_precondition(r[:, cols], e[cols], diag),
                               rtol=1e-14)

    sq = odav.column_squared_norms(r)
    sel = np.array([1, 2, 7], dtype=np.int32)
    dst = torch.empty((len(sel), npw), dtype=torch.complex128, device=DEV)
    dv.normalize_selected_columns(dev_block(r), torch.from_numpy(sq).to(DEV),
                                  torch.from_numpy(sel).to(DEV), dst, npw)
    np.testing.assert_allclose(host_block(dst), r[:, sel] / np.sqrt(sq[sel])[None, :],
                               rtol=1e-14)

    hv = torch.empty((nb, npw), dtype=torch.complex128, device=DEV)
    dv.restart_applied(dev_block(x), dev_block(r), torch.from_numpy(e).to(DEV), hv, npw)
    np.testing.assert_allclose(host_block(hv), x * e[None, :] + r, rtol=1e-14, atol=1e-14)


def test_permute_rows_round_trip_and_cast(blocks):
    from qe_python_amd import device as dv
    rng, npw, nb, x, _ = blocks
    perm = rng.permutation(npw).astype(np.int32)
    tp = torch.from_numpy(perm).to(DEV)
    g = torch.empty((nb, npw), dtype=torch.complex128, device=DEV)
    dv.permute_rows(0, tp, dev_block(x), g, npw)
    assert np.array_equal(host_block(g), x[perm])
    back = torch.empty_like(g)
    dv.permute_rows(1, tp, g, back, npw)
    assert np.array_equal(host_block(back), x)
    g32 = torch.empty((nb, npw), dtype=torch.complex64, device=DEV)
    dv.permute_rows(0, tp, dev_block(x), g32, npw)
    assert np.array_equal(host_block(g32), x[perm].astype(np.complex64))


def test_projector_diagonal_accumulation():
    from qe_python_amd import device as dv
    rng = np.random.default_rng(2)
    npw, nch = 777, 5
    beta, coupled = rand(rng, npw, nch), rand(rng, npw, nch)
    acc = torch.ones(npw, dtype=torch.float64, device=DEV)
    dv.accumulate_projector_diagonal(dev_block(coupled), dev_block(beta), npw, 3.0, acc)
    expect = 1.0 + 3.0 * np.real(np.einsum("gi,gi->g", coupled, beta.conj()))
    np.testing.assert_allclose(acc.cpu().numpy(), expect, rtol=1e-13)
