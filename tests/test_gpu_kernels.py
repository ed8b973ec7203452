"""Per-kernel GPU test of the quaternion GEMM on FP64 MFMA (zq_qgemm, the
kernel of the trailing update and of the back-transform) against a plain
FP64 product: quaternion matrices are multiplied through their 2 x 2
complex-block embedding H = [[A, -conj B], [B, conj A]] with numpy, a
representation independent of the kernel's 4-vector L(q) expansion."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _rand_q(rng, r, c):
    """A random quaternion matrix as its complex components (a, b)."""
    return (rng.normal(size=(r, c)) + 1j * rng.normal(size=(r, c)),
            rng.normal(size=(r, c)) + 1j * rng.normal(size=(r, c)))


def _embed(a, b):
    return np.block([[a, -b.conj()], [b, a.conj()]])


def _unembed(H, r, c):
    return H[:r, :c], H[r:2 * r, :c]


def _pack(a, b, ld):
    """Column-major device layout: element (i, j) at 4 doubles (Re a, Im a, Re b, Im b), leading dimension ld."""
    r, c = a.shape
    out = np.zeros((c, ld, 4))
    out[:, :r, 0] = a.real.T
    out[:, :r, 1] = a.imag.T
    out[:, :r, 2] = b.real.T
    out[:, :r, 3] = b.imag.T
    return out


def _unpack(buf, r, c):
    a = buf[:c, :r, 0].T + 1j * buf[:c, :r, 1].T
    b = buf[:c, :r, 2].T + 1j * buf[:c, :r, 3].T
    return a, b


def _ct(a, b):
    """Quaternion conjugate transpose of (a, b): elements (conj a, -b), transposed."""
    return a.conj().T, -b.T


# alpha = -1, beta = 1 are the trailing update's and the back-transform's.
@pytest.mark.parametrize("m,n,k,ta,tb,lower,alpha,beta", [
    (1, 1, 1, "N", "N", False, -0.75, 1.25), (37, 53, 19, "N", "N", False, -0.75, 1.25),
    (64, 64, 64, "N", "C", True, -0.75, 1.25), (100, 80, 70, "C", "N", False, -0.75, 1.25),
    (129, 200, 64, "C", "C", False, -0.75, 1.25), (300, 300, 64, "N", "C", True, -0.75, 1.25),
    (513, 129, 257, "N", "N", False, -0.75, 1.25), (70, 65, 0, "N", "N", False, -0.75, 1.25),
    (300, 300, 64, "N", "C", True, -1.0, 1.0), (513, 129, 128, "N", "N", False, -1.0, 1.0),
    (200, 100, 24, "N", "N", False, 1.0, -0.5), (129, 200, 40, "C", "N", False, 1.0, 2.0),
    (64, 64, 33, "N", "C", True, -1.0, 1.0), (1100, 70, 128, "N", "N", False, -1.0, 1.0),
    (90, 90, 256, "C", "C", True, 1.0, 0.0), (1030, 1040, 128, "N", "N", False, -1.0, 1.0),
    (1500, 1500, 64, "N", "C", True, -1.0, 1.0)])
@pytest.mark.parametrize("t64", [0, 1])
def test_qgemm_against_complex_embedding(gpu_ctx, m, n, k, ta, tb, lower, alpha, beta, t64):
    """Small products (16 x 32 tiles whatever t64 is) and two with more than two
    32 x 64 tiles per compute unit: t64 = 1 gives them 64-row tiles, 0 (the
    context's default threshold) 32-row ones."""
    import torch
    _say(f"case: qgemm m={m} n={n} k={k} {ta}{tb} lower={lower} alpha={alpha} beta={beta} t64={t64}")
    rng = np.random.default_rng(m * 1000 + n + k)
    Ar, Ac = (k, m) if ta == "C" else (m, k)
    Br, Bc = (n, k) if tb == "C" else (k, n)
    A = _rand_q(rng, Ar, Ac)
    B = _rand_q(rng, Br, Bc)
    C = _rand_q(rng, m, n)
    opA = _ct(*A) if ta == "C" else A
    opB = _ct(*B) if tb == "C" else B
    HA, HB, HC = _embed(*opA), _embed(*opB), _embed(*C)
    ref = _unembed(alpha * (HA @ HB) + beta * HC if k > 0 else beta * HC, m, n)
    lda, ldb, ldc = Ar + 3, Br + 1, m + 2
    dA = torch.from_numpy(_pack(*A, lda)).cuda()
    dB = torch.from_numpy(_pack(*B, ldb)).cuda()
    dC = torch.from_numpy(_pack(*C, ldc)).cuda()
    before = dC.clone()
    torch.cuda.synchronize()
    gpu_ctx.set_tile_shape(-1, t64)
    try:
        rc = gpu_ctx.qgemm_device(ta, tb, m, n, k, alpha, dA.data_ptr(), lda, dB.data_ptr(), ldb, beta, dC.data_ptr(),
                                  ldc, lower)
        gpu_ctx.synchronize()
    finally:
        gpu_ctx.set_tile_shape(-1, 0)
    assert rc == 0
    got = _unpack(dC.cpu().numpy(), m, n)
    scale = max(1.0, np.sqrt(k)) * 8.0
    mask = np.tril(np.ones((m, n), dtype=bool)) if lower else np.ones((m, n), dtype=bool)
    for g, r in zip(got, ref):
        assert np.abs(g - r)[mask].max() <= 1e-14 * scale, np.abs(g - r)[mask].max()
    if lower:   # the strict upper triangle is left as it was
        old = _unpack(before.cpu().numpy(), m, n)
        for g, o in zip(got, old):
            assert np.array_equal(g[~mask], o[~mask])
    # padding rows beyond m of every column are untouched
    assert torch.equal(dC[:, m:, :], before[:, m:, :])


@pytest.mark.parametrize("m,n,k,ta,tb,lower", [(1030, 1040, 128, "N", "N", False), (1500, 1500, 64, "N", "C", True),
                                               (1100, 1024, 96, "C", "N", False)])
def test_qgemm_tile_rows_change_no_result(gpu_ctx, m, n, k, ta, tb, lower):
    """The same product with 32-row and with 64-row tiles is bitwise equal
    (a batch and a solo solve may pick different tile rows for one problem)."""
    import torch
    _say(f"case: qgemm tile rows m={m} n={n} k={k} {ta}{tb} lower={lower}")
    rng = np.random.default_rng(m + 7 * k)
    Ar, Ac = (k, m) if ta == "C" else (m, k)
    Br, Bc = (n, k) if tb == "C" else (k, n)
    dA = torch.from_numpy(_pack(*_rand_q(rng, Ar, Ac), Ar)).cuda()
    dB = torch.from_numpy(_pack(*_rand_q(rng, Br, Bc), Br)).cuda()
    C0 = torch.from_numpy(_pack(*_rand_q(rng, m, n), m)).cuda()
    outs = []
    for t64 in (0, 1):
        dC = C0.clone()
        torch.cuda.synchronize()
        gpu_ctx.set_tile_shape(-1, t64)
        try:
            assert gpu_ctx.qgemm_device(ta, tb, m, n, k, -1.0, dA.data_ptr(), Ar, dB.data_ptr(), Br, 1.0,
                                        dC.data_ptr(), m, lower) == 0
            gpu_ctx.synchronize()
        finally:
            gpu_ctx.set_tile_shape(-1, 0)
        outs.append(dC)
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("m,n,k", [(1, 33, 16), (15, 31, 15), (16, 32, 16), (17, 33, 17), (33, 65, 31), (48, 64, 33),
                                   (160, 320, 1), (1000, 31, 48), (511, 511, 32)])
@pytest.mark.parametrize("ta,tb,lower", [("N", "N", False), ("C", "N", False), ("N", "C", True)])
def test_qgemm_small_tiles(gpu_ctx, m, n, k, ta, tb, lower):
    """Products of fewer than two 32 x 64 tiles per CU (16 x 32 tiles, K in
    stages of 16), at the edges of tiles and stages.  Each real component of
    C sums 4 k products of magnitude <= 1 in FMAs, then C itself: rounding at
    most (4 k + 2) eps (4 k + 1) with inputs in (-1, 1); 4x less is asserted
    (errors of random sign)."""
    import torch
    if lower:
        n = m
    _say(f"case: qgemm small tiles m={m} n={n} k={k} {ta}{tb} lower={lower}")
    rng = np.random.default_rng(m + 31 * n + 7 * k)

    def rand(r, c):
        return tuple(rng.uniform(-1, 1, (r, c)) + 1j * rng.uniform(-1, 1, (r, c)) for _ in range(2))

    A = rand(*((k, m) if ta == "C" else (m, k)))
    B = rand(*((n, k) if tb == "C" else (k, n)))
    C = rand(m, n)
    lda, ldb, ldc = A[0].shape[0] + 1, B[0].shape[0], m + 3
    dA = torch.from_numpy(_pack(*A, lda)).cuda()
    dB = torch.from_numpy(_pack(*B, ldb)).cuda()
    dC = torch.from_numpy(_pack(*C, ldc)).cuda()
    before = dC.clone()
    torch.cuda.synchronize()
    assert gpu_ctx.qgemm_device(ta, tb, m, n, k, -1.0, dA.data_ptr(), lda, dB.data_ptr(), ldb, 1.0, dC.data_ptr(), ldc,
                                lower) == 0
    gpu_ctx.synchronize()
    ref = _unembed(_embed(*C) - _embed(*(_ct(*A) if ta == "C" else A)) @ _embed(*(_ct(*B) if tb == "C" else B)), m, n)
    mask = np.tril(np.ones((m, n), dtype=bool)) if lower else np.ones((m, n), dtype=bool)
    bound = (4 * k + 2) * (4 * k + 1) * np.finfo(float).eps / 4
    for g, r in zip(_unpack(dC.cpu().numpy(), m, n), ref):
        assert np.abs(g - r)[mask].max() <= max(bound, 1e-14)
    for g, o in zip(_unpack(dC.cpu().numpy(), m, n), _unpack(before.cpu().numpy(), m, n)):
        assert np.array_equal(g[~mask], o[~mask])
    assert torch.equal(dC[:, m:, :], before[:, m:, :])


@pytest.mark.parametrize("m", [1504, 1505, 1567])
@pytest.mark.parametrize("k", [1, 8, 33])
def test_qgemm_lower_tiles(gpu_ctx, m, k):
    """Lower-triangle products from two 32 x 64 tiles per CU on (32 x 32 tiles):
    bound as above, every entry against torch's FP64 products, the strict
    upper triangle untouched."""
    import torch
    _say(f"case: qgemm lower tiles m={m} k={k}")
    g = torch.Generator(device="cuda").manual_seed(m + k)

    def rand(r, c):   # [column, row, component]
        return 2.0 * torch.rand(c, r, 4, dtype=torch.float64, device="cuda", generator=g) - 1.0

    A, B, C = rand(m, k), rand(m, k), rand(m, m)
    out = C.clone()
    torch.cuda.synchronize()
    assert gpu_ctx.qgemm_device("N", "C", m, m, k, -1.0, A.data_ptr(), m, B.data_ptr(), m, 1.0, out.data_ptr(), m,
                                True) == 0
    gpu_ctx.synchronize()
    # (a1, b1)(a2, b2)^* with (a, b)^* = (conj a, -b): a1 conj a2 + conj b1 b2, b1 conj a2 - conj a1 b2
    a1, b1 = (torch.complex(A[..., 2 * h], A[..., 2 * h + 1]).T for h in range(2))
    a2, b2 = (torch.complex(B[..., 2 * h], B[..., 2 * h + 1]).T for h in range(2))
    pa = a1 @ a2.mH.contiguous() + b1.conj() @ b2.T.contiguous()
    pb = b1 @ a2.mH.contiguous() - a1.conj() @ b2.T.contiguous()
    ref = C - torch.stack([pa.real.T, pa.imag.T, pb.real.T, pb.imag.T], -1)
    low = torch.ones(m, m, dtype=torch.bool, device="cuda").triu()   # [column, row]: row >= column
    bound = (4 * k + 2) * (4 * k + 1) * np.finfo(float).eps / 4
    assert (out - ref)[low].abs().max().item() <= max(bound, 1e-14)
    assert torch.equal(out[~low], C[~low])


# shape, lower, threshold of 64-row tiles (0: the default): the tiles that 256 CUs take
@pytest.mark.parametrize("m,n,lower,t64", [
    (896, 1024, False, 0),    # 16 x 32: 7 of them per CU
    (897, 1024, False, 0),    # 32 x 64: 16 x 32 would be more than 7 per CU
    (1027, 1031, False, 0),   # 32 x 64: two per CU
    (1027, 1031, False, 1),   # 64 x 64
    (1409, 1409, True, 0),    # 32 x 32
    (1409, 1409, True, 1)])   # 64 x 64
@pytest.mark.parametrize("ta,tb", [("N", "N"), ("C", "N"), ("N", "C"), ("C", "C")])
def test_qgemm_tile_shapes(gpu_ctx, m, n, lower, t64, ta, tb):
    """Every tile shape, all conjugations, K at and off a stage's end (1, 7, 8,
    33), beta = 0 over a C of NaNs (which it must not read) and beta != 0.
    Bound as above (|alpha| < 1, |beta C| <= 1.25), against torch's FP64 products."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(m + n)

    def rand(r, c):   # [column, row, component]
        return 2.0 * torch.rand(c, r, 4, dtype=torch.float64, device="cuda", generator=g) - 1.0

    def op(Q, conj):   # complex components (a, b) of op(Q)
        a, b = (torch.complex(Q[..., 2 * h], Q[..., 2 * h + 1]).T.contiguous() for h in range(2))
        return (a.mH.resolve_conj().contiguous(), -b.T.contiguous()) if conj else (a, b)

    low = torch.ones(n, m, dtype=torch.bool, device="cuda")   # [column, row]: the entries written
    if lower:
        low = low.triu()
    gpu_ctx.set_tile_shape(-1, t64)
    try:
        for k, alpha, beta in ((1, -1.0, 0.0), (7, -0.75, 1.25), (8, 1.0, 0.0), (33, 0.5, -1.25)):
            _say(f"case: qgemm tile shapes m={m} n={n} k={k} {ta}{tb} lower={lower} t64={t64} beta={beta}")
            A = rand(k, m) if ta == "C" else rand(m, k)
            B = rand(n, k) if tb == "C" else rand(k, n)
            C = rand(m, n) if beta else torch.full((n, m, 4), float("nan"), dtype=torch.float64, device="cuda")
            out = C.clone()
            torch.cuda.synchronize()
            assert gpu_ctx.qgemm_device(ta, tb, m, n, k, alpha, A.data_ptr(), A.shape[1], B.data_ptr(), B.shape[1],
                                        beta, out.data_ptr(), m, lower) == 0
            gpu_ctx.synchronize()
            (a1, b1), (a2, b2) = op(A, ta == "C"), op(B, tb == "C")
            pa = a1 @ a2 - b1.conj().resolve_conj() @ b2
            pb = b1 @ a2 + a1.conj().resolve_conj() @ b2
            ref = alpha * torch.stack([pa.real.T, pa.imag.T, pb.real.T, pb.imag.T], -1)
            if beta:
                ref = ref + beta * C
            bound = (4 * k + 2) * (4 * k + 2) * np.finfo(float).eps / 4
            assert (out - ref)[low].abs().max().item() <= max(bound, 1e-14)
            assert torch.equal(out[~low].view(torch.int64), C[~low].view(torch.int64))
    finally:
        gpu_ctx.set_tile_shape(-1, 0)


def test_qgemm_argument_errors(gpu_ctx):
    assert gpu_ctx.qgemm_device("X", "N", 2, 2, 2, 1.0, 0, 2, 0, 2, 0.0, 0, 2) == -2
    assert gpu_ctx.qgemm_device("N", "N", -1, 2, 2, 1.0, 0, 2, 0, 2, 0.0, 0, 2) == -4
    assert gpu_ctx.qgemm_device("N", "N", 2, 2, 2, 1.0, 0, 2, 0, 2, 0.0, 0, 2) == -5
