"""GPU parity of GGML_OP_MUL_MAT with F32, F16 and BF16 weights against the
CPU oracle (oracle_mul_mat_dense: compute.rs:1680-1745, vec_dot.rs:1700-1727).

The activations are rounded to the weight type as the reference rounds them
(f16 / bf16 round to nearest even), so every product is the same exact value
on both sides; only the fp32 summation order differs.  Bar: 1e-5 by
rel_err = max |a-b| / max(|b|, 1) (vec_dot.rs:2355).
"""
import numpy as np
import pytest

import oracle_lib as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

TOL = 1e-5


@pytest.fixture(scope="module")
def be():
    import ghip
    b = ghip.Backend(0)
    yield b
    b.close()


def rel_err(a, b):
    return float(np.max(np.abs(a - b) / np.maximum(np.abs(b), 1.0))) if a.size else 0.0


def make(ty, rows, k, seed, scale=0.02):
    rng = np.random.default_rng(seed)
    wf = (rng.standard_normal((rows, k)) * scale).astype(np.float32)
    if ty == O.F32:
        return torch.from_numpy(wf), wf
    if ty == O.F16:
        t = torch.from_numpy(wf).to(torch.float16)
    else:
        t = torch.from_numpy(wf).to(torch.bfloat16)
    return t, t.view(torch.int16).numpy().view(np.uint16)


@pytest.mark.parametrize("ty", [O.F32, O.F16, O.BF16])
@pytest.mark.parametrize("k,rows,cols", [(4096, 64, 1), (4096, 100, 3), (1000, 37, 8), (14336, 48, 2),
                                         (4096, 256, 11), (77, 9, 5), (128, 4096, 4)])
def test_dense_weights(be, ty, k, rows, cols):
    wt, wbits = make(ty, rows, k, k + rows + cols)
    x = np.random.default_rng(cols).standard_normal((cols, k)).astype(np.float32)
    want = O.mul_mat_dense(ty, wbits, k, rows, x, cols)
    print(f"dense type={ty} k={k} rows={rows} cols={cols}", flush=True)
    got = be.mul_mat(wt.cuda(), ty, k, torch.from_numpy(x).cuda()).cpu().numpy()
    assert rel_err(got, want) <= TOL, rel_err(got, want)


@pytest.mark.parametrize("ty", [O.F16, O.BF16])
def test_activation_rounding_is_the_references(be, ty):
    """activations that differ only below the weight type's precision (ties
    included) give the reference's rounding: exact outputs on unit weights"""
    k, rows = 256, 8
    w = np.zeros((rows, k), dtype=np.float32)
    w[np.arange(rows), np.arange(rows)] = 1.0
    wt = torch.from_numpy(w).to(torch.float16 if ty == O.F16 else torch.bfloat16)
    wbits = wt.view(torch.int16).numpy().view(np.uint16)
    base = np.float32(1.0)
    ulp = 2.0 ** -10 if ty == O.F16 else 2.0 ** -7
    x = np.zeros((1, k), dtype=np.float32)
    x[0, :rows] = base + np.array([0.5, 1.5, 0.25, 0.75, 2.5, -0.5, 0.49, 0.51], dtype=np.float32) * np.float32(ulp)
    want = O.mul_mat_dense(ty, wbits, k, rows, x, 1)
    got = be.mul_mat(wt.cuda(), ty, k, torch.from_numpy(x).cuda()).cpu().numpy()
    assert np.array_equal(got, want)


def test_dense_batched_planes(be):
    """F16 weights with broadcast planes (ne12 = 2 * ne02), as an FA-off KQ"""
    import ghip
    k, rows, m = 128, 64, 5
    w = torch.randn(2, rows, k, generator=torch.Generator().manual_seed(1)).to(torch.float16)
    x = torch.randn(4, m, k, generator=torch.Generator().manual_seed(2))
    import ctypes as C
    out = torch.empty(4, m, rows, device="cuda")
    wd, xd = w.cuda(), x.cuda()
    a, b, d = ghip.describe(wd, ghip.F16), ghip.describe(xd, ghip.F32), ghip.describe(out, ghip.F32)
    st = ghip.lib().ghip_mul_mat(be._ctx, C.byref(a), C.byref(b), C.byref(d), None)
    assert st == 0, ghip.lib().ghip_last_error(be._ctx)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    wb = w.view(torch.int16).numpy().view(np.uint16)
    for p in range(4):
        want = O.mul_mat_dense(O.F16, wb[p // 2], k, rows, x[p].numpy(), m)
        assert rel_err(got[p], want) <= TOL


@pytest.mark.parametrize("M,N,K", [
    (9, 33, 8),           # one step's first piece; 32 x 32 tiles, ragged rows
    (32, 32, 64),         # one whole step, one whole tile
    (33, 65, 72),         # a step of one piece
    (65, 127, 584),       # past the first eight steps
    (40, 70, 77),         # K not a multiple of 8: rows that end inside a piece
    (9, 16, 3),
    (200, 3841, 256),     # 64 x 64 tiles
    (520, 6017, 136),     # 128 x 128 tiles
])
@pytest.mark.parametrize("ty", ["f16", "bf16"])
def test_prefill_gemm(be, ty, M, N, K):
    """F16 / BF16 weights from 9 rows (the matrix cores) at the edges of tiles,
    steps and pieces, with strided rows, against 64-bit sums of the exact
    products.  Bound: every partial sum is rounded at most 64 times inside a
    step, 8 times over the steps of a group, K / 512 + 1 times over the groups
    and 3 times over wavefronts, each by 2^-24 of the terms' magnitude."""
    import ghip
    td = torch.float16 if ty == "f16" else torch.bfloat16
    g = torch.Generator().manual_seed(M + N + K)
    w = (torch.randn((N, K + 5), generator=g) * 0.02).to(td)
    w[0, : min(3, K)] = 1e-6  # f16 subnormals
    x = torch.randn((M, K + 3), generator=g)
    xr, wr = x[:, :K].to(td).double(), w[:, :K].double()
    want, mag = xr @ wr.t(), xr.abs() @ wr.abs().t()
    out = torch.full((M + 1, N + 2), 7.0, device="cuda")
    got = be.mul_mat(w.cuda()[:, :K], ghip.F16 if ty == "f16" else ghip.BF16, K, x.cuda()[:, :K], out=out[:M, :N])
    err = (got.cpu().double() - want).abs()
    assert bool((err <= (64 + 8 + K // 512 + 1 + 3) * 2.0 ** -24 * mag).all()), float((err / mag.clamp_min(1e-30)).max())
    assert bool((out[M] == 7.0).all()) and bool((out[:, N:] == 7.0).all())


@pytest.mark.parametrize("ty,M,N,K,decode", [
    ("f16", 9, 512, 14336, True),
    ("f16", 9, 64, 12288, True),
    ("f16", 12, 64, 8192, False),
    ("bf16", 17, 64, 8192, False),
    ("f16", 24, 1000, 4095, True),    # K not a multiple of 8
    ("bf16", 16, 1024, 8192, True),
    ("bf16", 10, 100, 2047, True),
    ("f16", 16, 512, 14336, False),
    ("bf16", 24, 512, 4096, False),
    ("f16", 64, 512, 1001, False),
])
def test_few_rows_long_k(be, ty, M, N, K, decode):
    """9 rows and more of a long K: the faster of the decode kernel (its bits:
    those of its groups of 8 rows) and the GEMM, whose K is one chain."""
    import ghip
    td = torch.float16 if ty == "f16" else torch.bfloat16
    g = torch.Generator().manual_seed(M + N + K)
    w, x = (torch.randn((N, K), generator=g) * 0.02).to(td), torch.randn((M, K), generator=g)
    t = ghip.F16 if ty == "f16" else ghip.BF16
    got = be.mul_mat(w.cuda(), t, K, x.cuda())
    first = be.mul_mat(w.cuda(), t, K, x[:8].cuda())
    assert torch.equal(got[:8], first) == decode
    xr, wr = x.to(td).double(), w.double()
    err = (got.cpu().double() - xr @ wr.t()).abs()
    assert bool((err <= (64 + 8 + K // 512 + 1 + 3) * 2.0 ** -24 * (xr.abs() @ wr.abs().t())).all())


@pytest.mark.parametrize("ty", ["f16", "bf16"])
@pytest.mark.parametrize("M,N,K", [(40, 70, 264), (300, 4000, 256), (12, 33, 77)])
def test_prefill_gemm_specials(be, ty, M, N, K):
    """Infinities and NaN in activations and weights, and activations that round
    to infinity, reach their own rows and columns only, as in 64 bits."""
    import ghip
    td = torch.float16 if ty == "f16" else torch.bfloat16
    g = torch.Generator().manual_seed(K)
    w, x = torch.randn((N, K), generator=g).to(td), torch.randn((M, K), generator=g)
    x[1, 3], x[5, K - 1], x[8, 0] = float("inf"), float("nan"), 3.4e38 if ty == "bf16" else 7e4
    x[9, 5] = 0.0
    w[2, 3], w[7, K - 1], w[11, 5], w[30, 0] = float("-inf"), float("nan"), float("inf"), 0.0
    got = be.mul_mat(w.cuda(), ghip.F16 if ty == "f16" else ghip.BF16, K, x.cuda()).cpu()
    want = x.to(td).double() @ w.double().t()
    assert bool(want.isnan().any()) and bool(want.isinf().any())
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(torch.where(want.isinf(), got, 0.0), torch.where(want.isinf(), want, 0.0).float())
    assert bool(got[want.isfinite()].isfinite().all())


def test_bf16_gemm_carries_its_sum(be):
    """BF16, one 32 x 32 tile, K shared by four wavefronts: the first 64-element group
    of each is 64, every later one 0.85 of half an ulp of that.  Every product and
    group is exact; what is left are half an ulp of the result, the roundings of
    the three additions of the wavefronts' parts and what these drop at the end."""
    import ghip
    M, N, K = 24, 64, 16384
    w = torch.full((N, K), 0.85 * 2.0 ** -24).to(torch.bfloat16)
    w[:, :256] = 1.0
    x = torch.ones((M, K))
    want = float(w[0].double().sum())
    got = be.mul_mat(w.cuda(), ghip.BF16, K, x.cuda()).cpu().double()
    assert float((got - want).abs().max()) <= 2 * 2.0 ** -23 * want, (float(got[0, 0]), want)
