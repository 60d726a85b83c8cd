"""The Q2_K / Q3_K / Q6_K prefill GEMM (ghip_kq.hip) and the Q4_K / Q5_K / Q6_K
short-batch tiles (ghip_moe.hip; Q4_0, Q8_0 and IQ4_XS too): integer super-block sums equal to the
oracle's, f32 results against 64-bit sums of the same terms."""
import numpy as np
import pytest

import oracle_lib as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# bytes of a block, offsets of d and dmin
BLOCK = {O.Q2_K: (84, 80, 82), O.Q3_K: (110, 108, None), O.Q6_K: (210, 208, None), O.Q4_K: (144, 0, 2), O.Q5_K: (176, 0, 2)}


@pytest.fixture(scope="module")
def be():
    import ghip
    b = ghip.Backend(0)
    yield b
    b.close()


def weights(ty, rows, k, seed):
    """random bytes (every scale and code, the extremes among them) with small
    finite d / dmin"""
    rng = np.random.default_rng(seed)
    size, *at = BLOCK[ty]
    w = rng.integers(0, 256, (rows, k // 256, size), dtype=np.uint8)
    for o in at:
        if o is not None:
            w[:, :, o:o + 2] = (rng.random((rows, k // 256)) * 0.01).astype(np.float16).view(np.uint8).reshape(rows, -1, 2)
    return w.reshape(rows, -1)


def exact(ty, w, k, sub, act):
    """float64 results and the summed magnitudes of their terms"""
    size, at_d, at_m = BLOCK[ty]
    blk = w.reshape(w.shape[0], k // 256, size)
    f16 = lambda o: blk[:, :, o:o + 2].copy().view(np.float16)[..., 0].astype(np.float64)
    d8 = act.reshape(act.shape[0], k // 256, 292)[:, :, :4].copy().view(np.float32)[..., 0].astype(np.float64)
    if at_m is not None:
        a, b = f16(at_d) * sub[..., 0], f16(at_m) * sub[..., 1]
    else:
        a, b = f16(at_d) * sub, 0.0
    return ((a - b) * d8[:, None, :]).sum(-1), ((np.abs(a) + np.abs(b)) * np.abs(d8)[:, None, :]).sum(-1)


@pytest.mark.parametrize("ty", [O.Q2_K, O.Q3_K, O.Q6_K])
@pytest.mark.parametrize("M,N,K", [
    (17, 24, 256),     # fewer rows than one 32-row tile, one super-block
    (64, 128, 512),    # one whole workgroup
    (65, 129, 1280),   # one row and one token past it; N % 4: no K split
    (33, 200, 2304),   # K split with a short last slice
    (130, 160, 4096),
])
def test_gemm(be, ty, M, N, K):
    if ty == O.Q6_K:
        M += 64  # its GEMM's range
    w = weights(ty, N, K, M + N)
    x = np.random.default_rng(K).standard_normal((M, K + 4)).astype(np.float32)
    wd, xd = torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda()[:, :K]
    print(f"kq gemm type={ty} M={M} N={N} K={K}", flush=True)
    act = be.mul_mat_act(wd, ty, K, xd).cpu().numpy()
    want_sub = np.asarray(O.mul_mat(ty, w, K, N, np.ascontiguousarray(x[:, :K]), M, want_subsums=True)[2])
    out = torch.full((M + 1, N + 4), 7.0, device="cuda")
    got = be.mul_mat(wd, ty, K, xd, out=out[:M, :N]).cpu().numpy()
    sub = be.mul_mat_subsums(wd, ty, K, xd).cpu().numpy()
    assert np.array_equal(sub, want_sub.reshape(sub.shape))
    want, mag = exact(ty, w, K, sub.astype(np.float64), act)
    # three roundings a term, then at most 4 + nb / 4 + 2 additions (K slices included)
    assert np.all(np.abs(got - want) <= (4 + 4 + K // 1024 + 2) * 2.0 ** -23 * mag)
    assert bool((out[M] == 7.0).all()) and bool((out[:, N:] == 7.0).all())
    # the kept records, and Q8_K rows in src1, give the same bits
    be.register_weight(wd, ty, K)
    again = be.mul_mat(wd, ty, K, xd).cpu().numpy()
    pre = be.mul_mat(wd, ty, K, torch.from_numpy(act).cuda()).cpu().numpy()
    be.unregister_weight(wd, ty, K)
    assert np.array_equal(again, got) and np.array_equal(pre, got)


@pytest.mark.parametrize("ty", [O.Q4_K, O.Q5_K, O.Q6_K])
@pytest.mark.parametrize("M,N,K", [
    (9, 24, 256),     # fewer rows than a block, one super-block: three idle wavefronts
    (32, 64, 1024),   # whole tiles, one super-block per wavefront
    (33, 33, 1280),   # one token and one row past them
    (63, 200, 768),
])
def test_short_batch(be, ty, M, N, K):
    w = weights(ty, N, K, M * N)
    x = np.random.default_rng(M).standard_normal((M, K + 4)).astype(np.float32)
    wd, xd = torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda()[:, :K]
    print(f"kq32 type={ty} M={M} N={N} K={K}", flush=True)
    act = be.mul_mat_act(wd, ty, K, xd).cpu().numpy()
    want_sub = np.asarray(O.mul_mat(ty, w, K, N, np.ascontiguousarray(x[:, :K]), M, want_subsums=True)[2])
    out = torch.full((M + 1, N + 4), 7.0, device="cuda")
    got = be.mul_mat(wd, ty, K, xd, out=out[:M, :N]).cpu().numpy()
    sub = be.mul_mat_subsums(wd, ty, K, xd).cpu().numpy()
    assert np.array_equal(sub, want_sub.reshape(sub.shape))
    want, mag = exact(ty, w, K, sub.astype(np.float64), act)
    # three roundings a term, a wavefront's chain, two additions over the wavefronts
    assert np.all(np.abs(got - want) <= (4 + K // 1024 + 3) * 2.0 ** -23 * mag)
    assert bool((out[M] == 7.0).all()) and bool((out[:, N:] == 7.0).all())
    pre = be.mul_mat(wd, ty, K, torch.from_numpy(act).cuda()).cpu().numpy()
    assert np.array_equal(pre, got)


@pytest.mark.parametrize("ty", [O.Q4_0, O.Q8_0, O.IQ4_XS])
@pytest.mark.parametrize("M,N,K,skew", [
    (9, 24, 256, 0),      # fewer rows than a block, one wavefront with work
    (32, 64, 2048, 0),    # whole tiles, a super-block for each of eight wavefronts
    (33, 33, 1280, 2),    # one token and one row past them; weights 2-byte aligned
    (64, 200, 2304, 0),
    (40, 8224, 256, 0),   # too wide for Q8_0, the 4-bit types unless registered
])
def test_short_batch_q8(be, ty, M, N, K, skew):
    qk, size = O.BLOCK[ty]
    rng = np.random.default_rng(M * N)
    w = rng.integers(0, 256, (N, K // qk, size), dtype=np.uint8)
    w[:, :, :2] = (rng.random((N, K // qk)) * 0.01).astype(np.float16).view(np.uint8).reshape(N, -1, 2)
    w = w.reshape(N, -1)
    x = rng.standard_normal((M, K + 4)).astype(np.float32)
    x[:, 32:64] = 0.0  # a zero block
    wd = torch.empty(w.size + 16, dtype=torch.uint8, device="cuda")[skew:skew + w.size].view(N, -1)
    wd.copy_(torch.from_numpy(w))
    xd = torch.from_numpy(x).cuda()[:, :K]
    print(f"kq32 type={ty} M={M} N={N} K={K}", flush=True)
    act = be.mul_mat_act(wd, ty, K, xd).cpu().numpy()
    w8 = np.concatenate([w, np.zeros((-N % 8, w.shape[1]), np.uint8)])  # (the oracle's Q4_0 rows go by eight)
    want_sub = np.asarray(O.mul_mat(ty, w8, K, len(w8), np.ascontiguousarray(x[:, :K]), M, want_subsums=True)[2])[:, :N]
    out = torch.full((M + 1, N + 4), 7.0, device="cuda")
    got = be.mul_mat(wd, ty, K, xd, out=out[:M, :N]).cpu().numpy()
    sub = be.mul_mat_subsums(wd, ty, K, xd).cpu().numpy()
    assert np.array_equal(sub, want_sub.reshape(sub.shape))
    d = w.reshape(N, -1, size)[:, :, :2].copy().view(np.float16)[..., 0].astype(np.float64)
    if ty == O.IQ4_XS:
        d8 = act.reshape(M, -1, 292)[:, :, :4].copy().view(np.float32)[..., 0].astype(np.float64)
    else:
        d8 = act.reshape(M, -1, 34)[:, :, :2].copy().view(np.float16)[..., 0].astype(np.float64)
    t = d * sub.reshape(M, N, -1) * d8[:, None, :]
    # three roundings a term (Q4_0 / Q8_0: one, in sums of eight), a carried chain,
    # carried additions over the wavefronts; the prefill GEMM: a chain over K / 32
    n = 16 if N <= 8192 else 4 + K // 32
    assert np.all(np.abs(got - t.sum(-1)) <= n * 2.0 ** -24 * np.abs(t).sum(-1))
    assert bool((out[M] == 7.0).all()) and bool((out[:, N:] == 7.0).all())
    if skew == 0:  # registered: this or the prefill GEMM
        be.register_weight(wd, ty, K)
        again = be.mul_mat(wd, ty, K, xd).cpu().numpy()
        be.unregister_weight(wd, ty, K)
        assert np.all(np.abs(again - t.sum(-1)) <= (4 + K // 32) * 2.0 ** -24 * np.abs(t).sum(-1))


@pytest.mark.parametrize("ty,M,N,K", [
    (O.Q4_K, 24, 136, 8448),   # 33 super-blocks: split K, one partial token tile
    (O.Q4_K, 33, 204, 8192),   # N % 8 != 0: row by row activations
    (O.Q4_K, 40, 8224, 256),
    (O.Q5_K, 100, 64, 1024),   # scales and mins 63, codes 31 and 0 (below)
    (O.Q5_K, 70, 136, 2048),
])
def test_q4_q5_gemm(be, ty, M, N, K):
    """The Q4_K GEMM where short batches reach it, and the Q5_K one, whose
    fifth-bit plane 2 * sc * bit the extreme blocks take to its ends."""
    w = weights(ty, N, K, M)
    if ty == O.Q5_K:
        blk = w.reshape(N, K // 256, 176)
        blk[::2, :, 4:16] = 0xFF
        blk[::4, :, 16:176] = 0xFF
        blk[1::4, :, 16:176] = 0
    x = np.random.default_rng(N).standard_normal((M, K)).astype(np.float32)
    wd, xd = torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda()
    print(f"gemm type={ty} M={M} N={N} K={K}", flush=True)
    sub = be.mul_mat_subsums(wd, ty, K, xd).cpu().numpy()
    want_sub = np.asarray(O.mul_mat(ty, w, K, N, x, M, want_subsums=True)[2])
    assert np.array_equal(sub, want_sub.reshape(sub.shape))
    out = torch.full((M + 1, N + 4), 7.0, device="cuda")
    got = be.mul_mat(wd, ty, K, xd, out=out[:M, :N]).cpu().numpy()
    want, mag = exact(ty, w, K, sub.astype(np.float64), be.mul_mat_act(wd, ty, K, xd).cpu().numpy())
    # three roundings a term, a chain over the super-blocks
    assert np.all(np.abs(got - want) <= (4 + K // 256) * 2.0 ** -23 * mag)
    assert bool((out[M] == 7.0).all()) and bool((out[:, N:] == 7.0).all())


@pytest.mark.parametrize("nb", [2, 3, 4, 5, 9, 10])
def test_split_k_slices(be, nb):
    """One super-block a slice: two, a few, and around eight slices after the first."""
    test_q4_q5_gemm(be, O.Q4_K, 70, 136, 256 * nb)


def test_wide_group(be):
    """Gate and up of a 37-row batch, together too wide for the tiles: the GEMM on
    the library's own workspace, against 64-bit sums."""
    import ghip
    M, N, K = 37, 5000, 512
    x = np.random.default_rng(7).standard_normal((M, K)).astype(np.float32)
    xd = torch.from_numpy(x).cuda()
    ws = [weights(O.Q4_K, N, K, 20 + i) for i in range(2)]
    wds = [torch.from_numpy(w).cuda() for w in ws]
    outs = [torch.full((M + 1, N + 4), 7.0, device="cuda") for _ in ws]
    be.graph_compute([ghip.mul_mat_node(wd, O.Q4_K, K, xd, o[:M, :N]) for wd, o in zip(wds, outs)])
    for w, wd, o in zip(ws, wds, outs):
        sub = be.mul_mat_subsums(wd, O.Q4_K, K, xd).cpu().numpy().astype(np.float64)
        want, mag = exact(O.Q4_K, w, K, sub, be.mul_mat_act(wd, O.Q4_K, K, xd).cpu().numpy())
        # three roundings a term, a chain over the super-blocks
        assert np.all(np.abs(o[:M, :N].cpu().numpy() - want) <= (4 + K // 256) * 2.0 ** -23 * mag)
        assert bool((o[M] == 7.0).all()) and bool((o[:, N:] == 7.0).all())


@pytest.mark.parametrize("ty,N", [(O.Q4_0, 8224), (O.IQ4_XS, 8224), (O.Q8_0, 6144)])
def test_registering_keeps_a_call_served(ty, N):
    """A wide weight that is registered after the call's first run: its capture
    may not grow the workspace, and a caller's need not hold the GEMM's layout."""
    import ghip
    M, K = 40, 256
    be = ghip.Backend(0)
    qk, size = O.BLOCK[ty]
    rng = np.random.default_rng(1)
    w = rng.integers(0, 256, (N, K // qk, size), dtype=np.uint8)
    w[:, :, :2] = (rng.random((N, K // qk)) * 0.01).astype(np.float16).view(np.uint8).reshape(N, -1, 2)
    wd = torch.from_numpy(w.reshape(N, -1)).cuda()
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).cuda()
    out = torch.empty((M, N), device="cuda")
    want = be.mul_mat(wd, ty, K, x, out=out).clone()
    be.register_weight(wd, ty, K)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        be.mul_mat(wd, ty, K, x, out=out)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
    del g
    be.set_workspace(torch.empty(16384, dtype=torch.uint8, device="cuda"))
    assert torch.equal(be.mul_mat(wd, ty, K, x), want)
    be.set_workspace(None)
    tol = 40 * 2.0 ** -24 * float(want.abs().max())
    assert float((be.mul_mat(wd, ty, K, x) - want).abs().max()) <= tol  # the GEMM over the copy
    be.unregister_weight(wd, ty, K)
    be.close()


def test_row_switch_holds_for_a_registered_weight(be, monkeypatch):
    """Q6_K with GHIP_GEMM_Q6K_MIN_ROWS raised: registered or not, the decode
    kernels in the workspace that ghip_workspace_size names."""
    import ghip
    M, N, K = 64, 128, 1024
    wd = torch.from_numpy(weights(O.Q6_K, N, K, 2)).cuda()
    x = torch.from_numpy(np.random.default_rng(3).standard_normal((M, K)).astype(np.float32)).cuda()
    monkeypatch.setenv("GHIP_GEMM_Q6K_MIN_ROWS", "1000")
    out = torch.empty((M, N), device="cuda")
    want = be.mul_mat(wd, O.Q6_K, K, x)
    be.register_weight(wd, O.Q6_K, K)
    be.set_workspace(torch.empty(be.workspace_size(ghip.mul_mat_node(wd, O.Q6_K, K, x, out)), dtype=torch.uint8, device="cuda"))
    got = be.mul_mat(wd, O.Q6_K, K, x, out=out)
    be.set_workspace(None)
    be.unregister_weight(wd, O.Q6_K, K)
    assert torch.equal(got, want)


def test_short_batch_carries_its_sum(be):
    """Q6_K, four wavefronts a tile, long K: the first super-block of every
    wavefront's share is large, each of the others 0.9 * 2^-25 of it, below half
    an ulp of the sum, so that a plain chain loses them all (5.8 * 2^-24 of the
    result).  Every term is exact; what is left are the result's own rounding
    and those of three additions, carried."""
    M, N, K = 40, 4128, 14336
    blk = np.zeros((K // 256, 210), np.uint8)
    blk[:, :128], blk[:, 128:192], blk[:, 192:208] = 0x11, 0xAA, 1  # every code 33 (value 1), scales 1
    d = np.full(K // 256, 0.9 * 2.0 ** -15, np.float16)
    d[:4] = 1024.0
    blk[:, 208:210] = d.view(np.uint8).reshape(-1, 2)
    wd = torch.from_numpy(blk.reshape(1, -1)).cuda().expand(N, -1).contiguous()
    x = torch.full((M, K), 127.0, device="cuda")
    got = be.mul_mat(wd, O.Q6_K, K, x).cpu().numpy().astype(np.float64)
    want = float(d.astype(np.float64).sum()) * 256 * 127
    assert np.all(np.abs(np.abs(got) - want) <= 2 * 2.0 ** -24 * want), (got[0, 0], want)


def test_q3_gemm_sums_in_fours(be):
    """Q3_K, whole K in one workgroup: a large super-block and seven of 0.9 * 2^-25 of
    it, below half an ulp.  Three of them meet it in its four and are lost (1.35 *
    2^-24 of the result), the other four reach the total; all seven are 3.15."""
    M, N, K = 300, 14336, 2048
    w = np.zeros((K // 256, 110), np.uint8)
    w[:, :32], w[:, 32:96], w[:, 96:104], w[:, 104:108] = 0xFF, 0x55, 0x11, 0xAA  # every code and scale 1
    d = np.full(K // 256, 0.9 * 2.0 ** -15, np.float16)
    d[0] = 1024.0
    w[:, 108:110] = d.view(np.uint8).reshape(-1, 2)
    wd = torch.from_numpy(w.reshape(1, -1)).cuda().expand(N, -1).contiguous()
    got = be.mul_mat(wd, O.Q3_K, K, torch.full((M, K), 127.0, device="cuda")).double().abs()
    want = float(d.astype(np.float64).sum()) * 256 * 127
    err = float((got - want).abs().max())
    assert err <= 2.4 * 2.0 ** -24 * want, (float(got[0, 0]), want)  # (and the result's own rounding, 1)


def test_short_batch_group(be):
    """Siblings too wide together for these tiles, in a workspace sized for each
    alone: the bits of the single calls."""
    import ghip
    M, N, K = 40, 4096, 256
    xd = torch.randn(M, K, device="cuda")
    ws = [torch.from_numpy(weights(O.Q4_K, N, K, i)).cuda() for i in range(3)]
    want = [be.mul_mat(w, O.Q4_K, K, xd) for w in ws]
    outs = [torch.empty_like(o) for o in want]
    nodes = [ghip.mul_mat_node(w, O.Q4_K, K, xd, o) for w, o in zip(ws, outs)]
    be.set_workspace(torch.empty(max(be.workspace_size(nd) for nd in nodes), dtype=torch.uint8, device="cuda"))
    be.graph_compute(nodes)
    torch.cuda.synchronize()
    be.set_workspace(None)
    assert all(torch.equal(a, b) for a, b in zip(outs, want))


@pytest.mark.parametrize("ty,M", [(O.Q2_K, 20), (O.Q3_K, 20), (O.Q6_K, 70), (O.Q4_K, 150), (O.Q4_K, 24), (O.Q5_K, 24), (O.Q6_K, 24)])
def test_infinite_scale(be, ty, M):
    """A block scale of infinity gives infinities (NaN where its sum is 0 or two
    of them cancel), K split and not, and leaves the other rows alone."""
    K, N = 4096, 136
    w = weights(ty, N, K, 9)
    size, at_d, _ = BLOCK[ty]
    blk = w.reshape(N, K // 256, size)
    for row, bs in ((3, (0,)), (40, (5,)), (100, (15,)), (135, (2, 9))):
        for b in bs:
            blk[row, b, at_d:at_d + 2] = np.array([np.inf], np.float16).view(np.uint8)
    x = np.random.default_rng(8).standard_normal((M, K)).astype(np.float32)
    wd, xd = torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda()
    got = be.mul_mat(wd, ty, K, xd).cpu().numpy()
    sub = be.mul_mat_subsums(wd, ty, K, xd).cpu().numpy().astype(np.float64)
    with np.errstate(invalid="ignore"):
        want, _ = exact(ty, w, K, sub, be.mul_mat_act(wd, ty, K, xd).cpu().numpy())
    assert np.isinf(want).any() and np.isfinite(want).any()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.where(np.isinf(want), got, 0), np.where(np.isinf(want), want, 0))
    assert np.isfinite(got[np.isfinite(want)]).all()


def same_specials(got, want):
    """NaN and infinities where the 64-bit value has them, finite elsewhere"""
    assert np.isinf(want).any() and np.isnan(want).any() and np.isfinite(want).any()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.where(np.isinf(want), got, 0), np.where(np.isinf(want), want, 0))
    assert np.isfinite(got[np.isfinite(want)]).all()


@pytest.mark.parametrize("ty,M", [(O.Q4_0, 24), (O.Q8_0, 24), (O.IQ4_XS, 24), (O.Q2_K, 20), (O.Q4_K, 24), (O.Q5_K, 24),
                                  (O.Q4_K, 150)])
def test_infinite_scale_or_min(be, ty, M):
    """The short-batch tiles' Q8_0-row types with an infinite block scale, the
    types with mins with an infinite dmin: infinities and NaN (zero sums, two
    infinities that cancel) as in 64 bits."""
    K, N = 2048, 136
    qk, size = O.BLOCK[ty]
    rng = np.random.default_rng(4)
    at = BLOCK[ty][2] if ty in BLOCK else 0
    if ty in BLOCK:
        w = weights(ty, N, K, 3).reshape(N, -1, size)
    else:
        w = rng.integers(0, 256, (N, K // qk, size), dtype=np.uint8)
        w[:, :, :2] = (rng.random((N, K // qk)) * 0.01).astype(np.float16).view(np.uint8).reshape(N, -1, 2)
    for row, bs in ((3, (0,)), (40, (5,)), (135, (1, 3, 6))):
        for i, b in enumerate(bs):
            w[row, b, at:at + 2] = np.array([-np.inf if i == 1 else np.inf], np.float16).view(np.uint8)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[::3, :1024] = 0.0  # zero blocks: infinity times zero
    wd, xd = torch.from_numpy(w.reshape(N, -1)).cuda(), torch.from_numpy(x).cuda()
    got = be.mul_mat(wd, ty, K, xd).cpu().numpy()
    sub = be.mul_mat_subsums(wd, ty, K, xd).cpu().numpy().astype(np.float64)
    act = be.mul_mat_act(wd, ty, K, xd).cpu().numpy()
    with np.errstate(invalid="ignore"):
        if ty in BLOCK:
            want, _ = exact(ty, w.reshape(N, -1), K, sub, act)
        else:
            d = w[:, :, :2].copy().view(np.float16)[..., 0].astype(np.float64)
            d8 = (act.reshape(M, -1, 292)[:, :, :4].copy().view(np.float32) if ty == O.IQ4_XS
                  else act.reshape(M, -1, 34)[:, :, :2].copy().view(np.float16))[..., 0].astype(np.float64)
            want = (d * sub.reshape(M, N, -1) * d8[:, None, :]).sum(-1)
    same_specials(got, want)


@pytest.mark.parametrize("ty", [O.Q2_K, O.Q3_K])
def test_small_workspace(be, ty):
    """A caller's workspace too small for the GEMM's layout still serves the
    call: without the K split, then on the decode kernels."""
    import ghip
    M, N, K = 20, 128, 4096
    w = weights(ty, N, K, 5)
    x = np.random.default_rng(6).standard_normal((M, K)).astype(np.float32)
    wd, xd = torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda()
    out = torch.empty((M, N), device="cuda")
    full = be.workspace_size(ghip.mul_mat_node(wd, ty, K, xd, out))
    ref = be.mul_mat(wd, ty, K, xd).cpu().numpy()
    sub = be.mul_mat_subsums(wd, ty, K, xd).cpu().numpy().astype(np.float64)
    want, mag = exact(ty, w, K, sub, be.mul_mat_act(wd, ty, K, xd).cpu().numpy())
    for n in (full, full - 1, M * K // 256 * 292):
        be.set_workspace(torch.empty(n, dtype=torch.uint8, device="cuda"))
        got = be.mul_mat(wd, ty, K, xd).cpu().numpy()
        be.set_workspace(None)
        assert n != full or np.array_equal(got, ref)
        # (the decode kernels: three roundings a term, 8 additions)
        assert np.all(np.abs(got - want) <= 16 * 2.0 ** -23 * mag)
    # capture may not grow the workspace: a fresh context's small one serves
    be2 = ghip.Backend(0)
    be2.mul_mat(wd, ty, K, xd[:8], out=out[:8])
    g = torch.cuda.CUDAGraph()
    be2.mul_mat_act(wd, ty, K, xd)
    with torch.cuda.graph(g):
        be2.mul_mat(wd, ty, K, xd[:17], out=out[:17])
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert np.all(np.abs(out[:17].cpu().numpy() - want[:17]) <= 16 * 2.0 ** -23 * mag[:17])
    del g
    be2.close()
