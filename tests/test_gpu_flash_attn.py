"""GPU parity of GGML_OP_FLASH_ATTN_EXT (f16 K/V) against the CPU oracle.

Bar: within 2e-3 max-abs of the reference path.  The
oracle follows the reference's dispatch (split-KV for single-row decode with
S >= 512, tiled for >= 64 query rows, one_chunk otherwise), pinned bit-exact
on parity/fa_ref.bin and fa_probe.bin (test_oracle_golden.py).
"""
import numpy as np
import pytest

import oracle_lib as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

TOL = 2e-3


@pytest.fixture(scope="module")
def be():
    import ghip
    b = ghip.Backend(0)
    yield b
    b.close()


def causal_mask(T, S):
    m = np.zeros((T, S), dtype=np.float16)
    for t in range(T):
        m[t, S - T + t + 1:] = -np.inf
    return m


def run(be, H, Hkv, D, T, S, mask="causal", sinks=False, softcap=0.0, max_bias=0.0, seed=0, n_chunks=8):
    rng = np.random.default_rng(seed)
    q = rng.standard_normal((H, T, D)).astype(np.float32)
    k = rng.standard_normal((Hkv, S, D)).astype(np.float16)
    v = rng.standard_normal((Hkv, S, D)).astype(np.float16)
    m = causal_mask(T, S) if mask == "causal" else (np.zeros((T, S), np.float16) if mask == "zero" else None)
    sk = rng.standard_normal(H).astype(np.float32) if sinks else None
    scale = 1.0 / np.sqrt(D)
    want, path = O.flash_attn_ext(q, k, v, m, sk, scale, max_bias, softcap, n_chunks=n_chunks)
    print(f"fa H={H} Hkv={Hkv} D={D} T={T} S={S} mask={mask} path={path}", flush=True)
    t = lambda a: torch.from_numpy(a).cuda() if a is not None else None
    got = be.flash_attn_ext(t(q), t(k), t(v), t(m), t(sk), scale, max_bias, softcap).cpu().numpy()
    err = float(np.max(np.abs(got - want)))
    assert err <= TOL, f"max-abs {err:.3e}"
    return err


@pytest.mark.parametrize("T,S", [(1, 64), (1, 100), (1, 600), (3, 40), (5, 700), (32, 96), (64, 64), (70, 130)])
def test_small(be, T, S):
    run(be, 4, 2, 64, T, S)
    run(be, 8, 2, 128, T, S, seed=1)


def test_variants(be):
    run(be, 4, 4, 128, 2, 300, mask=None)
    run(be, 4, 1, 64, 65, 200, sinks=True)
    run(be, 4, 2, 64, 70, 200, softcap=15.0)
    run(be, 8, 2, 64, 64, 128, max_bias=8.0, mask="zero")
    run(be, 4, 2, 128, 1, 513, sinks=True)


@pytest.mark.parametrize("H,Hkv,D,T,S", [(4, 4, 128, 100, 301), (6, 2, 128, 100, 258), (6, 2, 64, 130, 67),
                                         (8, 1, 128, 64, 150), (7, 1, 64, 96, 333), (16, 2, 128, 200, 1031)])
def test_head_groups(be, H, Hkv, D, T, S):
    """Tiled route for every head-group size: workgroups of G heads times
    ceil(4 / G) query tiles, ragged key counts and ragged query tiles."""
    run(be, H, Hkv, D, T, S, seed=H + T)


def test_fully_masked_rows(be):
    """Rows whose keys are all masked produce zeros (S == 0 -> S_inv = 0)."""
    H, Hkv, D, T, S = 4, 2, 64, 4, 80
    rng = np.random.default_rng(9)
    q = rng.standard_normal((H, T, D)).astype(np.float32)
    k = rng.standard_normal((Hkv, S, D)).astype(np.float16)
    v = rng.standard_normal((Hkv, S, D)).astype(np.float16)
    m = np.zeros((T, S), dtype=np.float16)
    m[1, :] = -np.inf
    want, _ = O.flash_attn_ext(q, k, v, m, None, 0.125)
    got = be.flash_attn_ext(*(torch.from_numpy(a).cuda() for a in (q, k, v, m)), None, 0.125).cpu().numpy()
    assert np.all(got[1] == 0.0)
    assert np.max(np.abs(got - want)) <= TOL


@pytest.mark.parametrize("T", [1, 512])
def test_config5(be, T):
    """Config 5: 32 query / 8 KV heads, D = 128, KV 8192, causal chunk at the
    end of the cache (decode T = 1, prefill T = 512)."""
    run(be, 32, 8, 128, T, 8192, seed=5, n_chunks=16)


def run_general(be, H, Hkv, DK, DV, T, S, kv=np.float16, sinks=False, seed=0, n_chunks=8):
    rng = np.random.default_rng(seed)
    q = rng.standard_normal((H, T, DK)).astype(np.float32)
    k = rng.standard_normal((Hkv, S, DK)).astype(kv)
    v = rng.standard_normal((Hkv, S, DV)).astype(kv)
    m = causal_mask(T, S)
    sk = rng.standard_normal(H).astype(np.float32) if sinks else None
    scale = 1.0 / np.sqrt(DK)
    want, path = O.flash_attn_ext(q, k, v, m, sk, scale, 0.0, 0.0, n_chunks=n_chunks)
    print(f"fa general H={H} Hkv={Hkv} DK={DK} DV={DV} T={T} S={S} kv={np.dtype(kv).name} path={path}", flush=True)
    t = lambda a: torch.from_numpy(a).cuda() if a is not None else None
    got = be.flash_attn_ext(t(q), t(k), t(v), t(m), t(sk), scale).cpu().numpy()
    err = float(np.max(np.abs(got - want)))
    assert err <= TOL, f"max-abs {err:.3e}"


@pytest.mark.parametrize("H,Hkv,DK,DV,T,S,kv", [
    (8, 2, 256, 256, 5, 300, np.float16),    # D = 256, row walk (f16 accumulator)
    (8, 2, 256, 256, 70, 200, np.float16),   # D = 256, tiled route
    (4, 2, 64, 128, 3, 90, np.float16),      # DK != DV
    (4, 2, 192, 128, 66, 130, np.float16),   # DK != DV, tiled route
    (4, 2, 32, 32, 40, 100, np.float16),
    (4, 2, 64, 64, 10, 80, np.float32),      # F32 K/V, row walk
    (4, 1, 128, 128, 64, 128, np.float32),   # F32 K/V, tiled route
    (32, 2, 64, 64, 4, 120, np.float16),     # H / H_kv = 16
    (16, 1, 80, 80, 1, 700, np.float16),     # split-KV route shape, head size 80
])
def test_general_shapes(be, H, Hkv, DK, DV, T, S, kv):
    """Shapes outside the tuned kernels (F32 K/V, DK != DV, head sizes other
    than 64 / 128, H / H_kv > 8) take the general row walk, still within 2e-3
    of the oracle's route for the shape."""
    run_general(be, H, Hkv, DK, DV, T, S, kv, sinks=(T % 2 == 1))


@pytest.mark.parametrize("T,S,m2,m3", [
    (1, 600, 2, 1),    # split-KV shape, per-head mask planes (row walk, fp32)
    (1, 600, 1, 2),    # split-KV decode kernel, per-sequence planes
    (5, 300, 8, 2),    # one-chunk walk (f16 accumulator)
    (70, 200, 4, 1),   # tiled route on the matrix cores, per-head planes
    (70, 200, 1, 1),
])
def test_mask_planes_and_sequences(be, T, S, m2, m3):
    """The rest of the operand contract (flash_attn.rs:30-37, :298): two
    sequences (ne3 = 2) with their own q, k and v planes, and mask planes
    broadcast to heads by h % ne2 and to sequences by i3 % ne3.  Each
    (sequence, head) is checked against the oracle's route for its shape on
    exactly the mask plane it must read."""
    H, Hkv, D, n_seq = 8, 2, 128, 2
    G = H // Hkv
    rng = np.random.default_rng(T * 1000 + m2 * 10 + m3)
    q = rng.standard_normal((n_seq, H, T, D)).astype(np.float32)
    k = rng.standard_normal((n_seq, Hkv, S, D)).astype(np.float16)
    v = rng.standard_normal((n_seq, Hkv, S, D)).astype(np.float16)
    m = np.zeros((m3, m2, T, S), dtype=np.float16)
    for i3 in range(m3):
        for i2 in range(m2):  # a different causal window per plane
            off = int(rng.integers(0, S // 3))
            for t in range(T):
                m[i3, i2, t, S - T + t + 1 - off:] = -np.inf
            m[i3, i2] += (rng.standard_normal((T, S)) * 0.5).astype(np.float16)
    sk = rng.standard_normal(H).astype(np.float32)
    scale = 1.0 / np.sqrt(D)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    got = be.flash_attn_ext(t(q), t(k), t(v), t(m), t(sk), scale).cpu().numpy()
    assert got.shape == (n_seq, T, H, D)
    worst = 0.0
    for i3 in range(n_seq):
        for h in range(H):
            want, path = O.flash_attn_ext(q[i3, h:h + 1], k[i3, h // G:h // G + 1], v[i3, h // G:h // G + 1],
                                          m[i3 % m3, h % m2], sk[h:h + 1], scale, 0.0, 0.0, n_chunks=8)
            worst = max(worst, float(np.max(np.abs(got[i3, :, h:h + 1] - want))))
    print(f"fa planes T={T} S={S} m2={m2} m3={m3} path={path} max-abs {worst:.2e}", flush=True)
    assert worst <= TOL


@pytest.mark.parametrize("T,S,m2", [(96, 640, 1), (70, 333, 2), (512, 2048, 1)])
def test_mask_tile_classes(be, T, S, m2):
    """The tiled route classifies each (32-query, 64-key) mask tile: all +-0
    (no mask loads), all -inf (no work), or mixed.  A mask made of such tiles
    (whole query blocks masked to -inf, -0.0 tiles, ragged T and S) gives the
    oracle's result, and the same bits as with the classes switched off
    (GHIP_FA_MASK_SCAN=0)."""
    import os
    H, Hkv, D = 8, 2, 128
    rng = np.random.default_rng(T + S + m2)
    q = rng.standard_normal((H, T, D)).astype(np.float32)
    k = rng.standard_normal((Hkv, S, D)).astype(np.float16)
    v = rng.standard_normal((Hkv, S, D)).astype(np.float16)
    m = np.zeros((m2, T, S), dtype=np.float16)
    for p2 in range(m2):
        for qb in range((T + 31) // 32):
            for tl in range((S + 63) // 64):
                c = int(rng.integers(0, 4))
                blk = m[p2, 32 * qb:32 * qb + 32, 64 * tl:64 * tl + 64]
                if c == 1:
                    blk[:] = -np.inf
                elif c == 2:
                    blk[:] = np.float16(-0.0)
                elif c == 3:
                    blk[:] = (rng.standard_normal(blk.shape) * 0.5).astype(np.float16)
        m[p2, 32:64, :] = -np.inf  # a whole query block with no visible key
    mm = m if m2 > 1 else m[0]
    scale = 1.0 / np.sqrt(D)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    outs = []
    for flag in ("0", "1"):
        os.environ["GHIP_FA_MASK_SCAN"] = flag
        try:
            outs.append(be.flash_attn_ext(t(q), t(k), t(v), t(mm), None, scale).cpu().numpy())
        finally:
            del os.environ["GHIP_FA_MASK_SCAN"]
    assert np.array_equal(outs[0], outs[1])
    assert np.all(outs[1][32:64] == 0.0)
    for h in range(H):
        want, _ = O.flash_attn_ext(q[h:h + 1], k[h // (H // Hkv):h // (H // Hkv) + 1],
                                   v[h // (H // Hkv):h // (H // Hkv) + 1], m[h % m2], None, scale, n_chunks=8)
        err = float(np.max(np.abs(outs[1][:, h:h + 1] - want)))
        assert err <= TOL, f"head {h}: max-abs {err:.3e}"


@pytest.mark.parametrize("sinks", [False, True])
def test_merge_preload_four(be, sinks):
    """At most 4 KV slices (T = 512, 32 / 8 heads: 4 slices) the merge loads
    exactly the slices it sums (ghip_fa_merge_rows_p4): the same bits as the
    16-slice preload (GHIP_FA_MERGE_P4=0), and the oracle's result."""
    import os
    H, Hkv, D, T, S = 32, 8, 128, 512, 2048
    rng = np.random.default_rng(5 + sinks)
    q = rng.standard_normal((H, T, D)).astype(np.float32)
    k = rng.standard_normal((Hkv, S, D)).astype(np.float16)
    v = rng.standard_normal((Hkv, S, D)).astype(np.float16)
    m = np.zeros((T, S), dtype=np.float16)
    for i in range(T):
        m[i, S - T + i + 1:] = -np.inf
    sk = (rng.standard_normal(H) * 2.0).astype(np.float32) if sinks else None
    scale = 1.0 / np.sqrt(D)
    t = lambda a: None if a is None else torch.from_numpy(np.ascontiguousarray(a)).cuda()
    print(f"fa merge preload 4 sinks={sinks}", flush=True)
    outs = []
    for flag in ("0", "1"):
        os.environ["GHIP_FA_MERGE_P4"] = flag
        try:
            outs.append(be.flash_attn_ext(t(q), t(k), t(v), t(m), t(sk), scale).cpu().numpy())
        finally:
            del os.environ["GHIP_FA_MERGE_P4"]
    assert np.array_equal(outs[0], outs[1])
    for h in (0, 13, 31):
        g = h // (H // Hkv)
        want, _ = O.flash_attn_ext(q[h:h + 1], k[g:g + 1], v[g:g + 1], m, None if sk is None else sk[h:h + 1], scale,
                                   n_chunks=8)
        err = float(np.max(np.abs(outs[1][:, h:h + 1] - want)))
        assert err <= TOL, f"head {h}: max-abs {err:.3e}"


@pytest.mark.parametrize("T,S,D,masked,sinks", [(96, 640, 128, True, True), (130, 1000, 64, False, False),
                                                (64, 300, 128, True, False), (200, 2048, 64, True, True)])
def test_single_slice_direct(be, monkeypatch, T, S, D, masked, sinks):
    """One KV slice (GHIP_FA_WGS=1 forces it at these sizes; long prefills
    get it by themselves): the forward kernel writes the normalized rows,
    no partials and no merge launch.  Same bits as the partial-and-merge
    route (GHIP_FA_DIRECT=0), and the oracle's result."""
    H, Hkv = 8, 2
    rng = np.random.default_rng(T + S + D + 1)
    q = rng.standard_normal((H, T, D)).astype(np.float32)
    k = rng.standard_normal((Hkv, S, D)).astype(np.float16)
    v = rng.standard_normal((Hkv, S, D)).astype(np.float16)
    m = None
    if masked:
        m = np.zeros((T, S), dtype=np.float16)
        for i in range(T):
            m[i, S - T + i + 1:] = -np.inf
        m[:32, :] = -np.inf  # a query block with no visible key
    sk = (rng.standard_normal(H) * 2.0).astype(np.float32) if sinks else None
    scale = 1.0 / np.sqrt(D)
    t = lambda a: None if a is None else torch.from_numpy(np.ascontiguousarray(a)).cuda()
    print(f"fa single slice T={T} S={S} D={D} masked={masked} sinks={sinks}", flush=True)
    monkeypatch.setenv("GHIP_FA_WGS", "1")
    outs = []
    for flag in ("0", "1"):
        monkeypatch.setenv("GHIP_FA_DIRECT", flag)
        outs.append(be.flash_attn_ext(t(q), t(k), t(v), t(m), t(sk), scale).cpu().numpy())
    assert np.array_equal(outs[0], outs[1])
    for h in (0, 5):
        g = h // (H // Hkv)
        want, _ = O.flash_attn_ext(q[h:h + 1], k[g:g + 1], v[g:g + 1], m, None if sk is None else sk[h:h + 1], scale,
                                   n_chunks=8)
        err = float(np.max(np.abs(outs[1][:, h:h + 1] - want)))
        assert err <= TOL, f"head {h}: max-abs {err:.3e}"


@pytest.mark.parametrize("H,Hkv,D,T,S,holes,sinks,softcap", [
    (8, 2, 128, 1, 1, False, True, 0.0),       # one key
    (8, 2, 64, 2, 63, True, False, 0.0),       # below one 64-key tile
    (6, 2, 128, 3, 64, False, True, 0.0),      # one whole tile; rows past the end of a workgroup
    (4, 4, 64, 7, 129, True, True, 0.0),       # one key in the last tile, one head per KV head
    (8, 1, 128, 5, 320, True, False, 20.0),    # softcap
    (64, 8, 64, 56, 200, True, True, 0.0),     # 448 workgroups: 8 rows each
    (64, 8, 128, 63, 70, False, False, 0.0),
])
def test_few_rows(be, H, Hkv, D, T, S, holes, sinks, softcap):
    """The few-row walk at its tile and row-group edges: masked keys scattered
    over the tiles (whole tiles among them) with infinities in their V rows,
    K and V with keys outside heads (strided rows), against the oracle."""
    rng = np.random.default_rng(H + T + S)
    q = rng.standard_normal((H, T, D)).astype(np.float32)
    k, v = (rng.standard_normal((S, Hkv, D)).astype(np.float16) for _ in range(2))
    m = causal_mask(T, S)
    if holes:
        m[:, rng.random(S) < 0.3] = -np.inf
        m[:, :S // 3] = -np.inf
        m[:, S - T:] = causal_mask(T, T)
        m += (rng.integers(-2, 3, (T, S)) * 0.5).astype(np.float16)
        dead = np.isinf(m).all(axis=0)
        v[dead] = np.inf
    sk = rng.standard_normal(H).astype(np.float32) if sinks else None
    kt, vt = (np.ascontiguousarray(a.transpose(1, 0, 2)) for a in (k, v))
    want, _ = O.flash_attn_ext(q, kt, vt, m, sk, 1.0 / np.sqrt(D), 0.0, softcap)
    t = lambda a: torch.from_numpy(a).cuda() if a is not None else None
    got = be.flash_attn_ext(t(q), t(k).permute(1, 0, 2), t(v).permute(1, 0, 2), t(m), t(sk), 1.0 / np.sqrt(D), 0.0,
                            softcap).cpu().numpy()
    assert np.max(np.abs(got - want)) <= TOL


def walk(q, k, v, m, sk, scale):
    """The few-row route key by key in torch: f32 fma chains (taken in float64,
    where a product of a half and a float is exact, and rounded), f16 accumulator."""
    H, T, D = q.shape
    S, G = k.shape[1], H // k.shape[0]
    kr, vr = k.repeat_interleave(G, 0), v.repeat_interleave(G, 0)
    q16, k64 = q.half().double(), kr.double()
    dot = torch.zeros(H, T, S, device=q.device)
    for d in range(D):
        dot = (q16[:, :, d, None] * k64[:, None, :, d] + dot.double()).float()
    s = dot * scale + m.float()
    acc = torch.zeros(H, T, D, device=q.device, dtype=torch.float16)
    M = torch.full((H, T), -np.inf, device=q.device)
    tot = torch.zeros(H, T, device=q.device)
    one = torch.ones_like(M)
    for j in range(S):
        sj, live = s[:, :, j], m[None, :, j].float() > -np.inf
        up = sj > M
        e = torch.exp(torch.where(up, M - sj, sj - M))
        ms, vs = torch.where(up, e, one), torch.where(up, one, e)
        a = torch.where(up[..., None], (acc.float() * ms[..., None]).half(), acc)
        a = (vr[:, j].double()[:, None, :] * vs.double()[..., None] + a.double()).float().half()
        acc = torch.where(live[..., None], a, acc)
        tot = torch.where(live, (tot.double() * ms.double() + vs.double()).float(), tot)
        M = torch.where(live & up, sj, M)
    a, h = acc.float(), torch.arange(H, device=q.device)[:, None]
    if sk is not None:
        b = sk[:, None].expand(H, T)
        up = b > M
        e = torch.exp(torch.where(up, M - b, b - M))
        a = torch.where(up[..., None], a * e[..., None], a)
        tot = torch.where(up, tot * e + 1.0, tot + e)
    return (a * (1.0 / tot)[..., None]).permute(1, 0, 2)


@pytest.mark.parametrize("H,Hkv,D,T,S,holes,sinks", [
    (8, 2, 64, 5, 300, False, True),
    (8, 2, 128, 3, 257, True, False),
    (64, 8, 64, 56, 200, False, False),   # 8 rows a workgroup
    (64, 8, 128, 56, 130, True, True),
])
def test_few_rows_rounding(be, H, Hkv, D, T, S, holes, sinks):
    """Every rounding of the walk, the scores', the row sum's and both of the
    accumulator's (f32, then f16): the outputs have its bits.  (A tie that
    float64 rounds twice moves an output one f16 step: 1 in 2^29 operations,
    S D of them behind an output.)"""
    g = torch.Generator(device="cuda").manual_seed(H + D + T + S)
    q = torch.randn(H, T, D, generator=g, device="cuda")
    k, v = (torch.randn(Hkv, S, D, generator=g, device="cuda").half() for _ in range(2))
    m = torch.from_numpy(causal_mask(T, S)).cuda()
    if holes:
        m[:, :S - T][:, torch.rand(S - T, generator=g, device="cuda") < 0.3] = -np.inf
    sk = torch.randn(H, generator=g, device="cuda") if sinks else None
    scale = float(np.float32(1.0 / np.sqrt(D)))
    print(f"fa walk H={H} Hkv={Hkv} D={D} T={T} S={S}", flush=True)
    got = be.flash_attn_ext(q, k, v, m, sk, scale)
    differ = float((got != walk(q, k, v, m, sk, scale)).float().mean())
    assert differ <= 1e-3, differ


@pytest.mark.parametrize("D", [64, 128])
def test_few_rows_specials(be, D):
    """Infinities and NaN in live rows: a V element, a K element (scores of both
    signs), a query that rounds to infinity, a score that overflows its f16
    accumulator; each as the walk has it, the other rows untouched."""
    H, Hkv, T, S = 8, 2, 5, 200
    g = torch.Generator(device="cuda").manual_seed(D)
    q = torch.randn(H, T, D, generator=g, device="cuda")
    k, v = (torch.randn(Hkv, S, D, generator=g, device="cuda").half() for _ in range(2))
    v[0, 10, 3], v[0, 70, 5], v[1, 100, 7] = float("inf"), float("nan"), 6e4
    k[1, 150, 2] = float("inf")
    q[1, 2, 4], q[6, 3, 9] = 1e5, float("nan")
    m = torch.from_numpy(causal_mask(T, S)).cuda()
    scale = float(np.float32(1.0 / np.sqrt(D)))
    got, want = be.flash_attn_ext(q, k, v, m, None, scale), walk(q, k, v, m, None, scale)
    assert bool(want.isnan().any()) and bool(want.isinf().any()) and bool(want.isfinite().any())
    assert torch.equal(got.isnan(), want.isnan())
    assert float((got != want)[~want.isnan()].float().mean()) <= 1e-3
