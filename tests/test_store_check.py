"""Host-side check of every MUL_MAT route's launch windows, without a GPU.

A dry-run context (ghip_init_dry_run) plans each op, takes a workspace
address range and, instead of launching, checks that the byte window every
kernel stores to -- worked out from that launch's own arguments -- lies inside
the buffers the op writes (dst, sub-sums, quantized activations, workspace).
The device pointers below are never dereferenced.  Every route (decode GEMV,
matrix-core decode, split K, the Q4_K / Q6_K / int8 GEMMs, batched planes)
must pass; a deliberately skewed leading dimension (GHIP_DEBUG_LDD_SKEW, a
wrong plan of the kind that once let kernels store past dst) must be caught.
"""
import ctypes as C
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "llama.rust_amd"))

W_BASE, X_BASE, D_BASE, S_BASE = 1 << 40, 2 << 40, 3 << 40, 5 << 40


def _lib():
    import ghip
    L = ghip.lib()
    L.ghip_init_dry_run.restype = C.c_int
    L.ghip_init_dry_run.argtypes = [C.POINTER(C.c_void_p)]
    return ghip, L


def _tensor(ghip, ty, ne, elem_bytes, blck, data):
    t = ghip.Tensor()
    t.type = ty
    ne = list(ne) + [1] * (4 - len(ne))
    t.ne[:] = ne
    nb0 = elem_bytes
    nb1 = ne[0] // blck * elem_bytes
    t.nb[:] = [nb0, nb1, nb1 * ne[1], nb1 * ne[1] * ne[2]]
    t.data = data
    return t


def _run(ty, k, n, m, planes=(1, 1), sub=False):
    ghip, L = _lib()
    ctx = C.c_void_p()
    assert L.ghip_init_dry_run(C.byref(ctx)) == 0
    try:
        blck, bs = ghip.BLOCK[ty]
        a = _tensor(ghip, ty, [k, n, 1, 1], bs, blck, W_BASE)
        b = _tensor(ghip, ghip.F32, [k, m, *planes], 4, 1, X_BASE)
        d = _tensor(ghip, ghip.F32, [n, m, *planes], 4, 1, D_BASE)
        if sub:
            st = L.ghip_mul_mat_subsums(ctx, C.byref(a), C.byref(b), C.c_void_p(S_BASE), None)
        else:
            st = L.ghip_mul_mat(ctx, C.byref(a), C.byref(b), C.byref(d), None)
        return st, L.ghip_last_error(ctx).decode()
    finally:
        L.ghip_free(ctx)


def _types():
    import ghip
    return [ghip.Q4_0, ghip.Q4_1, ghip.Q5_0, ghip.Q5_1, ghip.Q8_0, ghip.Q2_K, ghip.Q3_K, ghip.Q4_K, ghip.Q5_K,
            ghip.Q6_K, ghip.IQ4_NL, ghip.IQ4_XS, ghip.NVFP4, ghip.Q1_0, ghip.Q2_0, ghip.F32, ghip.F16, ghip.BF16,
            ghip.IQ2_XXS, ghip.IQ2_XS, ghip.IQ2_S, ghip.IQ3_XXS, ghip.IQ3_S, ghip.IQ1_S, ghip.IQ1_M]


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 8, 11, 16, 40, 64, 200, 512])
def test_every_route_stores_inside_its_buffers(m):
    import ghip
    for ty in _types():
        for k, n in [(4096, 4096), (4096, 14336), (14336, 4096), (1024, 100)]:
            st, msg = _run(ty, k, n, m)
            assert st == 0, (ty, k, n, m, msg)
            if m <= 8 and ty not in (ghip.F32, ghip.F16, ghip.BF16):
                st, msg = _run(ty, k, n, m, sub=True)
                assert st == 0, ("sub", ty, k, n, m, msg)


def test_batched_planes_store_inside_dst():
    import ghip
    for ty in (ghip.Q4_K, ghip.Q8_0, ghip.Q6_K):
        for m in (1, 5, 64):
            st, msg = _run(ty, 1024, 256, m, planes=(3, 2))
            assert st == 0, (ty, m, msg)


def test_skewed_leading_dimension_is_caught():
    """The same ops with a wrong leading dimension handed to the kernels: the
    check refuses the launch, for the decode, split-K and GEMM routes (from
    two activation rows: one row spans no stride)."""
    code = (
        "import sys; sys.path.insert(0, %r); sys.path.insert(0, %r)\n"
        "import test_store_check as T, ghip\n"
        "for ty, m in [(ghip.Q4_0, 2), (ghip.Q4_K, 2), (ghip.Q4_K, 6), (ghip.Q6_K, 6), (ghip.Q4_K, 64),"
        " (ghip.Q8_0, 64), (ghip.Q6_K, 128)]:\n"
        "    st, msg = T._run(ty, 4096, 4096, m)\n"
        "    assert st != 0 and 'store check' in msg, (ty, m, st, msg)\n"
        "    print(ty, m, msg)\n"
    ) % (os.path.join(ROOT, "tests"), os.path.join(ROOT, "llama.rust_amd"))
    env = dict(os.environ, GHIP_DEBUG_LDD_SKEW="1")
    r = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.count("store check") == 7


def test_mul_mat_id_stores_inside_dst():
    ghip, L = _lib()
    L.ghip_mul_mat_id.restype = C.c_int
    for ty in [t for t in _types() if t not in (ghip.F32, ghip.F16, ghip.BF16)] + [ghip.MXFP4]:
        for n_tokens, n_ids, ne11 in [(1, 4, 1), (12, 2, 2), (64, 4, 1)]:
            ctx = C.c_void_p()
            assert L.ghip_init_dry_run(C.byref(ctx)) == 0
            try:
                k, rows, n_as = 2048, 96, 8
                blck, bs = ghip.BLOCK[ty]
                a = _tensor(ghip, ty, [k, rows, n_as, 1], bs, blck, W_BASE)
                b = _tensor(ghip, ghip.F32, [k, ne11, n_tokens, 1], 4, 1, X_BASE)
                ids = _tensor(ghip, ghip.I32, [n_ids, n_tokens, 1, 1], 4, 1, S_BASE)
                d = _tensor(ghip, ghip.F32, [rows, n_ids, n_tokens, 1], 4, 1, D_BASE)
                st = L.ghip_mul_mat_id(ctx, C.byref(a), C.byref(b), C.byref(ids), C.byref(d), None)
                assert st == 0, (ty, n_tokens, L.ghip_last_error(ctx).decode())
            finally:
                L.ghip_free(ctx)


def _grouped(ty, m, pad):
    """Two sibling MUL_MATs, the first one's weight rows `pad` blocks further
    apart: does a graph run them as one launch?  (A dry run under
    GHIP_DEBUG_LDD_SKEW: the skew reaches single launches only.)"""
    ghip, L = _lib()
    ctx = C.c_void_p()
    assert L.ghip_init_dry_run(C.byref(ctx)) == 0
    try:
        blck, bs = ghip.BLOCK[ty]
        k, n = 1024, 512
        ws = [_tensor(ghip, ty, [k, n, 1, 1], bs, blck, W_BASE + (i << 32)) for i in range(2)]
        for d, rows in ((1, 1), (2, n), (3, n)):
            ws[0].nb[d] += pad * bs * rows
        x = _tensor(ghip, ghip.F32, [k, m, 1, 1], 4, 1, X_BASE)
        ds = [_tensor(ghip, ghip.F32, [n, m, 1, 1], 4, 1, D_BASE + (i << 32)) for i in range(2)]
        arr = (ghip.GNode * 2)()
        for i in range(2):
            arr[i].op = ghip.OP_MUL_MAT
            arr[i].src[0], arr[i].src[1] = C.pointer(ws[i]), C.pointer(x)
            arr[i].dst = C.pointer(ds[i])
        st = L.ghip_graph_compute(ctx, arr, 2, None)
        assert st == 0 or "store check" in L.ghip_last_error(ctx).decode()
        return st == 0
    finally:
        L.ghip_free(ctx)


def test_groups_share_the_weight_row_stride():
    """A grouped launch has one row stride for its members: siblings that
    differ in it (a padded or strided view beside a packed matrix) run alone."""
    code = (
        "import sys; sys.path.insert(0, %r); sys.path.insert(0, %r)\n"
        "import test_store_check as T, ghip\n"
        "for ty, m in [(ghip.Q4_K, 2), (ghip.Q4_K, 6), (ghip.Q4_K, 24), (ghip.Q4_K, 100), (ghip.Q5_K, 2), (ghip.Q4_0, 2),"
        " (ghip.Q8_0, 4)]:\n"
        "    assert T._grouped(ty, m, 0), (ty, m)\n"
        "    assert not T._grouped(ty, m, 1), (ty, m)\n"
    ) % (os.path.join(ROOT, "tests"), os.path.join(ROOT, "llama.rust_amd"))
    env = dict(os.environ, GHIP_DEBUG_LDD_SKEW="1")
    r = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


def _route(ty, k, n, m):
    """the kernel that stores a MUL_MAT's dst (under GHIP_DEBUG_LDD_SKEW the store
    check refuses it by name)"""
    st, msg = _run(ty, k, n, m)
    assert st != 0 and "store check" in msg, msg
    return msg.split(" of ", 1)[1].split(" ", 1)[0]


def _switches():
    import ghip
    for ty, var in [(ghip.Q4_K, "GHIP_GEMM_MIN_ROWS"), (ghip.Q5_K, "GHIP_GEMM_Q5K_MIN_ROWS"),
                    (ghip.Q6_K, "GHIP_GEMM_Q6K_MIN_ROWS"), (ghip.Q4_0, "GHIP_GEMM_Q8_MIN_ROWS"),
                    (ghip.Q8_0, "GHIP_GEMM_Q8_MIN_ROWS"), (ghip.IQ4_XS, "GHIP_GEMM_Q8_MIN_ROWS")]:
        for m in (20, 40):
            assert "_kq32_" in _route(ty, 4096, 4096, m), (ty, m)
            os.environ[var] = str(m)
            at = _route(ty, 4096, 4096, m)
            os.environ[var] = str(m + 1)
            below = _route(ty, 4096, 4096, m)
            del os.environ[var]
            assert "gemm" in at and "_kq32_" not in at, (ty, m, at)
            assert "gemm" not in below, (ty, m, below)


def test_row_switches_part_gemm_and_decode():
    """GHIP_GEMM_*_MIN_ROWS, where set: the prefill GEMM from that many rows, the
    decode kernels below."""
    code = ("import sys; sys.path.insert(0, %r); sys.path.insert(0, %r)\n"
            "import test_store_check as T\nT._switches()\n") % (os.path.join(ROOT, "tests"), os.path.join(ROOT, "llama.rust_amd"))
    env = dict(os.environ, GHIP_DEBUG_LDD_SKEW="1")
    r = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


def _short_batches():
    import ghip
    for ty, k, n, m, tiles in [
            (ghip.Q4_K, 4096, 8192, 40, True), (ghip.Q4_K, 8192, 8192, 40, False), (ghip.Q4_K, 7168, 6144, 40, False),
            (ghip.Q4_K, 7168, 14336, 24, True), (ghip.Q4_K, 8192, 4096, 24, False), (ghip.Q5_K, 8192, 14336, 40, False),
            (ghip.Q5_K, 8192, 14336, 32, True), (ghip.Q6_K, 14336, 1024, 16, False), (ghip.Q6_K, 14336, 4096, 9, True),
            (ghip.Q6_K, 8192, 1024, 13, True), (ghip.Q6_K, 20480, 1024, 9, True), (ghip.IQ4_XS, 14336, 1024, 9, False),
            (ghip.IQ4_XS, 14336, 1024, 12, True), (ghip.Q8_0, 4096, 8192, 40, True)]:
        name = _route(ty, k, n, m)
        assert ("_kq32_" in name) == tiles, (ty, k, n, m, name)


def test_short_batch_routes():
    """Which short batches take the 32 x 32 tiles: not a long K of few or many
    weight rows that the GEMMs and decode kernels run faster."""
    code = ("import sys; sys.path.insert(0, %r); sys.path.insert(0, %r)\n"
            "import test_store_check as T\nT._short_batches()\n") % (os.path.join(ROOT, "tests"), os.path.join(ROOT, "llama.rust_amd"))
    env = dict(os.environ, GHIP_DEBUG_LDD_SKEW="1")
    r = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
