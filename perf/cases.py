"""The work that performance changes are measured on: MUL_MAT, MUL_MAT_ID and
FLASH_ATTN_EXT as a model runtime calls them through the Python binding
(llama.rust_amd/ghip.py).  Weights are GGUF blocks built here from the seed,
so that `exact` can state the same arithmetic in 64 bits without the package.
"""
import math
import os
import sys
import weakref

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "llama.rust_amd"))
import ghip  # noqa: E402

DEV = "cuda"
TYPES = {"q4_0": ghip.Q4_0, "q8_0": ghip.Q8_0, "q2_K": ghip.Q2_K, "q3_K": ghip.Q3_K, "q4_K": ghip.Q4_K,
         "q5_K": ghip.Q5_K, "q6_K": ghip.Q6_K, "iq4_xs": ghip.IQ4_XS, "mxfp4": ghip.MXFP4, "f16": ghip.F16,
         "bf16": ghip.BF16}
# (name, weight type, the activation it reads, its output's width) of one
# decoder layer's products; q/k/v and gate/up share an input
LAYER = [("q", "q4_K", "x_attn", "hidden"), ("k", "q4_K", "x_attn", "kv"), ("v", "q4_K", "x_attn", "kv"),
         ("o", "q4_K", "attn_out", "hidden"), ("gate", "q4_K", "x_ffn", "ffn"), ("up", "q4_K", "x_ffn", "ffn"),
         ("down", "q6_K", "h_ffn", "hidden")]


def listed():
    return [
        # one small product by itself, as a program that runs its graph node by
        # node calls it: launch and call latency
        {"name": "gemv_q4_0", "kind": "mul_mat", "type": "q4_0", "K": 4096, "N": 4096, "M": 1, "registered": False},
        # token generation: the seven products of an 8B layer (Q4_K_M mix), one
        # token, captured once and replayed as a generation loop does
        {"name": "decode_layer", "kind": "layer", "hidden": 4096, "kv": 1024, "ffn": 14336, "M": 1},
        # the same for six sequences that generate together
        {"name": "decode_layer_6", "kind": "layer", "hidden": 4096, "kv": 1024, "ffn": 14336, "M": 6},
        # a short user turn: 37 new tokens through the layer
        {"name": "prompt_layer_37", "kind": "layer", "hidden": 4096, "kv": 1024, "ffn": 14336, "M": 37},
        # a full prefill batch
        {"name": "prefill_layer_512", "kind": "layer", "hidden": 4096, "kv": 1024, "ffn": 14336, "M": 512},
        # prefill of a 3-bit model's gate / up product, a ragged batch
        {"name": "prefill_q3_K", "kind": "mul_mat", "type": "q3_K", "K": 4096, "N": 14336, "M": 300, "registered": True},
        # prefill of a model kept in half precision
        {"name": "prefill_f16", "kind": "mul_mat", "type": "f16", "K": 4096, "N": 4096, "M": 200, "registered": False},
        # mixture of experts, prefill batch, 32 MXFP4 experts, top-4
        {"name": "moe_mxfp4_gate_up", "kind": "moe", "type": "mxfp4", "K": 2880, "N": 5760, "experts": 32, "top": 4,
         "tokens": 256, "registered": True},
        # mixture of experts with K-quant experts, a short prompt
        {"name": "moe_q4_K", "kind": "moe", "type": "q4_K", "K": 2048, "N": 1536, "experts": 64, "top": 8,
         "tokens": 64, "registered": False},
        # attention, one new token over a long cache (32 query heads on 8)
        {"name": "attn_decode", "kind": "attn", "T": 1, "S": 8192, "H": 32, "H_kv": 8, "D": 128, "sinks": False},
        # attention, a prefill chunk at the end of a long cache
        {"name": "attn_prefill", "kind": "attn", "T": 512, "S": 8192, "H": 32, "H_kv": 8, "D": 128, "sinks": False},
        # attention, a short user turn over a conversation's cache, with sinks
        {"name": "attn_prompt", "kind": "attn", "T": 37, "S": 1061, "H": 64, "H_kv": 8, "D": 64, "sinks": True},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["mul_mat", "layer", "moe", "attn"])
    if kind == "mul_mat":
        while True:
            ty = rng.choice(["q4_0", "q8_0", "q2_K", "q3_K", "q4_K", "q5_K", "q6_K", "iq4_xs", "f16", "bf16"])
            c = {"kind": kind, "type": ty, "K": 256 * _log_int(rng, 2, 56), "N": _log_int(rng, 512, 16384),
                 "M": _log_int(rng, 1, 512), "registered": rng.random() < 0.5}
            if c["M"] * c["K"] * c["N"] <= (512 * 4096 * 4096 if ty in ("f16", "bf16") else 300 * 4096 * 14336):
                return c
    if kind == "layer":
        hidden = 256 * rng.randint(4, 16)
        return {"kind": kind, "hidden": hidden, "kv": hidden // rng.choice([1, 2, 4, 8]),
                "ffn": 256 * rng.randint(hidden // 128, 56), "M": _log_int(rng, 1, 512)}
    if kind == "moe":
        ty = rng.choice(["mxfp4", "q4_K", "q5_K", "q6_K"])
        blk = 32 if ty == "mxfp4" else 256
        return {"kind": kind, "type": ty, "K": blk * rng.randint(768 // blk, 2880 // blk), "N": rng.randint(768, 5760 if blk == 32 else 2304),
                "experts": rng.choice([8, 16, 32, 64] if blk == 256 else [8, 16, 32]), "top": rng.choice([1, 2, 4, 6]),
                "tokens": _log_int(rng, 1, 256 if blk == 32 else 64),
                "registered": ty == "mxfp4" and rng.random() < 0.5}  # K-quant experts are read as they are
    D = rng.choice([64, 128])
    T = _log_int(rng, 1, 512)
    H_kv = rng.choice([2, 4, 8])
    return {"kind": "attn", "T": T, "S": T + _log_int(rng, 1, 8192 - T if T >= 64 or T == 1 else 2048), "H": H_kv * rng.choice([1, 2, 4, 8 if D == 64 else 4]),
            "H_kv": H_kv, "D": D, "sinks": rng.random() < 0.3}


# ------------------------------------------------------------ GGUF weights
# Codes follow clipped normals as a quantizer leaves them; scales vary from
# block to block; the weights' spread is about 0.02.

KV_IQ4 = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]
KV_FP4 = [0, 1, 2, 3, 4, 6, 8, 12, 0, -1, -2, -3, -4, -6, -8, -12]


def _codes(g, shape, centre, spread, lo, hi):
    return torch.randn(shape, generator=g, device=DEV).mul_(spread).add_(centre).round_().clamp_(lo, hi).to(torch.uint8)


def _f16_bytes(x):
    return x.to(torch.float16).contiguous().view(torch.uint8).view(*x.shape, 2)


def _nibbles(q):
    """[.., 32] codes -> [.., 16] bytes, element j low and element j + 16 high"""
    return q[..., :16] | (q[..., 16:] << 4)


def _pack_k4(sc, mn):
    """eight 6-bit scales and mins -> the 12 bytes of Q4_K / Q5_K"""
    out = torch.empty(*sc.shape[:-1], 12, dtype=torch.uint8, device=DEV)
    out[..., 0:4] = sc[..., :4] | ((sc[..., 4:] >> 4) << 6)
    out[..., 4:8] = mn[..., :4] | ((mn[..., 4:] >> 4) << 6)
    out[..., 8:12] = (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)
    return out


def _unpack_k4(b):
    lo, hi, x = b[..., 0:4], b[..., 4:8], b[..., 8:12]
    return (torch.cat([lo & 63, (x & 15) | ((lo >> 6) << 4)], -1),
            torch.cat([hi & 63, (x >> 4) | ((hi >> 6) << 4)], -1))


def make_weight(ty, rows, K, g):
    """uint8 [rows, row bytes] of GGUF blocks, or a f16 / bf16 matrix [rows, K]"""
    if ty in ("f16", "bf16"):
        return (torch.randn((rows, K), generator=g, device=DEV) * 0.02).to(torch.float16 if ty == "f16" else torch.bfloat16)
    blk = ghip.BLOCK[TYPES[ty]][0]
    B = (rows, K // blk)
    vary = 0.7 + 0.6 * torch.rand(B, generator=g, device=DEV)
    if ty == "q4_0":
        parts = [_f16_bytes(vary * 0.0065), _nibbles(_codes(g, (*B, 32), 8, 3, 0, 15))]
    elif ty == "q8_0":
        q = torch.randn((*B, 32), generator=g, device=DEV).mul_(45).round_().clamp_(-127, 127).to(torch.int8)
        parts = [_f16_bytes(vary * 0.00045), q.view(torch.uint8)]
    elif ty in ("q4_K", "q5_K"):
        sc, mn = _codes(g, (*B, 8), 50, 7, 1, 63), _codes(g, (*B, 8), 50, 7, 0, 63)
        top, d = (15, 0.006) if ty == "q4_K" else (31, 0.003)
        q = _codes(g, (*B, 4, 2, 32), top / 2, top / 5, 0, top)
        head = [_f16_bytes(vary * (d / 50)), _f16_bytes(vary * (d * top / 2 / 50)), _pack_k4(sc, mn)]
        if ty == "q5_K":
            bits = torch.zeros((*B, 32), dtype=torch.uint8, device=DEV)
            for j in range(4):
                bits |= ((q[..., j, 0, :] >> 4) << (2 * j)) | ((q[..., j, 1, :] >> 4) << (2 * j + 1))
            head.append(bits)
        parts = head + [((q[..., 0, :] & 15) | ((q[..., 1, :] & 15) << 4)).reshape(*B, 128)]
    elif ty == "q6_K":
        q = _codes(g, (*B, 2, 4, 32), 32, 10, 0, 63)
        ql = torch.cat([(q[..., 0, :] & 15) | ((q[..., 2, :] & 15) << 4), (q[..., 1, :] & 15) | ((q[..., 3, :] & 15) << 4)], -1)
        qh = (q[..., 0, :] >> 4) | ((q[..., 1, :] >> 4) << 2) | ((q[..., 2, :] >> 4) << 4) | ((q[..., 3, :] >> 4) << 6)
        sc = torch.randn((*B, 16), generator=g, device=DEV).mul_(12).add_(80).round_().clamp_(20, 127)
        sc = (sc * (1 - 2 * (torch.rand((*B, 16), generator=g, device=DEV) < 0.5).float())).to(torch.int8)
        parts = [ql.reshape(*B, 128), qh.reshape(*B, 64), sc.view(torch.uint8), _f16_bytes(vary * (0.002 / 80))]
    elif ty == "q2_K":
        sc = _codes(g, (*B, 16), 11, 2, 1, 15) | (_codes(g, (*B, 16), 11, 2, 0, 15) << 4)
        q = _codes(g, (*B, 2, 4, 32), 1.5, 0.9, 0, 3)
        qs = q[..., 0, :] | (q[..., 1, :] << 2) | (q[..., 2, :] << 4) | (q[..., 3, :] << 6)
        parts = [sc, qs.reshape(*B, 64), _f16_bytes(vary * (0.02 / 11)), _f16_bytes(vary * (0.03 / 11))]
    elif ty == "q3_K":
        q = _codes(g, (*B, 2, 4, 32), 4, 1.6, 0, 7)
        qs = (q[..., 0, :] & 3) | ((q[..., 1, :] & 3) << 2) | ((q[..., 2, :] & 3) << 4) | ((q[..., 3, :] & 3) << 6)
        hm = torch.zeros((*B, 32), dtype=torch.uint8, device=DEV)
        for n in range(2):
            for j in range(4):
                hm |= (q[..., n, j, :] >> 2) << (4 * n + j)
        s = _codes(g, (*B, 16), 54, 5, 1, 63)
        flip = torch.rand((*B, 16), generator=g, device=DEV) < 0.5
        s = torch.where(flip, 64 - s, s)  # the 6-bit scale is offset by 32
        lo = (s[..., :8] & 15) | ((s[..., 8:] & 15) << 4)
        hi = (s[..., 0:4] >> 4) | ((s[..., 4:8] >> 4) << 2) | ((s[..., 8:12] >> 4) << 4) | ((s[..., 12:16] >> 4) << 6)
        parts = [hm, qs.reshape(*B, 64), lo, hi, _f16_bytes(vary * (0.0125 / 22))]
    elif ty == "iq4_xs":
        ls = _codes(g, (*B, 8), 54, 5, 1, 63)
        ls = torch.where(torch.rand((*B, 8), generator=g, device=DEV) < 0.5, 64 - ls, ls)
        sh = torch.zeros(B, dtype=torch.int32, device=DEV)
        for i in range(8):
            sh |= (ls[..., i].int() >> 4) << (2 * i)
        sl = (ls[..., 0::2] & 15) | ((ls[..., 1::2] & 15) << 4)
        parts = [_f16_bytes(vary * (0.0004 / 22)), (sh & 255).to(torch.uint8)[..., None], (sh >> 8).to(torch.uint8)[..., None],
                 sl, _nibbles(_codes(g, (*B, 8, 32), 7.5, 3, 0, 15)).reshape(*B, 128)]
    elif ty == "mxfp4":
        e = torch.randint(119, 122, B, generator=g, device=DEV).to(torch.uint8)[..., None]
        parts = [e, _nibbles(torch.randint(0, 16, (*B, 32), generator=g, device=DEV, dtype=torch.uint8))]
    return torch.cat(parts, -1).reshape(rows, -1)


def dequantize(ty, w, K):
    """The float64 values [rows, K] of make_weight's blocks, by the formats' definitions."""
    if ty in ("f16", "bf16"):
        return w.double()
    blk, size = ghip.BLOCK[TYPES[ty]]
    rows = w.shape[0]
    b = w.view(rows, K // blk, size)
    f16 = lambda at: b[..., at:at + 2].contiguous().view(torch.float16).double()  # noqa: E731  [.., 1]
    nib = lambda q: torch.cat([q & 15, q >> 4], -1)  # noqa: E731
    if ty == "q4_0":
        v = f16(0) * (nib(b[..., 2:]).double() - 8)
    elif ty == "q8_0":
        v = f16(0) * b[..., 2:].contiguous().view(torch.int8).double()
    elif ty in ("q4_K", "q5_K"):
        sc, mn = _unpack_k4(b[..., 4:16])
        qs = b[..., size - 128:].reshape(rows, -1, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], -2)  # [.., chunk, half, 32]
        if ty == "q5_K":
            qh = b[..., 16:48]
            q = q | (torch.stack([torch.stack([(qh >> (2 * j + h)) & 1 for h in range(2)], -2) for j in range(4)], -3) << 4)
        q = q.reshape(rows, -1, 8, 32)
        v = f16(0)[..., None] * sc.double()[..., None] * q.double() - f16(2)[..., None] * mn.double()[..., None]
    elif ty == "q6_K":
        ql, qh = b[..., 0:128].reshape(rows, -1, 2, 2, 32), b[..., 128:192].reshape(rows, -1, 2, 32)
        sc = b[..., 192:208].contiguous().view(torch.int8).double()
        q = torch.stack([(ql[..., 0, :] & 15) | ((qh & 3) << 4), (ql[..., 1, :] & 15) | (((qh >> 2) & 3) << 4),
                         (ql[..., 0, :] >> 4) | (((qh >> 4) & 3) << 4), (ql[..., 1, :] >> 4) | ((qh >> 6) << 4)], -2)
        v = f16(208)[..., None] * sc[..., None] * (q.reshape(rows, -1, 16, 16).double() - 32)
    elif ty == "q2_K":
        sc, qs = b[..., 0:16], b[..., 16:80].reshape(rows, -1, 2, 32)
        q = torch.stack([(qs >> (2 * j)) & 3 for j in range(4)], -2).reshape(rows, -1, 16, 16).double()
        v = f16(80)[..., None] * (sc & 15).double()[..., None] * q - f16(82)[..., None] * (sc >> 4).double()[..., None]
    elif ty == "q3_K":
        hm, qs = b[..., 0:32], b[..., 32:96].reshape(rows, -1, 2, 32)
        lo = torch.cat([b[..., 96:104] & 15, b[..., 96:104] >> 4], -1)
        hi = torch.cat([(b[..., 104:108] >> (2 * j)) & 3 for j in range(4)], -1)
        sc = (lo | (hi << 4)).double() - 32
        q = torch.stack([(qs >> (2 * j)) & 3 for j in range(4)], -2)
        h = torch.stack([torch.stack([(hm >> (4 * n + j)) & 1 for j in range(4)], -2) for n in range(2)], -3)
        q = (q.double() - 4 * (1 - h.double())).reshape(rows, -1, 16, 16)
        v = f16(108)[..., None] * sc[..., None] * q
    elif ty == "iq4_xs":
        sh = b[..., 2].int() | (b[..., 3].int() << 8)
        lo = torch.stack([b[..., 4:8] & 15, b[..., 4:8] >> 4], -1).reshape(rows, -1, 8).int()
        ls = torch.stack([lo[..., i] | (((sh >> (2 * i)) & 3) << 4) for i in range(8)], -1).double() - 32
        kv = torch.tensor(KV_IQ4, dtype=torch.float64, device=DEV)
        v = f16(0)[..., None] * ls[..., None] * kv[nib(b[..., 8:].reshape(rows, -1, 8, 16)).long()]
    elif ty == "mxfp4":
        kv = torch.tensor(KV_FP4, dtype=torch.float64, device=DEV)
        v = torch.exp2(b[..., 0:1].double() - 128) * kv[nib(b[..., 1:]).long()]
    return v.reshape(rows, K)


def activation_values(ty, x, n_mat=0):
    """float64 values of the rows of x as the weight type's dot reads them:
    rounded to f16 / bf16, or quantized to Q8_0 / Q8_K.  Rows before n_mat
    take the Q8_K scale 127 / max|x|, the others -127 / x at the first max|x|."""
    if ty in ("f16", "bf16"):
        return x.to(torch.float16 if ty == "f16" else torch.bfloat16).double()
    blk = 32 if ty in ("q4_0", "q8_0", "mxfp4") else 256
    b = x.reshape(x.shape[0], -1, blk)
    amax = b.abs().amax(-1, keepdim=True)
    over = lambda n, v: torch.full_like(v, n) / v  # noqa: E731  (a number / tensor rounds twice in torch)
    if blk == 32:
        q = (b * torch.where(amax > 0, over(127.0, amax), torch.zeros_like(amax))).round()
        return (q.double() * (amax / 127.0).to(torch.float16).double()).reshape(x.shape)
    first = torch.gather(b, -1, (b.abs() == amax).to(torch.uint8).argmax(-1, keepdim=True))
    mat = (torch.arange(x.shape[0], device=DEV) < n_mat).view(-1, 1, 1)
    iscale = torch.where(mat, over(127.0, amax), over(-127.0, first))
    iscale = torch.where(amax > 0, iscale, torch.ones_like(iscale))
    q = (b * iscale).round().clamp(-128, 127)
    return (q.double() * over(1.0, iscale).double()).reshape(x.shape)


def _product(ty, w, x, K, N):
    M = x.shape[0]
    n_mat = M - M % 4 if ty == "q4_K" and N % 8 == 0 else 0  # rows quantized four at a time
    return activation_values(ty, x, n_mat) @ dequantize(ty, w, K).t()


# ------------------------------------------------------------ cases

_backend = None


def _be():
    global _backend
    if _backend is None:
        _backend = ghip.Backend(0)
    return _backend


class Registered:
    """A loaded model's weight: registered until it is dropped."""

    def __init__(self, w, ty, K):
        self.w = w
        _be().register_weight(w, TYPES[ty], K)
        weakref.finalize(self, _be().unregister_weight, w, TYPES[ty], K)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _layer_shapes(case):
    width = {"hidden": case["hidden"], "kv": case["kv"], "ffn": case["ffn"]}
    return [(nm, ty, x, case["ffn"] if x == "h_ffn" else case["hidden"], width[n]) for nm, ty, x, n in LAYER]


def _inputs(case, seed):
    """tensors made from the seed alone"""
    g, kind = _gen(seed), case["kind"]
    if kind == "mul_mat":
        return {"x": torch.randn((case["M"], case["K"]), generator=g, device=DEV),
                "w": make_weight(case["type"], case["N"], case["K"], g)}
    if kind == "layer":
        s = {n: torch.randn((case["M"], case["ffn"] if n == "h_ffn" else case["hidden"]), generator=g, device=DEV)
             for n in ("x_attn", "attn_out", "x_ffn", "h_ffn")}
        for nm, ty, _, K, N in _layer_shapes(case):
            s[nm] = make_weight(ty, N, K, g)
        return s
    if kind == "moe":
        logits = torch.randn((case["tokens"], case["experts"]), generator=g, device=DEV)
        return {"x": torch.randn((case["tokens"], 1, case["K"]), generator=g, device=DEV),
                "ids": logits.topk(case["top"], -1).indices.to(torch.int32).contiguous(),
                "w": make_weight(case["type"], case["experts"] * case["N"], case["K"], g).view(case["experts"], case["N"], -1)}
    T, S, H, Hk, D = (case[n] for n in ("T", "S", "H", "H_kv", "D"))
    s = {"q": torch.randn((H, T, D), generator=g, device=DEV),
         "k": torch.randn((Hk, S, D), generator=g, device=DEV).half(),
         "v": torch.randn((Hk, S, D), generator=g, device=DEV).half(),
         "sinks": torch.randn(H, generator=g, device=DEV) if case["sinks"] else None}
    hidden = torch.arange(S, device=DEV)[None, :] > torch.arange(S - T, S, device=DEV)[:, None]
    s["mask"] = torch.zeros((T, S), dtype=torch.float16, device=DEV).masked_fill_(hidden, float("-inf"))
    return s


def prepare(case, seed):
    s, be, kind = _inputs(case, seed), _be(), case["kind"]
    s["case"] = case
    new = lambda *shape: torch.empty(shape, dtype=torch.float32, device=DEV)  # noqa: E731
    if kind == "mul_mat":
        s["out"] = new(case["M"], case["N"])
        if case["registered"]:
            s["kept"] = Registered(s["w"], case["type"], case["K"])
    elif kind == "moe":
        s["out"] = new(case["tokens"], case["top"], case["N"])
        if case["registered"]:
            s["kept"] = Registered(s["w"], case["type"], case["K"])
    elif kind == "attn":
        s["out"] = new(case["T"], case["H"], case["D"])
    else:
        shapes = _layer_shapes(case)
        s["kept"] = [Registered(s[nm], ty, K) for nm, ty, _, K, _ in shapes]
        s["out"] = {nm: new(case["M"], N) for nm, _, _, _, N in shapes}
        s["nodes"] = [ghip.mul_mat_node(s[nm], TYPES[ty], K, s[x], s["out"][nm]) for nm, ty, x, K, _ in shapes]
        if case["M"] <= 8:  # a generation loop replays its step
            be.graph_compute(s["nodes"])
            torch.cuda.synchronize()
            s["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(s["graph"]):
                be.graph_compute(s["nodes"])
    return s


def run(s):
    case, be = s["case"], _be()
    kind = case["kind"]
    if kind == "mul_mat":
        return be.mul_mat(s["w"], TYPES[case["type"]], case["K"], s["x"], out=s["out"])
    if kind == "moe":
        return be.mul_mat_id(s["w"], case["K"], s["x"], s["ids"], out=s["out"], ty=TYPES[case["type"]])
    if kind == "attn":
        return be.flash_attn_ext(s["q"], s["k"], s["v"], s["mask"], s["sinks"], 1.0 / math.sqrt(case["D"]), out=s["out"])
    if "graph" in s:
        s["graph"].replay()
    else:
        be.graph_compute(s["nodes"])
    return s["out"]


def exact(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind == "mul_mat":
        return _product(case["type"], s["w"], s["x"], case["K"], case["N"])
    if kind == "layer":
        return {nm: _product(ty, s[nm], s[x], K, N) for nm, ty, x, K, N in _layer_shapes(case)}
    if kind == "moe":
        a = activation_values(case["type"], s["x"][:, 0])
        out = torch.empty((case["tokens"], case["top"], case["N"]), dtype=torch.float64, device=DEV)
        for e in range(case["experts"]):
            t, j = (s["ids"] == e).nonzero(as_tuple=True)
            if t.numel():
                out[t, j] = a[t] @ dequantize(case["type"], s["w"][e], case["K"]).t()
        return out
    T, S, H, Hk, D = (case[n] for n in ("T", "S", "H", "H_kv", "D"))
    q = s["q"].half().double()  # an F16 cache reads the query in f16
    out = torch.empty((T, H, D), dtype=torch.float64, device=DEV)
    for h in range(H):
        k, v = s["k"][h // (H // Hk)].double(), s["v"][h // (H // Hk)].double()
        z = q[h] @ k.t().contiguous() / math.sqrt(D) + s["mask"].double()
        if case["sinks"]:
            z = torch.cat([z, s["sinks"][h].double().expand(T, 1)], -1)
            v = torch.cat([v, torch.zeros((1, D), dtype=torch.float64, device=DEV)])
        out[:, h] = torch.softmax(z, -1) @ v
    return out


def work(case):
    kind = case["kind"]
    if kind == "attn":
        T, S, H, Hk, D = (case[n] for n in ("T", "S", "H", "H_kv", "D"))
        keys = T * (S - T) + T * (T + 1) // 2
        return {"bytes": 4 * Hk * S * D + 8 * T * H * D + 2 * T * S, "flops": 4 * D * H * keys}
    size = lambda ty, n: n * 2 if ty in ("f16", "bf16") else n // ghip.BLOCK[TYPES[ty]][0] * ghip.BLOCK[TYPES[ty]][1]  # noqa: E731
    if kind == "layer":
        M, total = case["M"], {"bytes": 4 * case["M"] * (3 * case["hidden"] + case["ffn"]), "flops": 0}
        for _, ty, _, K, N in _layer_shapes(case):
            total["bytes"] += size(ty, K) * N + 4 * M * N
            total["flops"] += 2 * M * K * N
        return total
    K, N = case["K"], case["N"]
    if kind == "mul_mat":
        return {"bytes": size(case["type"], K) * N + 4 * case["M"] * (K + N), "flops": 2 * case["M"] * K * N}
    pairs = case["tokens"] * case["top"]
    # the experts that are met, on average over the routing's draws
    met = case["experts"] * (1 - (1 - case["top"] / case["experts"]) ** case["tokens"])
    return {"bytes": int(met * size(case["type"], K) * N) + 4 * case["tokens"] * (K + case["top"]) + 4 * pairs * N,
            "flops": 2 * pairs * K * N}


def tolerance(case):
    if case["kind"] == "attn":
        if case["T"] == 1 and case["S"] >= 512:  # 32-bit scores and sums; 2.5e-7 from exact
            return {"rel": 1e-6, "max": 1e-5}
        # from 64 rows f16 probabilities (2e-4 from exact); below, the output
        # accumulates in f16 over the keys (5e-3 at 1000 keys)
        return {"rel": 1e-3, "max": 1e-2} if case["T"] >= 64 else {"rel": 2e-2, "max": 2e-1}
    # exact integer block sums (exact products of halves), folded in 32 bits: 1e-7 to 2e-7 from exact
    return {"rel": 1e-6, "max": 1e-5}
