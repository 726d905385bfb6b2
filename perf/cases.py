"""Performance cases of the quantized linear path: what a program serving a
Llama-3-8B-shaped model (hidden 4096, gate/up 14336, QKV 6144, and its
tensor-parallel shards) has this library do on one GPU.

Every case is one call (or the two or three calls that belong together)
through the Python binding, on weights that are already quantized and laid
out, with the output buffer in hand, as a serving loop keeps them:

  w4        one W4A16 linear: a decode row, a decode batch, a larger batch of
            decode rows (the range between decode and prefill), a prompt
  w4_mlp    the W4A16 SwiGLU block in one call
  w4_perm   a W4A16 linear with GPTQ act-order weights, prepared at load
  w8        a W8 weight-only layer with fp32 activations (SNEPPXQLayer, the
            drop-in for the fp32 matmuls of attention and the LM head)
  w8a8      a W8A8 linear from bf16 activations (int8 per token or fp8 per
            tensor, quantized inside the call)
  mx        an MX linear: fp32 activations quantized, brought into the matrix
            cores' form where the format needs it, and multiplied
  quant     a weight matrix quantized on the device at load time

Sizes, types and options are those of bench.py and the tests.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sneppx-alg_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import sneppx_quant  # noqa: E402

DEV = "cuda:0"
BF16, F32 = torch.bfloat16, torch.float32


def _w4(name, M, N, K, group=128, zeros=True, bias=False, out="bf16"):
    return {"name": name, "kind": "w4", "M": M, "N": N, "K": K, "group": group, "zeros": zeros, "bias": bias,
            "out": out}


def listed():
    return [
        # one rank's share of a W8 projection under tensor parallelism, one
        # token: the smallest call, where launch and latency are what counts
        {"name": "w8_token_shard", "kind": "w8", "M": 1, "N": 512, "K": 4096, "bias": False},
        # a prompt of 384 tokens through an attention projection of the fp32
        # model whose weights were swapped for W8 layers
        {"name": "w8_prompt", "kind": "w8", "M": 384, "N": 4096, "K": 4096, "bias": True},
        # single-stream decoding: one token through a gate or up projection
        _w4("w4_token", 1, 11008, 4096),
        # 16 streams decoding together, down projection (long K)
        _w4("w4_batch16_down", 16, 4096, 14336),
        # a loaded server: 96 decode rows in one step, QKV projection
        _w4("w4_batch96_qkv", 96, 6144, 4096, bias=True),
        # 32 decode rows through the whole SwiGLU block
        {"name": "w4_mlp_batch32", "kind": "w4_mlp", "M": 32, "N": 4096, "K": 4096, "F": 14336, "zeros": True},
        # a packed batch of 16 decode rows and 8 prefill chunks (1849 tokens)
        # through the SwiGLU block: the largest call
        {"name": "w4_mlp_prefill", "kind": "w4_mlp", "M": 1849, "N": 4096, "K": 4096, "F": 14336, "zeros": True},
        # GPTQ act-order weights, 8 streams decoding
        {"name": "w4_perm_batch8", "kind": "w4_perm", "M": 8, "N": 11008, "K": 4096, "out": "bf16"},
        # W8A8 prefill, activations quantized per token inside the call
        {"name": "w8a8_int8_prefill", "kind": "w8a8", "fp8": False, "M": 2048, "N": 14336, "K": 4096, "bias": False},
        # W8A8 fp8 decode batch of 48 rows
        {"name": "w8a8_fp8_batch48", "kind": "w8a8", "fp8": True, "M": 48, "N": 14336, "K": 4096, "bias": False},
        # MXFP8 linear of a 512-token chunk, from fp32 activations
        {"name": "mxfp8_chunk512", "kind": "mx", "fmt": "mxfp8_e4m3", "M": 512, "N": 4096, "K": 4096, "out": "bf16"},
        # a gate projection quantized to W4 while a model loads
        {"name": "quant_w4_load", "kind": "quant", "how": "w4_awq", "N": 14336, "K": 4096, "group": 128},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["w4", "w4", "w4", "w4_mlp", "w4_perm", "w8", "w8a8", "w8a8", "mx", "quant"])
    while True:
        M, N, K = _log(rng, 1, 2048), _log(rng, 256, 16384), 128 * _log(rng, 4, 112)
        if M * N * K <= 4e10:
            break
    if rng.random() < 0.7:
        N = (N + 15) // 16 * 16          # model dimensions; the others are vocabulary- or head-shaped
    out = rng.choice(["bf16", "bf16", "f32"])
    if kind == "w4":
        group = rng.choice([128, 128, 128, 128, 64, 32, 256])
        c = _w4("", M, N, (K + group - 1) // group * group, group, rng.random() < 0.7, rng.random() < 0.3, out)
        del c["name"]
        return c
    if kind == "w4_mlp":
        return {"kind": kind, "M": min(M, 1024), "N": 128 * _log(rng, 8, 32), "K": 128 * _log(rng, 8, 32),
                "F": 128 * _log(rng, 8, 112), "zeros": rng.random() < 0.7}
    if kind == "w4_perm":
        return {"kind": kind, "M": min(M, 1024), "N": N, "K": K, "out": out}
    if kind == "w8":
        if rng.random() < 0.2:
            K -= rng.choice([16, 48, 60])   # widths that are no multiple of a slice
        return {"kind": kind, "M": min(M, 512), "N": min(N, 4096), "K": min(K, 8192), "bias": rng.random() < 0.5}
    if kind == "w8a8":
        if rng.random() < 0.2:
            K -= rng.choice([32, 64])
        return {"kind": kind, "fp8": rng.random() < 0.5, "M": M, "N": N, "K": K, "bias": rng.random() < 0.3}
    if kind == "mx":
        return {"kind": kind, "fmt": rng.choice(["mxfp8_e4m3", "mxfp8_e5m2", "mxfp6_e3m2", "mxfp6_e2m3", "mxfp4_e2m1"]),
                "M": M, "N": N, "K": K, "out": out}
    how = rng.choice(["w4_awq", "w4_gptq", "int8_rows", "fp8_tensor"])
    return {"kind": "quant", "how": how, "N": N, "K": K, "group": 128}


# ------------------------------------------------------------------ inputs
def _normal(g, shape, std=1.0):
    return torch.randn(shape, device=DEV, generator=g) * std


def _w4_weights(g, N, K, group, zeros):
    """Group-quantized N(0, 0.02) weights in plain torch: codes [N][K], the
    fp16 scales [N][G] and the zero points [N][G] (8 where there are none)."""
    w = _normal(g, (N, K // group, group), 0.02)
    if zeros:
        lo, hi = w.amin(-1), w.amax(-1)
        s = ((hi - lo) / 15).to(torch.float16)
        z = (-lo / s.float()).round().clamp(0, 15)
        q = (w / s.float()[..., None] + z[..., None]).round().clamp(0, 15)
    else:
        s = (w.abs().amax(-1) / 7).to(torch.float16)
        z = torch.full_like(s, 8, dtype=F32)
        q = ((w / s.float()[..., None]).round() + 8).clamp(1, 15)
    return q.to(torch.int32).reshape(N, K), s, z.to(torch.int32)


def _nibbles(q):
    """int32 words of 8 nibbles each, element 8 w + t at bits 4 t (rows padded)."""
    N, K = q.shape
    if K % 8:
        q = torch.nn.functional.pad(q, (0, 8 - K % 8))
    q = q.reshape(N, -1, 8)
    w = torch.zeros(q.shape[:2], dtype=torch.int32, device=q.device)
    for t in range(8):
        w |= q[..., t] << (4 * t)
    return w.contiguous()


def _w4_device(q, s, z, zeros):
    return _nibbles(q), s.view(torch.int16).contiguous(), _nibbles(z) if zeros else None


def _w4_value(q, s, z, group):
    N, K = q.shape
    d = (q.double().reshape(N, -1, group) - z.double()[..., None]) * s.double()[..., None]
    return d.reshape(N, K)


def _int8_rows(w):
    """Symmetric int8 per row in fp32: scale max/127, ties away from zero."""
    s = (w.abs().amax(-1).double() / 127).float()
    v = w * (1.0 / s.double()).float()[:, None]
    r = v.trunc()
    r = r + torch.where((v - r).abs() >= 0.5, v.sign(), torch.zeros_like(v))
    return r.clamp(-128, 127), s


def _e4m3_scaled(x):
    """x / s with s = max|x| / 240, the significand cut to 3 bits: (values, s)."""
    s = (x.abs().amax().double() / 240).float()
    v = (x.double() / s.double()).float()
    c = (v.view(torch.int32) & ~0xFFFFF).view(F32)
    return torch.where(v.abs() < 2.0 ** -6, torch.zeros_like(c), c), s


def _e4m3_codes(v):
    """Bytes of e4m3 values (normal numbers and zeros)."""
    b = v.view(torch.int32)
    mag = ((((b >> 23) & 0xFF) - 120) << 3) | ((b >> 20) & 7)
    mag = torch.where(v == 0, torch.zeros_like(mag), mag)
    return (mag | torch.where(v < 0, 0x80, 0)).to(torch.uint8)


_MX = {"mxfp8_e4m3": (4, 3, 7), "mxfp8_e5m2": (5, 2, 15), "mxfp6_e3m2": (3, 2, 3), "mxfp6_e2m3": (2, 3, 1),
       "mxfp4_e2m1": (2, 1, 1)}      # exponent bits, mantissa bits, bias
_MX_BITS = {"mxfp8_e4m3": 8, "mxfp8_e5m2": 8, "mxfp6_e3m2": 6, "mxfp6_e2m3": 6, "mxfp4_e2m1": 4}


def _mx_value(x, fmt):
    """x after a round trip through an MX format with blocks of 32, in 64 bits:
    a power-of-two scale that brings the block's peak under the largest
    element, significands rounded half to even and clipped."""
    eb, mb, bias = _MX[fmt]
    emax = (1 << eb) - 1 - bias
    top = 2.0 - 2.0 ** -mb               # largest significand
    b = x.double().reshape(x.shape[0], -1, 32)
    m, e = torch.frexp(b.abs().amax(-1))   # peak = m 2^e, m in [0.5, 1)
    sc = (e - 1) - emax + (2 * m > top).to(e.dtype)
    v = torch.ldexp(b, -sc[..., None])
    m, e = torch.frexp(v.abs())
    e = e - 1
    sub = e <= -bias                     # below the smallest normal: one fixed step
    sig = torch.where(sub, torch.ldexp(v.abs(), torch.full_like(e, mb + bias - 1)), (2 * m - 1) * 2 ** mb).round()
    sig = sig.clamp(max=2 ** mb - 1)
    r = torch.where(sub, torch.ldexp(sig, torch.full_like(e, 1 - bias - mb)),
                    torch.ldexp(1 + sig / 2 ** mb, e))
    r = torch.where(e > emax, torch.full_like(r, top * 2.0 ** emax), r)
    return (torch.ldexp(r, sc[..., None]) * v.sign()).reshape(x.shape)


def _out(c, M, N):
    return torch.empty((M, N), dtype=F32 if c.get("out") == "f32" else BF16, device=DEV)


def _inputs(c, seed):
    """The values of a case, the same for prepare() and exact()."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    kind, N, K = c["kind"], c["N"], c["K"]
    i = {}
    if kind == "quant":
        i["w"] = _normal(g, (N, K), 0.02)
        return i
    x = _normal(g, (c["M"], K))
    i["x"] = x if kind in ("w8", "mx") else x.to(BF16)
    i["bias"] = _normal(g, (N,)) if c.get("bias") else None
    if kind == "w4":
        i["w"] = _w4_weights(g, N, K, c["group"], c["zeros"])
    elif kind == "w4_mlp":
        i["gu"] = _w4_weights(g, 2 * c["F"], K, 128, c["zeros"])
        i["dn"] = _w4_weights(g, N, c["F"], 128, c["zeros"])
    elif kind == "w4_perm":
        i["w"] = _w4_weights(g, N, K, 128, False)      # columns in group order
        i["perm"] = torch.randperm(K, device=DEV, generator=g)
    elif kind == "w8":
        i["w"] = _normal(g, (K, N), 0.02)
    else:
        i["w"] = _normal(g, (N, K), 0.02)
    return i


def prepare(case, seed):
    lib = sneppx_quant.load()
    c, i = case, _inputs(case, seed)
    kind, N, K = c["kind"], c["N"], c["K"]
    st = {"lib": lib, "case": c, "x": i.get("x"), "bias": i.get("bias")}
    if kind == "quant":
        st["w"] = i["w"]
        how, G = c["how"], K // c["group"]
        if how == "int8_rows":
            st["q"] = torch.empty((N, K), dtype=torch.int8, device=DEV)
            st["s"] = torch.empty(N, device=DEV)
        elif how == "fp8_tensor":
            st["q"] = torch.empty((N, K), dtype=torch.uint8, device=DEV)
            st["s"] = torch.empty(1, device=DEV)
        else:
            st["q"] = torch.empty((N, K // 8), dtype=torch.int32, device=DEV)
            st["s"] = torch.empty((N, G), dtype=torch.int16, device=DEV)
            st["z"] = torch.empty((N, (G + 7) // 8), dtype=torch.int32, device=DEV)
        if how == "w4_gptq":
            g = torch.Generator(device=DEV).manual_seed(seed + 1)
            order = torch.randperm(K, device=DEV, generator=g)
            st["g_idx"] = (order // c["group"]).to(torch.int32)
        return st
    M = c["M"]
    if kind == "w4":
        st["w"] = _w4_device(*i["w"], c["zeros"])
        st["y"] = _out(c, M, N)
    elif kind == "w4_mlp":
        st["gu"], st["dn"] = _w4_device(*i["gu"], c["zeros"]), _w4_device(*i["dn"], c["zeros"])
        st["y"] = _out(c, M, N)
    elif kind == "w4_perm":
        q, s, z = i["w"]
        order = i["perm"]                              # sorted position -> column
        cols = torch.empty_like(q)
        cols[:, order] = q
        g_idx = torch.empty(K, dtype=torch.int32, device=DEV)
        g_idx[order] = (torch.arange(K, device=DEV) // 128).to(torch.int32)
        st["s"] = s.view(torch.int16).contiguous()
        st["q"] = torch.empty((N, K // 8), dtype=torch.int32, device=DEV)
        st["perm"] = torch.empty(K, dtype=torch.int16, device=DEV)
        lib.qlinear_w4_actorder_prepare(_nibbles(cols), g_idx, K // 128, st["q"], st["perm"])
        st["y"] = _out(c, M, N)
    elif kind == "w8":
        st["layer"] = lib.qlayer_create_kn(i["w"], "w8")
        if st["bias"] is not None:
            st["layer"].set_bias(st["bias"])
        st["y"] = torch.empty((M, N), device=DEV)
    elif kind == "w8a8":
        if c["fp8"]:
            v, s = _e4m3_scaled(i["w"])
            st["w"], st["s"] = _e4m3_codes(v), s.reshape(1)
        else:
            q, s = _int8_rows(i["w"])
            st["w"], st["s"] = q.to(torch.int8), s
        st["y"] = _out(c, M, N)
    else:
        packed, scales = lib.dev_quantize_mx(i["w"], c["fmt"])
        if c["fmt"].startswith("mxfp8"):
            packed, scales, _ = lib.mx_to_mfma(packed, scales, N, K, c["fmt"])
        st["w"], st["s"] = packed, scales
        st["y"] = _out(c, M, N)
    return st


def run(st):
    lib, c = st["lib"], st["case"]
    kind, K = c["kind"], c["K"]
    if kind == "quant":
        how, w, q, s = c["how"], st["w"], st["q"], st["s"]
        if how == "int8_rows":
            lib.dev_quantize_int8_channel(w, q, s)
            return [q, s]
        if how == "fp8_tensor":
            lib.dev_quantize_fp8_e4m3_scaled(w, q, s)
            return [q, s]
        if how == "w4_gptq":
            lib.dev_quantize_w4_gptq(w, st["g_idx"], K // c["group"], q, s)
            return [q, s]
        lib.dev_quantize_w4_awq(w, q, s, st["z"], c["group"])
        return [q, s, st["z"]]
    x, y = st["x"], st["y"]
    if kind == "w4":
        q, s, z = st["w"]
        lib.qlinear_w4a16(x, q, s, z, None, 0, y, c["group"], bias=st["bias"])
    elif kind == "w4_mlp":
        lib.qlinear_w4a16_mlp(x, st["gu"], st["dn"], y, 128)
    elif kind == "w4_perm":
        lib.qlinear_w4a16_actorder(x, st["q"], st["s"], None, st["perm"], y, 128)
    elif kind == "w8":
        st["layer"].forward_f32(x, y)
    elif kind == "w8a8":
        lib.qlinear_w8a8_dyn(x, st["w"], st["s"], y, fp8=c["fp8"], bias=st["bias"])
    else:
        fmt = c["fmt"]
        a, sa = lib.dev_quantize_mx(x, fmt)
        if fmt.startswith("mxfp8"):
            a, sa, _ = lib.mx_to_mfma(a, sa, c["M"], K, fmt)
        lib.qlinear_mx_gemm(a, sa, st["w"], st["s"], fmt, y, c["M"], c["N"], K, mfma_form=True)
    return y


def _w4_bytes(N, K, group, zeros):
    G = K // group
    return N * (K // 2 + 2 * G + (4 * ((G + 7) // 8) if zeros else 0))


def work(case):
    c = case
    kind, N, K = c["kind"], c["N"], c["K"]
    if kind == "quant":
        made = {"int8_rows": N * K + 4 * N, "fp8_tensor": N * K + 4,
                "w4_awq": _w4_bytes(N, K, c["group"], True), "w4_gptq": _w4_bytes(N, K, c["group"], False) + 4 * K}
        # a magnitude scan, a scaled rounding: about four operations an element
        return {"bytes": 4 * N * K + made[c["how"]], "flops": 4 * N * K}
    M = c["M"]
    y = M * N * (4 if kind == "w8" or c.get("out") == "f32" else 2)
    bias = 4 * N if c.get("bias") else 0
    flops = 2 * M * N * K
    if kind == "w4":
        b = 2 * M * K + _w4_bytes(N, K, c["group"], c["zeros"])
    elif kind == "w4_mlp":
        F = c["F"]
        b = 2 * M * K + _w4_bytes(2 * F, K, 128, c["zeros"]) + _w4_bytes(N, F, 128, c["zeros"])
        flops = 2 * M * (2 * F * K + F * N)
    elif kind == "w4_perm":
        b = 2 * M * K + _w4_bytes(N, K, 128, False) + 2 * K
    elif kind == "w8":
        b = 4 * M * K + N * K + 4 * N
    elif kind == "w8a8":
        b = 2 * M * K + N * K + 4 * (1 if c["fp8"] else N)
    else:
        b = 4 * M * K + N * K * _MX_BITS[c["fmt"]] // 8 + N * (K // 32)
    return {"bytes": b + y + bias, "flops": flops}


def tolerance(case):
    c = case
    if c["kind"] == "quant":
        return "exact"
    if c["kind"] == "w8":
        return {"rel": 2e-6, "max": 2e-5}          # fp32 in, fp32 sums
    if c.get("out") == "f32":
        # fp32 sums of exact bf16 x uint4 products; of fp8 / fp6 / fp4 products
        return {"rel": 4e-6, "max": 4e-5} if c["kind"] != "mx" else {"rel": 1e-5, "max": 1e-4}
    if c["kind"] == "w4_mlp":
        return {"rel": 1e-2, "max": 4e-2}          # two bf16 roundings, the first summed over F
    return {"rel": 7e-3, "max": 1.6e-2}            # one bf16 rounding of an fp32 sum


def exact(case, seed):
    c = case
    if c["kind"] == "quant":
        return None                                # codes and scales are bit patterns
    i = _inputs(c, seed)
    kind = c["kind"]
    x = i["x"].double()
    if kind == "w4_mlp":
        F = c["F"]
        gu = x @ _w4_value(*i["gu"], 128).t()
        act = torch.nn.functional.silu(gu[:, :F]) * gu[:, F:]
        return act @ _w4_value(*i["dn"], 128).t()
    if kind == "w4":
        y = x @ _w4_value(*i["w"], c["group"]).t()
    elif kind == "w4_perm":
        y = x[:, i["perm"]] @ _w4_value(*i["w"], 128).t()
    elif kind == "w8":
        q, s = _int8_rows(i["w"].t().contiguous())
        y = (x @ q.double().t()) * s.double()
    elif kind == "w8a8" and c["fp8"]:
        a, sa = _e4m3_scaled(i["x"].float())
        v, s = _e4m3_scaled(i["w"])
        y = (a.double() @ v.double().t()) * (sa.double() * s.double())
    elif kind == "w8a8":
        a, sa = _int8_rows(i["x"].float())
        q, s = _int8_rows(i["w"])
        y = (a.double() @ q.double().t()) * sa.double()[:, None] * s.double()
    else:
        y = _mx_value(i["x"], c["fmt"]) @ _mx_value(i["w"], c["fmt"]).t()
    return y if i["bias"] is None else y + i["bias"].double()
