"""Performance cases: the work a program gives this framework, through woolly_amd.ops.

Each case is one call (or one whole decode step) of the device-level entry
points on a Llama-shaped layer: the sizes are those of the benchmark
(hidden 4096, 14336 feed-forward rows, 32 / 8 heads of 128, context 4096), of the tests'
smaller layers (hidden 2048, 5632 feed-forward rows) and what lies between.
The GGUF block bytes are generated on the GPU from the seed.

  op        one pass
  matvec    quantized_matvec, one token
  qkv       attention_qkv: RMSNorm and the stacked q / k / v projection, one token
  matmul    quantized_matmul(_x), several tokens, f32 or bf16 activations
  ffn       ffn_swiglu: RMSNorm, gate, up, SwiGLU, down
  attn      attention_decode over an f16 KV cache
  step      LlamaModel.forward_token: token id to logits, every layer
  dequant   dequantize of a whole matrix
"""
import math

import numpy as np
import torch

from woolly_amd import device, ops

F32, BF16 = 0, 30
Q4_0, Q4_1, Q8_0, Q4_K, Q6_K = 2, 3, 8, 12, 14
TYPE_SIZE = {Q4_0: 18, Q4_1: 20, Q8_0: 34, Q4_K: 144, Q6_K: 210}
BLOCK = {Q4_0: 32, Q4_1: 32, Q8_0: 32, Q4_K: 256, Q6_K: 256}
EPS = 1e-5
ROPE_BASE = 500000.0


def listed():
    return [
        # one token through the first projection of a layer: the smallest call
        dict(name="qkv_q4_0_m1", op="qkv", type=Q4_0, hidden=4096, q_rows=4096, kv_rows=1024),
        # one decode projection, the headline of the benchmark
        dict(name="matvec_q4_0_14336x4096", op="matvec", type=Q4_0, n=14336, k=4096),
        # the feed-forward layer of a decode step
        dict(name="ffn_q4_0_m1", op="ffn", type=Q4_0, hidden=4096, n_ff=14336, m=1, prepared=False),
        # attention of a decode step at a long context
        dict(name="attn_ctx4096", op="attn", heads=32, kv_heads=8, head_dim=128, pos=4095),
        # a whole decode step of a file with per-tensor types (v, down and head Q6_K, the rest Q4_K)
        dict(name="step_q4_k_m_32_layers", op="step", type=Q4_K, type_v=Q6_K, type_down=Q6_K, type_head=Q6_K,
             layers=32, hidden=4096, heads=32, kv_heads=8, head_dim=128, n_ff=14336, vocab=128256, pos=4095),
        # a projection for eight sequences decoded together
        dict(name="matmul_q4_k_m8", op="matmul", type=Q4_K, n=14336, k=4096, m=8, x=F32, prepared=True),
        # the feed-forward layer for a short prompt, or many sequences decoded together
        dict(name="ffn_q4_k_m32", op="ffn", type=Q4_K, hidden=4096, n_ff=14336, m=32, prepared=True),
        # prefill: the feed-forward layer for 512 prompt tokens (the benchmark's second figure)
        dict(name="ffn_q4_0_m512", op="ffn", type=Q4_0, hidden=4096, n_ff=14336, m=512, prepared=False),
        # prefill on Q4_K_M files: gate / up are Q4_K, down is Q6_K; handles prepared once
        dict(name="matmul_q4_k_m512", op="matmul", type=Q4_K, n=14336, k=4096, m=512, x=F32, prepared=True),
        dict(name="matmul_q6_k_m512", op="matmul", type=Q6_K, n=4096, k=14336, m=512, x=F32, prepared=True),
        # a prompt of odd length in bf16 on a small layer
        dict(name="matmul_q8_0_bf16_m777", op="matmul", type=Q8_0, n=5632, k=2048, m=777, x=BF16, prepared=False),
        # a whole matrix to f32
        dict(name="dequant_q4_k_14336x4096", op="dequant", type=Q4_K, n=14336, k=4096),
    ]


# ------------------------------------------------------------------ drawing
def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def _k(rng, t, lo, hi):
    """A reduction length: whole blocks, and whole heads of 64 for the 32-element types."""
    step = 256 if BLOCK[t] == 256 else 64
    return max(step, _log(rng, lo, hi) // step * step)


def draw(rng):
    t = rng.choice([Q4_0, Q4_0, Q4_1, Q8_0, Q4_K, Q4_K, Q6_K])
    op = rng.choice(["matvec", "matvec", "qkv", "ffn", "ffn", "ffn", "matmul", "matmul", "matmul", "matmul", "attn",
                     "step", "dequant"])
    prepared = BLOCK[t] == 256 and rng.random() < 0.7
    if op == "matvec":
        return dict(op=op, type=t, n=_log(rng, 2048, 32000), k=_k(rng, t, 2048, 14336))
    if op == "qkv":
        d, kv = rng.choice([64, 128]), rng.choice([4, 8])
        heads = kv * rng.randint(1, 8)
        return dict(op=op, type=t, hidden=_k(rng, t, 2048, 8192), q_rows=heads * d, kv_rows=kv * d)
    if op == "ffn":
        h, m = _k(rng, t, 1024, 5120), _log(rng, 1, 1024)
        f = _k(rng, t, 2 * h, min(4 * h, 14336))
        while 6 * h * f * m > 2.0e11:
            m = m // 2 + 1
        return dict(op=op, type=t, hidden=h, n_ff=f, m=m, prepared=prepared)
    if op == "matmul":
        n, k, m = _log(rng, 512, 14336), _k(rng, t, 1024, 14336), _log(rng, 2, 2048)
        while 2 * n * k * m > 2.0e11:
            m = m // 2 + 1
        return dict(op=op, type=t, n=n, k=k, m=m, x=rng.choice([F32, F32, BF16]), prepared=prepared)
    if op == "attn":
        kv = rng.choice([2, 4, 8, 8, 16])
        return dict(op=op, heads=kv * rng.randint(1, 8), kv_heads=kv, head_dim=rng.choice([64, 128, 128]),
                    pos=_log(rng, 16, 16383))
    if op == "step":
        kv, g = rng.choice([4, 8]), rng.choice([2, 4])
        h = kv * g * 128
        f = _k(rng, Q4_K, 2 * h, 4 * h)
        down = rng.choice([t, Q6_K]) if BLOCK[t] == 256 else t
        return dict(op=op, type=t, type_v=down, type_down=down, type_head=rng.choice([Q8_0, Q6_K]),
                    layers=rng.randint(1, 6), hidden=h, heads=kv * g, kv_heads=kv, head_dim=128, n_ff=f,
                    vocab=_log(rng, 8000, 64000), pos=_log(rng, 16, 4095))
    return dict(op=op, type=t, n=_log(rng, 512, 14336), k=_k(rng, t, 1024, 14336))


# ------------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _f16(v):
    return v.to(torch.float16).view(torch.uint8).reshape(-1, 2)


def _bell(g, shape, keep):
    """Random bytes, each masked field the mean of two uniform ones: quants gather around their middle."""
    a = torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=g)
    b = torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=g)
    return ((a >> 1) & keep) + ((b >> 1) & keep) + (a & b & ~(keep << 1) & 0x11)


def _blocks(t, rows, k, g):
    """A rows x k matrix in GGUF blocks (weights of about 0.02), as a flat uint8 tensor."""
    nb = rows * (k // BLOCK[t])
    out = torch.empty((nb, TYPE_SIZE[t]), dtype=torch.uint8, device="cuda")
    scale = torch.exp(0.3 * torch.randn(nb, device="cuda", generator=g))
    if t == Q4_0:
        sign = torch.randint(0, 2, (nb,), device="cuda", generator=g) * 2 - 1
        out[:, 0:2] = _f16(0.006 * scale * sign)
        out[:, 2:] = _bell(g, (nb, 16), 0x77)
    elif t == Q4_1:
        out[:, 0:2] = _f16(0.006 * scale)
        out[:, 2:4] = _f16(-7.5 * 0.006 * scale * (1 + 0.1 * torch.randn(nb, device="cuda", generator=g)))
        out[:, 4:] = _bell(g, (nb, 16), 0x77)
    elif t == Q8_0:
        out[:, 0:2] = _f16(0.0004 * scale)
        out[:, 2:] = _bell(g, (nb, 32), 0x7F) ^ 0x80
    elif t == Q4_K:
        out[:, 0:12] = torch.randint(0, 256, (nb, 12), dtype=torch.uint8, device="cuda", generator=g)
        out[:, 12:14] = _f16(0.00016 * scale)
        out[:, 14:16] = _f16(-0.00016 * 31.5 * 7.5 * scale * (1 + 0.1 * torch.randn(nb, device="cuda", generator=g)))
        out[:, 16:] = _bell(g, (nb, 128), 0x77)
    else:
        out[:, 0:128] = _bell(g, (nb, 128), 0x77)
        out[:, 128:192] = torch.randint(0, 256, (nb, 64), dtype=torch.uint8, device="cuda", generator=g)
        out[:, 192:208] = torch.randint(64, 256, (nb, 16), dtype=torch.uint8, device="cuda", generator=g)
        out[:, 208:210] = _f16(0.0005 * scale)
    return out.reshape(-1)


def _acts(g, m, k):
    """Activations: normal, with a few channels that are larger than the rest."""
    x = torch.randn((m, k), device="cuda", generator=g)
    big = torch.rand(k, device="cuda", generator=g) < 0.005
    return torch.where(big, 12.0 * x, x)


def _gamma(g, k):
    return 1.0 + 0.1 * torch.randn(k, device="cuda", generator=g)


def _inv_freq(d):
    return torch.tensor([ROPE_BASE ** (-2.0 * i / d) for i in range(d // 2)], dtype=torch.float64).float().cuda()


def _layer_shapes(c):
    h, d = c["hidden"], c["head_dim"]
    q, kv, f, t = c["heads"] * d, c["kv_heads"] * d, c["n_ff"], c["type"]
    return dict(wq=(t, q, h), wk=(t, kv, h), wv=(c["type_v"], kv, h), wo=(t, h, q), w_gate=(t, f, h), w_up=(t, f, h),
                w_down=(c["type_down"], h, f))


def _inputs(case, seed):
    """The tensors of a case, from the seed alone."""
    g, op = _gen(seed), case["op"]
    if op == "matvec":
        return dict(w=_blocks(case["type"], case["n"], case["k"], g), x=_acts(g, 1, case["k"]))
    if op == "qkv":
        t, h = case["type"], case["hidden"]
        return dict(wq=_blocks(t, case["q_rows"], h, g), wk=_blocks(t, case["kv_rows"], h, g),
                    wv=_blocks(t, case["kv_rows"], h, g), gamma=_gamma(g, h), x=_acts(g, 1, h))
    if op == "ffn":
        t, h, f = case["type"], case["hidden"], case["n_ff"]
        return dict(gate=_blocks(t, f, h, g), up=_blocks(t, f, h, g), down=_blocks(t, h, f, g), gamma=_gamma(g, h),
                    x=_acts(g, case["m"], h))
    if op == "matmul":
        x = _acts(g, case["m"], case["k"])
        return dict(w=_blocks(case["type"], case["n"], case["k"], g), x=x.bfloat16() if case["x"] == BF16 else x)
    if op == "attn":
        h, kv, d, ctx = case["heads"], case["kv_heads"], case["head_dim"], case["pos"] + 1
        return dict(qkv=torch.randn((h + 2 * kv) * d, device="cuda", generator=g),
                    k=torch.randn((ctx, kv, d), device="cuda", generator=g).half(),
                    v=torch.randn((ctx, kv, d), device="cuda", generator=g).half(), inv=_inv_freq(d))
    if op == "step":
        h, kv, d, ctx = case["hidden"], case["kv_heads"], case["head_dim"], case["pos"] + 1
        layers = []
        for _ in range(case["layers"]):
            layer = {n: _blocks(*s, g) for n, s in _layer_shapes(case).items()}
            layer["attn_norm"], layer["ffn_norm"] = _gamma(g, h), _gamma(g, h)
            layers.append(layer)
        return dict(layers=layers, caches=torch.randn((case["layers"], 2, ctx, kv, d), device="cuda", generator=g).half(),
                    embd=_blocks(Q4_0, case["vocab"], h, g), norm=_gamma(g, h),
                    head=_blocks(case["type_head"], case["vocab"], h, g), inv=_inv_freq(d),
                    token=torch.randint(0, case["vocab"], (1,), device="cuda", generator=g).int())
    return dict(w=_blocks(case["type"], case["n"], case["k"], g))


def _weight(t, rows, k, w, prepared):
    """A weight handle as a loader makes it (its blocks converted once for prefill), or the device bytes as they are."""
    if not prepared:
        return w
    handle = ops.Weight(t, rows, k, w.cpu().numpy())
    handle.prepare_prefill()
    return handle


def _ptr(w):
    return w.data_ptr() if isinstance(w, torch.Tensor) else w.ptr


def _empty(*shape):
    return torch.empty(shape, dtype=torch.float32, device="cuda")


def _space(nbytes):
    return torch.empty(max(int(nbytes), 256), dtype=torch.uint8, device="cuda")


def prepare(case, seed):
    torch.cuda.init()
    device.init(torch.cuda.current_device())
    s = dict(case=case, **_inputs(case, seed))
    op = case["op"]
    if op == "matvec":
        s["out"] = _empty(case["n"])
    elif op == "qkv":
        s["out"] = _empty(case["q_rows"] + 2 * case["kv_rows"])
        s["ws"] = _space(ops.attention_qkv_workspace_bytes(case["hidden"]))
    elif op == "ffn":
        t, h, f, m = case["type"], case["hidden"], case["n_ff"], case["m"]
        for name, rows, k in (("gate", f, h), ("up", f, h), ("down", h, f)):
            s[name] = _weight(t, rows, k, s[name], case["prepared"])
        s["out"], s["ws"] = _empty(m, h), _space(ops.ffn_workspace_bytes(h, f, m, t))
    elif op == "matmul":
        t, n, k, m = case["type"], case["n"], case["k"], case["m"]
        s["nbytes"] = s["w"].numel()
        s["w"] = _weight(t, n, k, s["w"], case["prepared"])
        s["out"], s["ws"] = _empty(m, n), _space(ops.matmul_x_workspace_bytes(t, n, k, m, case["x"]))
    elif op == "attn":
        s["out"] = _empty(case["heads"] * case["head_dim"])
        s["ws"] = _space(ops.attention_workspace_bytes(case["heads"], case["kv_heads"], case["head_dim"], case["pos"] + 1))
    elif op == "step":
        dims = dict(hidden=case["hidden"], n_heads=case["heads"], n_kv_heads=case["kv_heads"], head_dim=case["head_dim"],
                    n_ff=case["n_ff"], max_ctx=case["pos"] + 1, vocab=case["vocab"], eps=EPS)
        types = {n + "_type": sh[0] for n, sh in _layer_shapes(case).items()}
        layers = []
        for i, layer in enumerate(s["layers"]):
            ptrs = {n: v.data_ptr() for n, v in layer.items()}
            layers.append(dict(ptrs, **types, k_cache=s["caches"][i, 0].data_ptr(), v_cache=s["caches"][i, 1].data_ptr()))
        s["model"] = ops.LlamaModel(case["type"], dims, layers, s["inv"].data_ptr(), s["norm"].data_ptr(),
                                    s["head"].data_ptr(), case["type_head"], s["embd"].data_ptr(), Q4_0)
        s["x"], s["logits"], s["ws"] = _empty(case["hidden"]), _empty(case["vocab"]), _space(s["model"].workspace_bytes())
    else:
        s["out"] = _empty(case["n"], case["k"])
    return s


def run(s):
    c = s["case"]
    op = c["op"]
    if op == "matvec":
        ops.quantized_matvec(c["type"], s["w"].data_ptr(), s["w"].numel(), s["x"].data_ptr(), s["out"].data_ptr(), c["n"], c["k"])
        return s["out"]
    if op == "qkv":
        ops.attention_qkv(c["type"], s["wq"].data_ptr(), s["wk"].data_ptr(), s["wv"].data_ptr(), c["q_rows"], c["kv_rows"],
                          c["hidden"], s["gamma"].data_ptr(), EPS, s["x"].data_ptr(), s["out"].data_ptr(),
                          s["ws"].data_ptr(), s["ws"].numel())
        return s["out"]
    if op == "ffn":
        ops.ffn_swiglu(c["type"], _ptr(s["gate"]), _ptr(s["up"]), _ptr(s["down"]), c["hidden"], c["n_ff"],
                       s["gamma"].data_ptr(), EPS, s["x"].data_ptr(), c["m"], s["out"].data_ptr(), s["ws"].data_ptr(),
                       s["ws"].numel())
        return s["out"]
    if op == "matmul":
        ops.quantized_matmul_x(c["type"], _ptr(s["w"]), s["nbytes"], c["n"], c["k"], s["x"].data_ptr(), c["x"], c["m"],
                               s["out"].data_ptr(), s["ws"].data_ptr(), s["ws"].numel())
        return s["out"]
    if op == "attn":
        ops.attention_decode(s["qkv"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), c["pos"], c["heads"], c["kv_heads"],
                             c["head_dim"], s["inv"].data_ptr(), s["out"].data_ptr(), s["ws"].data_ptr(), s["ws"].numel())
        return dict(out=s["out"], k=s["k"], v=s["v"])
    if op == "step":
        s["model"].forward_token(s["token"].data_ptr(), c["pos"], s["x"].data_ptr(), s["logits"].data_ptr(),
                                 s["ws"].data_ptr(), s["ws"].numel())
        return dict(logits=s["logits"], x=s["x"], caches=s["caches"])
    ops.dequantize(c["type"], s["w"].data_ptr(), s["w"].numel(), c["n"] * c["k"], s["out"].data_ptr())
    return s["out"]


# --------------------------------------------------------------- what it takes
def _wbytes(t, n, k):
    return n * (k // BLOCK[t]) * TYPE_SIZE[t]


def work(case):
    """Every input read once, every output written once; two operations per multiply-add."""
    c, op = case, case["op"]
    if op == "matvec":
        return dict(bytes=_wbytes(c["type"], c["n"], c["k"]) + 4 * (c["n"] + c["k"]), flops=2 * c["n"] * c["k"])
    if op == "qkv":
        n = c["q_rows"] + 2 * c["kv_rows"]
        return dict(bytes=_wbytes(c["type"], n, c["hidden"]) + 4 * (n + 2 * c["hidden"]), flops=2 * n * c["hidden"])
    if op == "ffn":
        h, f, m = c["hidden"], c["n_ff"], c["m"]
        return dict(bytes=2 * _wbytes(c["type"], f, h) + _wbytes(c["type"], h, f) + 4 * h * (2 * m + 1), flops=6 * m * h * f)
    if op == "matmul":
        n, k, m = c["n"], c["k"], c["m"]
        return dict(bytes=_wbytes(c["type"], n, k) + m * k * (2 if c["x"] == BF16 else 4) + 4 * m * n, flops=2 * m * n * k)
    if op == "attn":
        d, h, kv, p = c["head_dim"], c["heads"], c["kv_heads"], c["pos"] + 1
        return dict(bytes=4 * p * kv * d + 4 * (2 * h + 2 * kv) * d, flops=4 * p * h * d)
    if op == "step":
        d, h, kv, p = c["head_dim"], c["heads"], c["kv_heads"], c["pos"] + 1
        shapes = list(_layer_shapes(c).values())
        head = (c["type_head"], c["vocab"], c["hidden"])
        return dict(bytes=c["layers"] * (sum(_wbytes(*s) for s in shapes) + 4 * p * kv * d + 8 * c["hidden"]) + _wbytes(*head)
                    + 4 * c["vocab"],
                    flops=2 * (c["layers"] * (sum(s[1] * s[2] for s in shapes) + 2 * p * h * d) + c["vocab"] * c["hidden"]))
    return dict(bytes=_wbytes(c["type"], c["n"], c["k"]) + 4 * c["n"] * c["k"], flops=0)


def tolerance(case):
    """About four times what the sums in f32 show against exact()."""
    op = case["op"]
    if op == "dequant":
        return "exact"
    if op == "step":
        # every layer's rounding runs through those behind it, and the new k / v are rounded to f16
        return dict(rel=4e-5, max=1e-2)
    if op == "attn":
        return dict(rel=4e-6, max=1e-3)
    return dict(rel=2e-6, max=4e-5)


# --------------------------------------------------------------------- 64 bits
def _half(b):
    return b.contiguous().view(torch.float16).double()


def _dequant(t, w, rows, k):
    """The matrix in f64 (rows x k)."""
    b = w.view(-1, TYPE_SIZE[t])
    if t in (Q4_0, Q4_1):
        qs = b[:, 2 if t == Q4_0 else 4:]
        q = torch.cat([qs & 15, qs >> 4], 1).double()
        v = _half(b[:, 0:2]) * (q - 8) if t == Q4_0 else _half(b[:, 0:2]) * q + _half(b[:, 2:4])
    elif t == Q8_0:
        v = _half(b[:, 0:2]) * b[:, 2:].contiguous().view(torch.int8).double()
    elif t == Q4_K:
        i = torch.arange(8, device=b.device)
        src = 3 * i // 2
        raw = b[:, :12].int()
        odd = (raw[:, src] >> 6) | ((raw[:, (src + 1).clamp(max=11)] & 15) << 2)
        sc = torch.where(i % 2 == 0, raw[:, src] & 63, odd).double()
        qs = b[:, 16:]
        q = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).double()
        v = (_half(b[:, 12:14]) * sc)[:, :, None] * q + _half(b[:, 14:16])[:, :, None]
    else:
        i = torch.arange(256, device=b.device)
        ql, qh = b[:, :128][:, 16 * (i // 32) + i % 16].int(), b[:, 128:192].int()
        at, shift = 8 * (i // 32) + (i % 32) // 4, 2 * (i % 4)
        word = qh | (torch.nn.functional.pad(qh[:, 1:], (0, 1)) << 8)
        hi = word[:, at] >> torch.where(i < 128, shift, shift + 2)
        q = (torch.where(i < 128, ql & 15, ql >> 4) | ((hi & 3) << 4)) - 32
        v = _half(b[:, 208:210]) * b[:, 192:208][:, i // 16].double() * q.double() / 64.0
    return v.reshape(rows, k)


def _mm(t, w, rows, k, x):
    """x W^T in f64, some rows at a time."""
    out = torch.empty((x.shape[0], rows), dtype=torch.float64, device="cuda")
    step = max(1, (1 << 25) // k)
    per = w.numel() // rows
    for r in range(0, rows, step):
        n = min(step, rows - r)
        out[:, r:r + n] = x @ _dequant(t, w[r * per:(r + n) * per], n, k).t().contiguous()
    return out


def _rms(x, gamma):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + float(np.float32(EPS))) * gamma.double()


def _rope(v, inv, pos):
    """v [heads][d] rotated; the angle is formed in f32, as the reference does."""
    ang = (torch.tensor(float(pos), device="cuda") * inv).double()
    a, b = v.chunk(2, -1)
    return torch.cat([a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos()], -1)


def _attention(qkv, kc, vc, inv, heads, kv, d, pos):
    """The attention output and the caches with the new row, in f64."""
    q, k, v = qkv.view(-1, d).split([heads, kv, kv])
    kc, vc = kc.double(), vc.double()
    kc[pos], vc[pos] = _rope(k, inv, pos).float().half().double(), v.float().half().double()
    q = _rope(q, inv, pos).view(kv, heads // kv, d)
    out = torch.empty_like(q)
    for h in range(kv):
        p = torch.softmax(q[h] @ kc[:, h].t().contiguous() / math.sqrt(d), -1)
        out[h] = p @ vc[:, h].contiguous()
    return out.reshape(-1), kc, vc


def _ffn(s, t, h, f, gamma, x):
    xh = _rms(x, gamma)
    g, u = _mm(t["gate"], s["gate"], f, h, xh), _mm(t["up"], s["up"], f, h, xh)
    return _mm(t["down"], s["down"], h, f, g * torch.sigmoid(g) * u)


def exact(case, seed):
    s, c, op = _inputs(case, seed), case, case["op"]
    if op == "matvec":
        return _mm(c["type"], s["w"], c["n"], c["k"], s["x"].double())[0]
    if op == "qkv":
        xh = _rms(s["x"].double(), s["gamma"])
        rows = dict(wq=c["q_rows"], wk=c["kv_rows"], wv=c["kv_rows"])
        return torch.cat([_mm(c["type"], s[n], r, c["hidden"], xh)[0] for n, r in rows.items()])
    if op == "ffn":
        return _ffn(s, dict.fromkeys(("gate", "up", "down"), c["type"]), c["hidden"], c["n_ff"], s["gamma"], s["x"].double())
    if op == "matmul":
        return _mm(c["type"], s["w"], c["n"], c["k"], s["x"].double())
    if op == "attn":
        out, k, v = _attention(s["qkv"].double(), s["k"], s["v"], s["inv"], c["heads"], c["kv_heads"], c["head_dim"], c["pos"])
        return dict(out=out, k=k, v=v)
    if op == "step":
        h, f, shapes = c["hidden"], c["n_ff"], _layer_shapes(c)
        x = _dequant(Q4_0, s["embd"].view(c["vocab"], -1)[int(s["token"])].clone(), 1, h)
        caches = []
        for i, layer in enumerate(s["layers"]):
            xh = _rms(x, layer["attn_norm"])
            qkv = torch.cat([_mm(shapes[n][0], layer[n], shapes[n][1], h, xh)[0] for n in ("wq", "wk", "wv")])
            att, k, v = _attention(qkv, s["caches"][i, 0], s["caches"][i, 1], s["inv"], c["heads"], c["kv_heads"],
                                   c["head_dim"], c["pos"])
            caches.append(torch.stack([k, v]))
            x = x + _mm(shapes["wo"][0], layer["wo"], h, shapes["wo"][2], att[None])
            mats = dict(gate=layer["w_gate"], up=layer["w_up"], down=layer["w_down"])
            types = dict(gate=shapes["w_gate"][0], up=shapes["w_up"][0], down=shapes["w_down"][0])
            x = x + _ffn(mats, types, h, f, layer["ffn_norm"], x)
        logits = _mm(c["type_head"], s["head"], c["vocab"], h, _rms(x, s["norm"]))[0]
        return dict(logits=logits, x=x[0], caches=torch.stack(caches))
    return _dequant(c["type"], s["w"], c["n"], c["k"])
