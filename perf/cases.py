"""The work that a program on this inference path has it do, as measurable cases.

Kinds (``case["kind"]``), each called as the reference's modules or a serving
loop call it:
  ffn          one Paraplex FFN sublayer through ``loom_amd.ops``: W_real, the
               compact W_imag product over [Q | Kctx | C | U | D], the fused
               pointwise chain, W2
  depth        one DepthAttn read over S earlier-depth states
  tria_window  one fire window of a block's Tria state: gated depth step, the
               temporal carry's endpoint, PolARM, the readout of the new key
  tria_chunked the Tria path of a whole chunked forward (all layers, carry every
               W tokens) and the readout of its document keys
  final_ca     the sequence form of the final cross-attention over document keys
  gqa_decode   one layer's decode attention (RoPE, cache append, both readouts)
  gqa_prefill  one layer's causal attention of a prompt chunk over the cache
  decode       token-by-token steps of the model over a known prompt
  prefill      the chunked prefill of a prompt by the model

The model of the last two is the nano_chk configuration with four of its ten
(equal) layers in bf16, where the logits of two correct orders of rounding are
1% apart (at ten layers 3 to 5%), and the fp32 reference configuration whole.
Widths are those of the nano configurations (8 q heads of 96 over 2 kv heads,
H = 3072), the drawn ones also 8 heads of 64 or 128; batches run from one
sequence to 32, sequences from one token to 4096.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "loomformer-paraplex_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from loom_amd import _lib, ops  # noqa: E402
from loom_amd.config import NANO, NANO_CHK, ModelConfig  # noqa: E402
from loom_amd.engine import LoomDecoder  # noqa: E402
from loom_amd.weights import init_state_dict, rope_tables  # noqa: E402

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
SIZE = {"bf16": 2, "fp32": 4}
QH, KVH = 8, 2
ALPHA, POLARM, POWLU_M = 0.0375, 0.1, 3.0


def listed():
    return [
        # a decode step of 32 sequences through the modules: launches and latency
        dict(name="ffn_bf16_32x1", kind="ffn", dtype="bf16", B=32, T=1, HD=96),
        # the fp32 reference configuration: one 128-token prompt
        dict(name="ffn_fp32_1x128", kind="ffn", dtype="fp32", B=1, T=128, HD=96),
        # a few prompts of a ragged length
        dict(name="ffn_bf16_3x333", kind="ffn", dtype="bf16", B=3, T=333, HD=96),
        # the Paraplex microbenchmark: 8192 tokens
        dict(name="ffn_bf16_8x1024", kind="ffn", dtype="bf16", B=8, T=1024, HD=96),
        # the DepthAttn microbenchmark: 16384 tokens, 24 states
        dict(name="depth_bf16_16384x24", kind="depth", dtype="bf16", B=1, T=16384, S=24, HD=96),
        # one 128-token fire window of 32 sequences (serving prefill)
        dict(name="tria_window_bf16_32x128", kind="tria_window", dtype="bf16", B=32, T=128, H=3072, axis=1),
        # the Tria microbenchmark: 24 layers over 8 x 4096 tokens, carry every 64
        dict(name="tria_chunked_fp32_8x4096", kind="tria_chunked", dtype="fp32", L=24, B=8, T=4096, H=3072, W=64),
        # the final cross-attention of 8 sequences of 2048 tokens over their 15 earlier fires
        dict(name="final_ca_bf16_8x2048", kind="final_ca", dtype="bf16", B=8, T=2048, K=15, HD=96),
        # the decode workload's attention at the middle of its generation
        dict(name="gqa_decode_bf16_32x2176", kind="gqa_decode", dtype="bf16", B=32, len=2176, HD=96),
        # a prompt chunk half way through a 2048-token prompt, 8 sequences
        dict(name="gqa_prefill_bf16_8x128", kind="gqa_prefill", dtype="bf16", B=8, T=128, start=1024, HD=96),
        # token-by-token decoding, 32 sequences
        dict(name="decode_bf16_32x512", kind="decode", dtype="bf16", B=32, P=512),
        # the prompt of the decode workload
        dict(name="prefill_bf16_32x2048", kind="prefill", dtype="bf16", B=32, P=2048),
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["ffn", "ffn", "ffn", "depth", "tria_window", "tria_chunked", "final_ca", "gqa_decode",
                       "gqa_prefill", "decode", "prefill", "prefill"])
    dtype = "fp32" if rng.random() < 0.3 else "bf16"
    HD = rng.choice([96, 96, 64, 128])
    B = _log(rng, 1, 32)
    if kind == "ffn":
        rows = _log(rng, 1, 8192 if dtype == "bf16" else 2048)
        B = min(B, rows)
        return dict(kind=kind, dtype=dtype, B=B, T=max(1, rows // B), HD=HD)
    if kind == "depth":
        rows = _log(rng, 1, 16384)
        B = min(B, rows)
        return dict(kind=kind, dtype=dtype, B=B, T=max(1, rows // B), S=rng.randint(1, 24), HD=HD)
    if kind == "tria_window":
        return dict(kind=kind, dtype=dtype, B=B, T=rng.choice([128, 64, rng.randint(1, 128)]),
                    H=32 * HD, axis=rng.randint(0, 2))
    if kind == "tria_chunked":
        B = _log(rng, 1, 8)
        return dict(kind=kind, dtype=dtype, L=rng.choice([10, 24]), B=B, T=_log(rng, 130, 4096 // B), H=32 * HD,
                    W=rng.choice([64, 128]))
    if kind == "final_ca":
        T = _log(rng, 130, 2048)
        return dict(kind=kind, dtype=dtype, B=_log(rng, 1, 8), T=T, K=max(1, (T - 1) // 128), HD=HD)
    if kind == "gqa_decode":
        return dict(kind=kind, dtype=dtype, B=B, len=_log(rng, 1, 4096), HD=HD)
    if kind == "gqa_prefill":
        return dict(kind=kind, dtype=dtype, B=_log(rng, 1, 8), T=rng.choice([128, rng.randint(1, 128)]),
                    start=rng.randint(0, 1024), HD=HD)
    if kind == "decode":
        return dict(kind=kind, dtype=dtype, B=B, P=_log(rng, 16, 512 if dtype == "bf16" else 128))
    if dtype == "fp32":
        return dict(kind=kind, dtype=dtype, B=_log(rng, 1, 4), P=_log(rng, 64, 512))
    return dict(kind=kind, dtype=dtype, B=B, P=_log(rng, 64, 2048))


# ------------------------------------------------------------------ inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _kaiming(g, out_f, in_f):
    """nn.Linear's default weight draw."""
    return (torch.rand(out_f, in_f, generator=g, device=DEV) * 2 - 1) / math.sqrt(in_f)


def _unit_carry(g, *shape):
    """Carried 3x3 records as they are stored: products of rotations times (I + K) with a small K, at unit RMS."""
    w, x, y, z = torch.nn.functional.normalize(torch.randn(4, *shape, generator=g, device=DEV), dim=0)
    c = torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                     2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                     2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], -1).unflatten(-1, (3, 3))
    c = c.add_(torch.randn(*shape, 3, 3, generator=g, device=DEV), alpha=0.05)
    return c.div_(c.square().mean(dim=(-1, -2), keepdim=True).add_(1e-6).sqrt_())


def _readout_params(g, N, dt):
    key_w = torch.randn(32, 9, generator=g, device=DEV) * 1.5
    raw = key_w.t() @ torch.randn(32, generator=g, device=DEV)
    return dict(score_w=(raw / raw.norm()).to(dt), proj_w=_kaiming(g, 32, 9).to(dt),
                proj_b=torch.randn(32, generator=g, device=DEV) * 0.1, up_w=_kaiming(g, N, 32).to(dt),
                up_b=torch.randn(N, generator=g, device=DEV) * 0.1)


_WEIGHTS = {}


def _config(dtype):
    return ModelConfig.from_dict(dict(NANO_CHK, layers=4) if dtype == "bf16" else NANO).with_seq_len(4096)


def _model(dtype):
    """The model's weights, as a checkpoint holds them."""
    if dtype not in _WEIGHTS:
        cfg = _config(dtype)
        _WEIGHTS[dtype] = (cfg, init_state_dict(cfg, 2 if dtype == "bf16" else 0))
    return _WEIGHTS[dtype]


def prepare(case, seed):
    kind, dt, g = case["kind"], DTYPES[case["dtype"]], _gen(seed)
    rn = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dt)  # noqa: E731
    s = dict(kind=kind)
    if kind == "ffn":
        B, T, HD = case["B"], case["T"], case["HD"]
        N, H = QH * HD, 4 * QH * HD
        s.update(u=rn(B, T, N), q=rn(B, T, QH, HD), kctx=rn(B, T, QH, HD), c=rn(B, T, QH, HD), d=rn(B, T, QH, HD),
                 w_real=_kaiming(g, H, N).to(dt), b_real=torch.randn(H, generator=g, device=DEV) * 0.02,
                 w_imag=_kaiming(g, H, N + 4 * HD).to(dt), b_imag=torch.randn(H, generator=g, device=DEV) * 0.02,
                 trace=torch.tanh(torch.randn(B, H, generator=g, device=DEV)).to(dt),
                 trace_w=torch.rand(H, generator=g, device=DEV) - 0.5, anchor=torch.ones((), device=DEV),
                 reset=torch.empty(0, dtype=torch.bool, device=DEV), w2=_kaiming(g, N, H).to(dt),
                 b2=torch.randn(N, generator=g, device=DEV) * 0.02, Hq=H // QH, HD=HD)
    elif kind == "depth":
        B, T, S, HD = case["B"], case["T"], case["S"], case["HD"]
        s.update(k=rn(B, T, S, QH, HD), v=rn(B, T, S, QH, HD),
                 q=(torch.randn(QH, HD, generator=g, device=DEV) * 0.1).to(dt))
    elif kind == "tria_window":
        B, T, H = case["B"], case["T"], case["H"]
        reset = torch.zeros(B, T, dtype=torch.bool, device=DEV)
        s.update(r=rn(B, T, H), i=torch.tanh(rn(B, T, H)), o=rn(B, T, H), prev=_unit_carry(g, B, T, H).to(dt),
                 w=torch.softmax(torch.randn(9, generator=g, device=DEV), 0).to(dt), reset=reset,
                 state=_unit_carry(g, B, H).to(dt), valid=torch.ones(B, dtype=torch.bool, device=DEV),
                 axis=case["axis"], read=_readout_params(g, H // 4, dt))
    elif kind == "tria_chunked":
        L, B, T, H = case["L"], case["B"], case["T"], case["H"]
        r, i, o = (torch.empty(L, B, T, H, dtype=dt, device=DEV).normal_(generator=g) for _ in range(3))
        s.update(r=r, i=i, o=o, W=case["W"], read=_readout_params(g, H // 4, torch.float32))
    elif kind == "final_ca":
        B, T, K, N = case["B"], case["T"], case["K"], QH * case["HD"]
        fires = 128 * (torch.arange(K, device=DEV) + 1)
        allowed = (torch.arange(T, device=DEV)[:, None] >= fires[None, :])[None].expand(B, T, K).contiguous()
        s.update(q=rn(B, T, N), k=rn(B, K, N), v=rn(B, K, N), allowed=allowed, scale=N ** -0.5)
    elif kind in ("gqa_decode", "gqa_prefill"):
        B, HD = case["B"], case["HD"]
        T = case.get("T", 1)
        cap = case["len"] if kind == "gqa_decode" else case["start"] + T
        cos, sin = rope_tables(ModelConfig.from_dict(dict(NANO, model_dim=QH * HD, head_dim=HD)).with_seq_len(4096), cap)
        s.update(qkv=rn(B, T, (QH + 2 * KVH) * HD), kc=rn(B, KVH, cap, HD), vc=rn(B, KVH, cap, HD),
                 cos=cos.to(DEV), sin=sin.to(DEV), q=torch.empty(B, T, QH, HD, dtype=dt, device=DEV),
                 c=torch.empty(B, T, QH * HD, dtype=dt, device=DEV), kctx=torch.empty(B, T, QH * HD, dtype=dt, device=DEV),
                 code=_lib.DTYPE_CODE[dt], B=B, T=T, cap=cap, HD=HD)
        if kind == "gqa_decode":
            nb = _lib.load().loom_gqa_workspace_bytes(B, cap, QH, KVH, HD)
            s.update(ws=torch.empty(nb // 4 + 1, device=DEV), ws_bytes=nb)
    else:
        cfg, state = _model(case["dtype"])
        eng = LoomDecoder(cfg, state, batch=case["B"], dtype=dt, max_len=case["P"] + 1)
        prompt = torch.randint(0, cfg.V, (case["B"], case["P"]), generator=g, device=DEV)
        if kind == "decode":
            eng.start(prompt)
            eng.warm_graphs()
        s.update(eng=eng, prompt=prompt)
    return s


# ------------------------------------------------------------------ one pass

def run(s):
    kind = s["kind"]
    if kind == "ffn":
        R = ops.linear(s["u"], s["w_real"], s["b_real"])
        beta = ops.beta_forward_cuda(s["u"], s["q"], s["kctx"], s["c"], s["d"], s["w_imag"], s["Hq"], s["HD"], QH,
                                     False)[0]
        act, phase, trace, _ = ops.paraplex_forward(R, R, beta, s["b_imag"], s["trace"], s["trace_w"], s["reset"],
                                                    s["anchor"], 1, False, 0.99, POWLU_M)
        return dict(R=R, beta=beta, act=act, phase=phase, trace=trace, out=ops.linear(act, s["w2"], s["b2"]))
    if kind == "depth":
        d, lse = ops.depth_attn_stacked_forward(s["q"], s["k"], s["v"])
        return dict(d=d, lse=lse)
    if kind == "tria_window":
        carry, p, scale = ops.tria_step_gate_forward(s["r"], s["i"], s["o"], s["prev"], s["w"], ALPHA, s["axis"])
        end, end32 = ops.temporal_carry_endpoint_forward(carry, s["reset"], s["state"], s["valid"])
        key = ops.polarm(end, POLARM)
        return dict(carry=carry, p=p, scale=scale, end=end, end32=end32, key=key,
                    a=ops.tria_readout(key[:, None], **s["read"]))
    if kind == "tria_chunked":
        keys, _ = ops.tria_chunked_forward(s["r"], s["i"], s["o"], ALPHA, s["W"], POLARM)
        return dict(keys=keys, a=ops.tria_readout(keys, **s["read"]) if keys.shape[1] else keys)
    if kind == "final_ca":
        out, lse = ops.final_ca_sparse_forward(s["q"], s["k"], s["v"], s["allowed"], s["scale"])
        return dict(out=out, lse=lse)
    if kind in ("gqa_decode", "gqa_prefill"):
        P, B, T, cap, HD = _lib.ptr, s["B"], s["T"], s["cap"], s["HD"]
        if kind == "gqa_decode":
            _lib.call("loom_gqa_decode_step", s["code"], P(s["qkv"]), P(s["kc"]), P(s["vc"]), KVH * cap * HD, HD,
                      cap * HD, P(s["cos"]), P(s["sin"]), P(s["q"]), P(s["c"]), P(s["kctx"]), QH * HD, P(s["ws"]),
                      s["ws_bytes"], B, cap, None, QH, KVH, HD, _lib.stream_of(s["qkv"]))
        else:
            _lib.call("loom_gqa_prefill", s["code"], P(s["qkv"]), (QH + 2 * KVH) * HD, P(s["kc"]), P(s["vc"]),
                      KVH * cap * HD, HD, cap * HD, P(s["cos"]), P(s["sin"]), P(s["q"]), P(s["c"]), P(s["kctx"]),
                      QH * HD, B, T, cap - T, cap, QH, KVH, HD, _lib.stream_of(s["qkv"]))
        return dict(q=s["q"], c=s["c"], kctx=s["kctx"], kc=s["kc"], vc=s["vc"])
    eng = s["eng"]
    if kind == "decode":
        eng.start(s["prompt"])
        eng.replay_steps(s["prompt"].shape[1] - 1)
    else:
        eng.prefill(s["prompt"])
    return dict(logits=eng.logits, kc=eng.k_cache, vc=eng.v_cache, trace=eng.trace)


# ------------------------------------------------------------------ what a pass cannot do without

def work(case):
    kind, e = case["kind"], SIZE[case["dtype"]]
    if kind == "ffn":
        HD = case["HD"]
        M, N, H, B = case["B"] * case["T"], QH * HD, 4 * QH * HD, case["B"]
        K = N + 4 * HD
        return dict(bytes=e * (M * 5 * N + H * (2 * N + K) + M * (4 * H + N) + 2 * B * H) + 4 * (3 * H + N),
                    flops=2 * M * H * (2 * N + K))
    if kind == "depth":
        rows, S, HD = case["B"] * case["T"] * QH, case["S"], case["HD"]
        return dict(bytes=rows * (2 * S * HD * e + HD * e + 4), flops=rows * S * HD * 4)
    if kind == "tria_window":
        B, H = case["B"], case["H"]
        n, N = B * case["T"] * H, H // 4
        return dict(bytes=n * ((3 + 9 + 9 + 1) * e + 4) + B * H * (27 * e + 36) + B * N * e,
                    flops=n * 260 + B * N * 64)
    if kind == "tria_chunked":
        B, T, H = case["B"], case["T"], case["H"]
        n, K, N = case["L"] * B * T * H, -(-T // case["W"]) - 1, H // 4
        return dict(bytes=3 * n * e + B * K * (H * 36 + 4 * N), flops=n * 130 + B * T * H * 80)
    if kind == "final_ca":
        B, T, K, N = case["B"], case["T"], case["K"], QH * case["HD"]
        return dict(bytes=e * (2 * B * T * N + 2 * B * K * N) + B * T * (K + 4), flops=4 * B * T * K * N)
    if kind == "gqa_decode":
        B, n, HD = case["B"], case["len"], case["HD"]
        return dict(bytes=e * B * HD * (2 * KVH * n + (QH + 2 * KVH) + 3 * QH), flops=6 * B * QH * n * HD)
    if kind == "gqa_prefill":
        B, T, s0, HD = case["B"], case["T"], case["start"], case["HD"]
        pairs = T * s0 + T * (T + 1) // 2
        return dict(bytes=e * B * HD * (2 * KVH * (s0 + T) + T * (QH + 2 * KVH) + 3 * T * QH),
                    flops=6 * B * QH * pairs * HD)
    c, B, P = _config(case["dtype"]), case["B"], case["P"]
    block = c.N * (c.N + 2 * c.KV) + c.N * c.N + c.H * (2 * c.N + c.imag_in)      # qkv, o, W_real, W_imag, W2
    depth = 2 * (2 * c.N * c.N + c.N * c.N)                                       # kv and readout, twice a block
    pairs = B * c.QH * P * (P + 1) // 2
    weights = e * (c.L * block + 3 * c.N * c.N + 3 * c.N * c.N + c.V * c.N)       # shared depth, final CA, head
    cache = e * 2 * c.L * B * c.KV
    if case["kind"] == "decode":       # every step reads the weights and the cache so far
        return dict(bytes=P * weights + cache * (P * (P + 1) // 2 + P),
                    flops=2 * P * B * (c.L * (block + depth) + c.V * c.N) + 6 * c.L * pairs * c.HD)
    return dict(bytes=weights + 8 * B * P + cache * P + e * B * c.V,
                flops=2 * P * B * c.L * (block + depth) + 2 * B * c.V * c.N + 6 * c.L * pairs * c.HD)


def tolerance(case):
    # about four times what the path measures against exact() (single layers) or
    # against the same engine's other order of sums (whole model)
    kind, bf16 = case["kind"], case["dtype"] == "bf16"
    if kind in ("decode", "prefill"):
        return {"rel": 3e-2} if bf16 else {"rel": 1e-4}
    if kind in ("tria_window", "tria_chunked") and not bf16:     # products of up to 4096 carriers
        return {"rel": 5e-5}
    return {"rel": 1.5e-2, "max": 0.3} if bf16 else {"rel": 1e-5, "max": 1e-3}


# ------------------------------------------------------------------ the same in 64 bits

def _mm3(a, b):
    return (a.unsqueeze(-1) * b.unsqueeze(-3)).sum(-2)


def _rms9(m):
    return m.square().mean(dim=(-1, -2), keepdim=True).add(1e-6).sqrt()


def _norm9(m):
    return m / _rms9(m)


def _carrier(r, i, o, axis):
    """(I + K(a, b, c)) R_axis: K the cross-product matrix of alpha tanh of the RMS-normalised (ri, ro, io), R a
    quarter turn about z, x or y."""
    x = torch.stack([r * i, r * o, i * o], -1)
    a, b, c = (ALPHA * torch.tanh(x / (x.square().mean(-1, keepdim=True) + 1e-6).sqrt())).unbind(-1)
    n1 = torch.ones_like(a)
    ik = torch.stack([n1, -c, b, c, n1, -a, -b, a, n1], -1).unflatten(-1, (3, 3))
    turn = ([[0, -1, 0], [1, 0, 0], [0, 0, 1]], [[1, 0, 0], [0, 0, -1], [0, 1, 0]], [[0, 0, 1], [0, 1, 0], [-1, 0, 0]])[axis]
    return ik @ torch.tensor(turn, dtype=a.dtype, device=a.device)


def _polarm(m):
    gram = _mm3(m.transpose(-1, -2), m)
    eye = torch.eye(3, dtype=m.dtype, device=m.device)
    s = gram.diagonal(dim1=-2, dim2=-1).mean(-1).clamp_min(1e-6)[..., None, None]
    return _mm3(m, eye - 0.5 * POLARM * (gram / s - eye))


def _readout(carry, p):
    flat = carry.flatten(-2)
    w = torch.softmax(flat @ p["score_w"].double(), dim=-1)
    pooled = (w.unsqueeze(-1) * flat).sum(-2)
    return (pooled @ p["proj_w"].double().t() + p["proj_b"].double()) @ p["up_w"].double().t() + p["up_b"].double()


def _rotate(x, cos, sin):
    half = x.shape[-1] // 2
    return x * cos + torch.cat([-x[..., half:], x[..., :half]], -1) * sin


def _attend(q, k, v, mask):
    """q [B,T,QH,HD] over k, v [B,KVH,L,HD]: A.V and A.K, both [B,T,QH*HD]."""
    B, T, _, HD = q.shape
    qg = q.view(B, T, KVH, QH // KVH, HD).permute(0, 2, 3, 1, 4).reshape(B, KVH, -1, HD)
    sc = (qg @ k.transpose(-1, -2).contiguous()) / math.sqrt(HD)
    sc = sc.view(B, KVH, QH // KVH, T, -1).masked_fill(~mask, -math.inf)
    w = torch.softmax(sc, -1).reshape(B, KVH, -1, k.shape[2])
    back = lambda x: (w @ x).view(B, KVH, QH // KVH, T, HD).permute(0, 3, 1, 2, 4).reshape(B, T, QH * HD)  # noqa: E731
    return back(v), back(k)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        return None
    s = prepare(case, seed)
    f = {k: v if kind in ("depth", "tria_chunked") and v.numel() > 1 << 20 else v.double()
         for k, v in s.items() if torch.is_tensor(v) and v.is_floating_point()}
    if kind == "ffn":
        B, T, HD = case["B"], case["T"], case["HD"]
        R = f["u"] @ f["w_real"].t() + f["b_real"]
        w, beta = f["w_imag"].view(QH, s["Hq"], -1), []
        for g in range(QH):
            x = torch.cat([f["q"][:, :, g], f["kctx"][:, :, g], f["c"][:, :, g], f["u"], f["d"][:, :, g]], -1)
            beta.append(x @ w[g].t())
        beta = torch.cat(beta, -1)
        b = beta + f["b_imag"]
        base = torch.sin(0.5 * math.pi * b / (1 + b * b).sqrt())
        prev = torch.cat([f["trace"][:, None], base[:, :-1]], 1)
        raw = base + f["trace_w"] * prev
        phase = raw / (1 + raw * raw).sqrt()
        amp = torch.where(R > 20, R, torch.log1p(torch.exp(R.clamp_max(20))))
        safe = amp.clamp_min(1e-12)
        act = (R + amp * phase) * safe ** (POWLU_M / (safe.sqrt() + 1)) * torch.sigmoid(amp)
        return dict(R=R, beta=beta, act=act, phase=phase, trace=base[:, -1], out=act @ f["w2"].t() + f["b2"])
    if kind == "depth":
        d, lse = [], []
        for k, v in zip(s["k"].flatten(0, 1).split(4096), s["v"].flatten(0, 1).split(4096)):
            sc = (k.double() * f["q"]).sum(-1) / math.sqrt(case["HD"])
            d.append((torch.softmax(sc, 1).unsqueeze(-1) * v.double()).sum(1))
            lse.append(torch.logsumexp(sc, 1))
        sh = (case["B"], case["T"], QH)
        return dict(d=torch.cat(d).view(*sh, -1), lse=torch.cat(lse).view(sh))
    if kind == "tria_window":
        carry, p, scale = [], [], []
        w = f["w"].view(3, 3)
        for b in range(case["B"]):
            pre = _mm3(_carrier(f["r"][b], f["i"][b], f["o"][b], s["axis"]), f["prev"][b])
            rms = _rms9(pre)
            carry.append(pre / rms)
            p.append((carry[-1] * w).sum((-1, -2)))
            scale.append(rms.flatten())
        carry, end = torch.stack(carry), f["state"]
        for t in range(case["T"]):          # over the carries as the step stores them
            end = _norm9(_mm3(carry[:, t].to(DTYPES[case["dtype"]]).double(), end))
        key = _polarm(end)
        return dict(carry=carry, p=torch.stack(p), scale=torch.cat(scale), end=end, end32=end, key=key,
                    a=_readout(key[:, None], s["read"]))
    if kind == "tria_chunked":
        L, B, T, W = case["L"], case["B"], case["T"], case["W"]
        local = lambda layer, at: _carrier(*(s[x][(layer, *at)].double() for x in "rio"), layer % 3)  # noqa: E731
        depth, firsts, every = [], range(0, T, W), slice(None)
        for b in range(B):
            D = None
            for layer in range(L):
                m = local(layer, (b,))
                D = _norm9(m if D is None else _mm3(m, D))
            depth.append(D)
        depth, keys, state = torch.stack(depth), [], None
        for c, t0 in enumerate(firsts):
            acc = depth[:, t0]
            if state is not None:      # the chunk's first token starts from the fired state
                acc = state
                for layer in range(L):
                    acc = _norm9(_mm3(local(layer, (every, t0)), acc))
            for t in range(t0 + 1, min(t0 + W, T)):
                acc = _norm9(_mm3(depth[:, t], acc))
            if c + 1 < len(firsts):
                state = _polarm(acc)
                keys.append(state)
        keys = torch.stack(keys, 1) if keys else depth[:, :0]
        return dict(keys=keys, a=_readout(keys, s["read"]) if keys.shape[1] else keys)
    if kind == "final_ca":
        sc = (f["q"] @ f["k"].transpose(1, 2).contiguous() * s["scale"]).masked_fill(~s["allowed"], -math.inf)
        w = torch.softmax(sc, -1).nan_to_num(0.0)          # a row without a key gives zero
        return dict(out=w @ f["v"], lse=torch.logsumexp(sc, -1))
    B, T, cap, HD = s["B"], s["T"], s["cap"], s["HD"]
    x = f["qkv"].view(B, T, QH + 2 * KVH, HD)
    at = torch.arange(cap - T, cap, device=DEV)
    cos, sin = f["cos"][at][None, :, None], f["sin"][at][None, :, None]
    q, k, v = x.split([QH, KVH, KVH], 2)
    q, k = _rotate(q, cos, sin), _rotate(k, cos, sin)
    kc, vc = f["kc"].clone(), f["vc"].clone()
    kc[:, :, cap - T:], vc[:, :, cap - T:] = k.transpose(1, 2), v.transpose(1, 2)
    c, kctx = _attend(q, kc, vc, torch.arange(cap, device=DEV)[None, :] <= at[:, None])
    return dict(q=q, c=c, kctx=kctx, kc=kc, vc=vc)
