"""The work this framework is used for, as a list of cases that can be timed and compared.

A case is a dict of plain values; `prepare` makes its inputs on the GPU from a seed,
`run` makes one pass through the public entry points, `work` states the bytes and
floating-point operations of that pass and `exact` restates it in 64 bits in plain
torch.  Kinds of case:

  attn      attn_sm80.attn / h3attn.attn_fwd on [B,H,S,128] tensors: dense attention
  layer     a DiT attention layer through the patched Attention.forward: in-place
            qk-RMSNorm + RoPE on the fused QKV output, attention on its strided
            views, O as [S, H*128]; with `blk`, under the block-sparse override
            (block means from the prologue, block map, block-sparse attention).
            The QKV and output projections are the model's own matrix products,
            so the layer has identities in their places.
  sla       h3attn.sla.sparse_attention on [1,H,S,128] tensors: block map from q
            and k, then block-sparse attention
  map       a caller's own 0/1 block map -> LUT -> block-sparse attention
  prologue  the in-place qk-RMSNorm + RoPE alone, on the fused QKV layout

H = 56 and S = 42120 are the video DiT's heads and packed tokens; 28 and 14 heads are
a rank's share when 2 or 4 GPUs split the heads.
"""
from __future__ import annotations

import math
import os
import sys

import torch

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "minimaxh3-on-a100-x4_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import attn_sm80  # noqa: E402
from h3attn import hooks, ops, sla  # noqa: E402

D = 128
EPS = 1e-6
FULL_S, FULL_H = 42120, 56


# ---------------------------------------------------------------------------
# cases
def listed():
    return [
        # A short sequence through the drop-in attn(): what a call costs before any work.
        {"name": "attn_h2_s300", "kind": "attn", "B": 1, "H": 2, "Sq": 300, "Skv": 300},
        # The small benchmark shape: a preview-sized clip on few heads, a launch-bound layer.
        {"name": "attn_h4_s2048", "kind": "attn", "B": 1, "H": 4, "Sq": 2048, "Skv": 2048},
        # Ragged lengths, a batch, and keys of another length than the queries, as padded
        # sequence shards give.
        {"name": "attn_b2_h14_q1160_kv4104", "kind": "attn", "B": 2, "H": 14, "Sq": 1160, "Skv": 4104},
        # One rank's 14 heads of the full sequence.
        {"name": "attn_h14_s42120", "kind": "attn", "B": 1, "H": 14, "Sq": FULL_S, "Skv": FULL_S},
        # The headline: all heads of the full sequence, 50 of these per denoise step.
        {"name": "attn_h56_s42120", "kind": "attn", "B": 1, "H": 56, "Sq": FULL_S, "Skv": FULL_S},
        # A whole layer of a shorter clip: prologue, dense attention on strided views.
        {"name": "layer_h56_s8192", "kind": "layer", "H": 56, "S": 8192},
        # A block-sparse layer of a short clip on a rank's heads, at the node's default keep and block.
        {"name": "layer_sla64_h14_s4104", "kind": "layer", "H": 14, "S": 4104, "blk": 64, "topk": 0.35},
        # The block-sparse layer of the full model at the keep most layers of every preset use.
        {"name": "layer_sla64_h56_s42120", "kind": "layer", "H": 56, "S": FULL_S, "blk": 64, "topk": 0.15},
        # The 128x128 block-sparse workload: top 25 % plus the diagonal.
        {"name": "sla128_h56_s42120", "kind": "sla", "H": 56, "S": FULL_S, "blk": 128, "topk": 0.25, "diag": True},
        # One of the node's block sizes that run over masked 32-key columns, on two ranks' share.
        {"name": "layer_sla96_h28_s42120", "kind": "layer", "H": 28, "S": FULL_S, "blk": 96, "topk": 0.25},
        # A caller's own block map, turned into a LUT and attended over.
        {"name": "map128_h56_s8192", "kind": "map", "H": 56, "S": 8192, "blk": 128, "keep": 0.25},
        # The prologue alone, judged on bandwidth.
        {"name": "prologue_h56_s8192", "kind": "prologue", "H": 56, "S": 8192, "rot": 128},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _heads(rng):
    return rng.choice([4, 14, 28, 56, _log_int(rng, 1, FULL_H)])


def draw(rng):
    kind = rng.choice(["attn", "attn", "layer", "layer_sla", "layer_sla", "sla", "map", "prologue"])
    H = _heads(rng)
    if kind == "attn":
        B = rng.choice([1, 1, 1, 2])
        sq = _log_int(rng, 100, FULL_S // B)
        skv = sq if rng.random() < 0.7 else _log_int(rng, max(100, sq // 4), min(FULL_S // B, 4 * sq))
        return {"kind": "attn", "B": B, "H": H, "Sq": sq, "Skv": skv}
    if kind == "layer":
        return {"kind": "layer", "H": H, "S": _log_int(rng, 256, FULL_S)}
    if kind == "prologue":
        return {"kind": "prologue", "H": H, "S": _log_int(rng, 256, FULL_S), "rot": rng.choice([64, 128, 128])}
    if kind == "map":
        return {"kind": "map", "H": H, "S": _log_int(rng, 1024, 24000), "blk": rng.choice([64, 128, 128, 192, 256]),
                "keep": rng.choice([0.15, 0.25, 0.5])}
    # The node's default block size, the benchmark's 128, and every other multiple of 16 it offers.
    blk = rng.choice([64, 64, 64, 128, 128, rng.randrange(32, 257, 16)])
    case = {"kind": "layer" if kind == "layer_sla" else "sla", "H": H, "S": _log_int(rng, 1024, FULL_S), "blk": blk,
            "topk": rng.choice([0.15, 0.15, 0.25, 0.35])}
    if kind == "sla" and rng.random() < 0.5:
        case["diag"] = True
    return case


# ---------------------------------------------------------------------------
# inputs
def _smooth(gen, shape):
    """N(0,1) vectors that drift along the tokens (shape [..., S, 128]), a new one every 256 tokens."""
    *lead, S, d = shape
    z = torch.randn(*lead, S // 256 + 2, d, generator=gen, device="cuda")
    pos = torch.arange(S, device="cuda") / 256.0
    lo = pos.floor().long()
    w = (pos - lo)[:, None]
    return z.index_select(-2, lo) * torch.cos(w * (math.pi / 2)) + z.index_select(-2, lo + 1) * torch.sin(w * (math.pi / 2))


def _qkv(gen, B, H, Sq, Skv):
    """q, k, v bf16 [B,H,S,128]: q and k ~ N(0,1) per value, with a part that neighbouring
    tokens share (as neighbouring patches of a video do), v ~ 4 N(0,1)."""
    S = max(Sq, Skv)
    base = _smooth(gen, (B, H, S, D)).mul_(0.6)
    q = (torch.randn(B, H, Sq, D, generator=gen, device="cuda").mul_(0.8) + base[:, :, :Sq]).bfloat16()
    k = (torch.randn(B, H, Skv, D, generator=gen, device="cuda").mul_(0.8) + base[:, :, :Skv]).bfloat16()
    v = torch.randn(B, H, Skv, D, generator=gen, device="cuda").mul_(4.0).bfloat16()
    return q, k, v


def _rope(S, rot):
    """ComfyUI-style rotation table, float32 [1, S, 1, rot/2, 2, 2], theta 10000 over the token index."""
    i = torch.arange(rot // 2, dtype=torch.float64, device="cuda")
    ang = torch.arange(S, dtype=torch.float64, device="cuda")[:, None] * 10000.0 ** (-2.0 * i / rot)
    c, s = torch.cos(ang), torch.sin(ang)
    return torch.stack([c, -s, s, c], dim=-1).reshape(1, S, 1, rot // 2, 2, 2).float()


def _fused(gen, H, S, rot):
    """The fused projection output [S, 3*H*128] before the norm (a scale per token in 0.5 .. 4),
    the norm weights and the RoPE table."""
    q, k, v = _qkv(gen, 1, H, S, S)
    amp = torch.rand(1, 1, S, 1, generator=gen, device="cuda") * 3.5 + 0.5
    qkv = torch.empty(S, 3, H, D, dtype=torch.bfloat16, device="cuda")
    for i, t in enumerate((q * amp, k * amp, v)):
        qkv[:, i] = t[0].transpose(0, 1)
    w = [(1.0 + 0.05 * torch.randn(D, generator=gen, device="cuda")).bfloat16() for _ in range(2)]
    return qkv.view(S, 3 * H * D), w[0], w[1], _rope(S, rot)


def _inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind, H = case["kind"], case["H"]
    if kind == "attn":
        q, k, v = _qkv(gen, case["B"], H, case["Sq"], case["Skv"])
        return {"q": q, "k": k, "v": v}
    S = case["S"]
    if kind in ("layer", "prologue"):
        qkv, qw, kw, rope = _fused(gen, H, S, case.get("rot", D))
        return {"qkv": qkv, "qw": qw, "kw": kw, "rope": rope}
    q, k, v = _qkv(gen, 1, H, S, S)
    s = {"q": q, "k": k, "v": v}
    if kind == "map":
        n = -(-S // case["blk"])
        m = torch.rand(1, H, n, n, generator=gen, device="cuda") < case["keep"]
        m |= torch.eye(n, dtype=torch.bool, device="cuda")
        s["map"] = m.to(torch.uint8)
    return s


class _Norm(torch.nn.Module):
    def __init__(self, weight):
        super().__init__()
        self.weight = torch.nn.Parameter(weight, requires_grad=False)
        self.eps = EPS


class Attention(torch.nn.Module):
    """The parts of the DiT's attention module that the patched forward uses."""

    def __init__(self, heads, qw, kw):
        super().__init__()
        self.heads, self.head_dim = heads, D
        self.qkv_proj, self.out_proj = torch.nn.Identity(), torch.nn.Identity()
        self.q_norm, self.k_norm = _Norm(qw), _Norm(kw)

    def forward(self, x, rope_freqs=None, transformer_options={}):
        raise RuntimeError("this layer always has a rope table and runs the patched forward")


hooks.install(Attention)
hooks.install_scope_patch(Attention)


def _no_fallback(message):
    raise RuntimeError(message)


def prepare(case, seed):
    s = {"case": dict(case), **_inputs(case, seed)}
    if case["kind"] == "layer":
        s["attn"] = Attention(case["H"], s["qw"], s["kw"])
        s["options"] = {}
        if "blk" in case:
            s["options"]["optimized_attention_override"] = hooks.make_sla_override(case["topk"], case["blk"],
                                                                                   log=_no_fallback)
    return s


def _heads_of(s):
    """The q and k views [1,S,H,128] of the fused projection output."""
    S, H = s["qkv"].shape[0], s["case"]["H"]
    f = s["qkv"].view(1, S, 3, H, D)
    return f[:, :, 0], f[:, :, 1]


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "attn":
        return attn_sm80.attn(s["q"], s["k"], s["v"])
    if kind == "layer":
        out = s["attn"].forward(s["qkv"], rope_freqs=s["rope"], transformer_options=s["options"])
        q, k = _heads_of(s)  # normalised and rotated in place
        return {"out": out, "q": q, "k": k}
    if kind == "sla":
        return sla.sparse_attention(s["q"], s["k"], s["v"], case["topk"], case["blk"],
                                    force_diag=case.get("diag", False))
    if kind == "map":
        lut, counts = ops.block_map_to_lut(s["map"])
        out = ops.attn_fwd_blocksparse(s["q"], s["k"], s["v"], lut, counts, case["blk"], case["blk"])
        return {"out": out, "lut": lut, "counts": counts}
    q, k = _heads_of(s)
    ops.rms_rope_split_half_(q, k, s["rope"], s["qw"], s["kw"], epsilon=EPS, rot_dim=case["rot"])
    return {"q": q, "k": k}


# ---------------------------------------------------------------------------
# work and tolerance
def work(case):
    kind, H = case["kind"], case["H"]
    row = 2 * D * H  # bytes of one token of q, k, v or o
    if kind == "attn":
        B, sq, skv = case["B"], case["Sq"], case["Skv"]
        return {"bytes": B * row * (2 * sq + 2 * skv), "flops": 4 * B * H * sq * skv * D}
    S = case["S"]
    if kind == "prologue":
        return {"bytes": 4 * S * row + S * (case["rot"] // 2) * 16, "flops": 0}
    keys, score = S, 0
    if "blk" in case:
        n = -(-S // case["blk"])
        if kind == "map":
            kept = case["keep"] * n + (1 - case["keep"])  # kept at random, and the diagonal
        else:
            kept = sla.keep_count(case["topk"], n)
            if case.get("diag"):
                kept += 1 - kept / n  # the diagonal, where the scores did not keep it
            score = 2 * H * n * n * D
        keys = min(S, kept * case["blk"])
    flops = 4 * H * S * keys * D + score
    if kind == "layer":  # q and k are read and written, v is read, o is written
        return {"bytes": 6 * S * row + S * (D // 2) * 16, "flops": flops}
    return {"bytes": 4 * S * row + (H * n * n if kind == "map" else 0), "flops": flops}


def tolerance(case):
    # bf16 outputs (2^-9 relative rounding), probabilities rounded to bf16 before
    # their product with v, fp32 sums.  The block-sparse kinds select blocks from
    # fp32 scores, where another order of the sums may swap two nearly equal blocks
    # in a few rows (and change those rows by about sqrt(2 / kept blocks)).  Prologue:
    # one bf16 rounding of an fp32 result.  Against 64 bits the dense outputs are
    # 2.3e-3 off, the block-sparse ones 2.3e-3 to 2.6e-3, the prologue's 1.7e-3.
    if case["kind"] == "prologue":
        return {"rel": 6e-3, "max": 3e-2}
    if "topk" in case:
        return {"rel": 1e-2, "max": 0.95}
    return {"rel": 1e-2, "max": 0.3}


# ---------------------------------------------------------------------------
# the same in 64 bits
def _exact_attn(q, k, v, kept=None, blk=0):
    """softmax(q k^T / sqrt(128)) v in float64, [B,H,S,128]; `kept` [B,H,nq,nk] bool masks blocks of blk."""
    B, H, Sq, _ = q.shape
    Skv = k.shape[2]
    out = torch.empty(B, H, Sq, D, dtype=torch.float64, device=q.device)
    step = max(1, min(Sq, (1 << 27) // Skv))  # 1 GiB of scores
    if kept is not None:
        kcol = torch.arange(Skv, device=q.device) // blk
    for b in range(B):
        for h in range(H):
            kt, vh = k[b, h].double().t().contiguous(), v[b, h].double()
            for r in range(0, Sq, step):
                s = torch.mm(q[b, h, r:r + step].double(), kt).mul_(1.0 / math.sqrt(D))
                if kept is not None:
                    rows = kept[b, h].index_select(0, torch.arange(r, min(r + step, Sq), device=q.device) // blk)
                    s.masked_fill_(~rows.index_select(1, kcol), -math.inf)
                s = s.sub_(s.amax(dim=1, keepdim=True)).exp_()
                out[b, h, r:r + step] = torch.mm(s, vh) / s.sum(dim=1, keepdim=True)
    return out


def _exact_map(q, k, topk, blk, diag):
    """Kept blocks [1,H,n,n]: the top share of key blocks by the dot product of block means."""
    _, H, S, _ = q.shape
    n = -(-S // blk)

    def means(x):
        x = x.double()
        pad = torch.zeros(1, H, n * blk, D, dtype=torch.float64, device=x.device)
        pad[:, :, :S] = x
        rows = torch.full((n,), blk, dtype=torch.float64, device=x.device)
        rows[-1] = S - (n - 1) * blk
        return pad.view(1, H, n, blk, D).sum(3) / rows[:, None]

    score = torch.matmul(means(q), means(k).transpose(2, 3).contiguous())
    keep = max(1, min(n, int(math.floor(topk * n + 1e-9))))
    kept = torch.zeros(1, H, n, n, dtype=torch.bool, device=q.device)
    kept.scatter_(3, score.topk(keep, dim=3).indices, True)
    if diag:
        kept |= torch.eye(n, dtype=torch.bool, device=q.device)
    return kept


def _exact_prologue(s, H):
    """q and k [1,S,H,128] after the norm and the rotation, float64."""
    S = s["qkv"].shape[0]
    f = s["qkv"].view(1, S, 3, H, D)
    R = s["rope"].double()[0]  # [S, 1, rot/2, 2, 2]
    half = R.shape[2]
    got = []
    for i, w in ((0, s["qw"]), (1, s["kw"])):
        x = f[:, :, i].double()
        x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()
        a, c = x[..., :half].clone(), x[..., half:2 * half].clone()
        x[..., :half] = R[..., 0, 0] * a + R[..., 0, 1] * c
        x[..., half:2 * half] = R[..., 1, 0] * a + R[..., 1, 1] * c
        got.append(x)
    return got


def exact(case, seed):
    s = _inputs(case, seed)
    kind, H = case["kind"], case["H"]
    if kind == "attn":
        return _exact_attn(s["q"], s["k"], s["v"])
    if kind == "sla":
        kept = _exact_map(s["q"], s["k"], case["topk"], case["blk"], case.get("diag", False))
        return _exact_attn(s["q"], s["k"], s["v"], kept, case["blk"])
    if kind == "map":
        return {"out": _exact_attn(s["q"], s["k"], s["v"], s["map"].bool(), case["blk"]), "lut": None, "counts": None}
    q, k = _exact_prologue(s, H)
    if kind == "prologue":
        return {"q": q, "k": k}
    S = case["S"]
    # The layer stores q and k in its bf16 buffer, and attends over what it stored.
    qh, kh = (t.bfloat16().transpose(1, 2) for t in (q, k))
    vh = s["qkv"].view(1, S, 3, H, D)[:, :, 2].transpose(1, 2)
    kept = _exact_map(qh, kh, case["topk"], case["blk"], False) if "blk" in case else None
    out = _exact_attn(qh, kh, vh, kept, case.get("blk", 0))
    return {"out": out.transpose(1, 2).reshape(S, H * D), "q": q, "k": k}
