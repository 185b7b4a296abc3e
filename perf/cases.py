"""Performance cases of the sink-sparse attention path on one GPU.

A case is one pass through a public entry point of `sinkattn_amd` (the names that
`sinkattention.*` re-exports), at sizes a user of the framework meets:

  attention   `_block_sparse_attn` on a block mask the program keeps
  inner       `WanSinkSparseInnerAttention.forward`, the default runtime call (sparse
              attention plus the pooled-K/V compensation)
  record      `SinkMaskCalibrator.record`, one layer call of a calibration pass, in each of
              the three pooling modes
  package     a short calibration: two recorded calls, then the mask package
  mask        `_build_direct_mean_coverage_mask` on one layer's mean map
  wan_calib   `WanSinkCalibrationProcessor2_0`, the whole attention layer while calibrating
  zimage      `ZImageStaticSinkProcessor`, the whole attention layer at inference

`listed()` gives the named cases, `draw(rng)` more of the same ranges.  `prepare` makes what
the program holds before the call, `run` is the pass, `work` its unavoidable bytes and
operations, `tolerance` how far two correct implementations may differ, and `exact` the
result in 64 bits by plain torch.
"""
from __future__ import annotations

import math

import torch
import torch.nn as nn

from sinkattn_amd import sparse_attention as sa
from sinkattn_amd import wan_runtime as wr
from sinkattn_amd import zimage_runtime as zr

BLOCK = 128
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
BYTES = {"bf16": 2, "f16": 2, "f32": 4}
GAP = 30  # the compensation branch's default sample gap


def listed():
    return [
        # a short clip or a test-sized call: 16 q-blocks, latency is all of it
        dict(name="attn_short", kind="attention", dtype="bf16", B=1, H=2, N=1000, D=128,
             lo=0.5, hi=0.5, dense_heads=0, lse=True, layout="bnhd"),
        # the fp32 call a CPU user can check against (four sink keys, a mostly kept mask)
        dict(name="attn_f32", kind="attention", dtype="f32", B=1, H=12, N=4096, D=128,
             lo=0.74, hi=0.74, dense_heads=0, lse=True, layout="bhnd"),
        # head dim 64 in half precision, a ragged length
        dict(name="attn_d64_f16", kind="attention", dtype="f16", B=2, H=16, N=8100, D=64,
             lo=0.25, hi=0.25, dense_heads=0, lse=False, layout="bhnd"),
        # one 14B layer at 720p: 21 x 45 x 80 tokens, heads from 5% to 30% kept, one dense
        dict(name="attn_720p", kind="attention", dtype="bf16", B=1, H=40, N=75600, D=128,
             lo=0.05, hi=0.30, dense_heads=1, lse=False, layout="bnhd"),
        # the 1.3B layer at 480p with the default compensation, both halves of a CFG pair
        dict(name="wan_inner", kind="inner", dtype="bf16", B=2, H=12, N=32760, D=128,
             lo=0.20, hi=0.20, dense_heads=0, mode="pooled_kv"),
        # one recorded layer call in the default pooling mode of the config (block maxima)
        dict(name="record_max", kind="record", dtype="bf16", B=2, H=12, N=32760, D=128, block=128,
             pooling="triton"),
        # and with mean-pooled scores
        dict(name="record_mean", kind="record", dtype="bf16", B=2, H=12, N=32760, D=128, block=128,
             pooling="mean"),
        # one recorded call in the exact mode, the joint image + text sequence of a 2048^2 image
        dict(name="record_exact", kind="record", dtype="bf16", B=1, H=30, N=16896, D=128, block=128,
             pooling="exact"),
        # a short fp32 calibration and its package: the whole offline pass in small
        dict(name="package_f32", kind="package", dtype="f32", B=1, H=12, N=4096, D=128, block=128),
        # one layer's coverage mask from its mean map
        dict(name="mask_480p", kind="mask", H=12, nb=256),
        # the whole attention layer while calibrating: projections, norm, rotary, pooling, dense
        # attention, output projection
        dict(name="wan_calib", kind="wan_calib", dtype="bf16", B=1, H=12, N=32760, D=128),
        # the whole inference layer of a 1024^2 image pair with prompts of different lengths
        dict(name="zimage_1024", kind="zimage", dtype="bf16", H=30, D=128, side=64, text=224, text2=77,
             density=0.25, mode="pooled_kv", dense=False),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["attention", "attention", "attention", "inner", "record", "record", "record", "mask",
                       "package", "wan_calib", "zimage"])
    if kind == "attention":
        dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
        D = rng.choice([128, 128, 64, 32])
        H, N = rng.randint(1, 24), size(200, 30000 if dtype != "f32" else 9000)
        lo = rng.uniform(0.05, 0.5)
        return dict(kind=kind, dtype=dtype, B=rng.randint(1, 2), H=H, N=N, D=D, lo=round(lo, 3),
                    hi=round(rng.uniform(lo, 0.8), 3), dense_heads=rng.choice([0, 0, 1]),
                    lse=rng.choice([True, False]), layout=rng.choice(["bhnd", "bnhd"]))
    if kind == "inner":
        lo = rng.uniform(0.05, 0.3)
        return dict(kind=kind, dtype=rng.choice(["bf16", "f16"]), B=rng.randint(1, 2), H=rng.randint(2, 24),
                    N=size(2000, 33000), D=128, lo=round(lo, 3), hi=round(rng.uniform(lo, 0.5), 3),
                    dense_heads=rng.choice([0, 1]), mode=rng.choice(["pooled_kv", "pooled_kv", "none"]))
    if kind == "record":
        dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
        return dict(kind=kind, dtype=dtype, B=rng.randint(1, 2), H=rng.randint(2, 24),
                    N=size(1000, 24000 if dtype != "f32" else 7000),
                    D=128, block=rng.choice([128, 128, 64]), pooling=rng.choice(["exact", "triton", "mean"]))
    if kind == "package":
        return dict(kind=kind, dtype=rng.choice(["bf16", "f32"]), B=rng.randint(1, 2), H=rng.randint(2, 12),
                    N=size(600, 6000), D=128, block=128)
    if kind == "mask":
        return dict(kind=kind, H=rng.randint(2, 40), nb=size(20, 600))
    if kind == "wan_calib":
        return dict(kind=kind, dtype="bf16", B=rng.randint(1, 2), H=12, N=size(1500, 20000), D=128)
    return dict(kind=kind, dtype="bf16", H=30, D=128, side=rng.choice([32, 48, 64, 80]),
                text=rng.randint(8, 500), text2=rng.choice([0, rng.randint(8, 500)]),
                density=round(rng.uniform(0.1, 0.4), 3),
                mode=rng.choice(["none", "pooled_kv"]), dense=rng.random() < 0.25)


# --- inputs ------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _qkv(case, g):
    """N(0, 1) Q/K/V as [B, H, N, D] (views of [B, N, H, D] memory for the layout a projection
    gives), with four sink keys per head among the first 1024 tokens."""
    B, H, N, D = case["B"], case["H"], case["N"], case["D"]
    shape = (B, N, H, D) if case.get("layout", "bnhd") == "bnhd" else (B, H, N, D)
    out = [torch.randn(shape, device="cuda", dtype=DTYPES[case["dtype"]], generator=g) for _ in range(3)]
    if shape[1] != H or shape[2] != N:
        out = [t.permute(0, 2, 1, 3) for t in out]
    pos = torch.randint(0, min(N, 1024), (H, 4), device="cuda", generator=g)
    for h in range(H):
        out[1][:, h, pos[h]] *= 6.0
    return out


def _densities(case):
    H, dense = case["H"], min(case["dense_heads"], case["H"])
    d = [case["lo"] + (case["hi"] - case["lo"]) * h / max(1, H - 1) for h in range(H)]
    return [1.0] * dense + d[dense:]


def _head_mask(case, nb, g):
    """[H, nb, nb] bool: each head's own density, diagonal and first column always kept."""
    d = torch.tensor(_densities(case), device="cuda").view(-1, 1, 1)
    m = torch.rand(case["H"], nb, nb, device="cuda", generator=g) < d
    i = torch.arange(nb, device="cuda")
    m[:, i, i] = True
    m[:, :, 0] = True
    return m


def _kept(density, nb):
    """Expected kept blocks of one head's mask."""
    return nb * nb * density + (2 * nb - 1) * (1.0 - density)


class _Attn(nn.Module):
    """The attention module a diffusion transformer's block holds: projections, QK norms."""

    def __init__(self, heads, dim, norm_dim, dtype, g):
        super().__init__()
        self.heads = heads
        lin = [nn.Linear(dim, dim, device="meta") for _ in range(4)]
        norms = [nn.RMSNorm(norm_dim, eps=1e-6, device="meta") for _ in range(2)]
        for m in lin:
            m.weight = nn.Parameter((torch.randn(dim, dim, device="cuda", generator=g) / math.sqrt(dim)).to(dtype))
            m.bias = nn.Parameter((0.02 * torch.randn(dim, device="cuda", generator=g)).to(dtype))
        for m in norms:
            m.weight = nn.Parameter((1.0 + 0.1 * torch.randn(norm_dim, device="cuda", generator=g)).to(dtype))
        self.to_q, self.to_k, self.to_v = lin[:3]
        self.to_out = nn.ModuleList([lin[3], nn.Identity()])
        self.norm_q, self.norm_k = norms
        self.add_k_proj = self.add_v_proj = self.norm_added_k = None


def _angles(n, half, g):
    inv = torch.pow(10000.0, -torch.arange(half, device="cuda", dtype=torch.float32) / half)
    return torch.arange(n, device="cuda", dtype=torch.float32).view(-1, 1) * inv


def _zimage_config(case):
    return zr.build_zimg_sink_config(config_overrides=dict(
        token_width=case["side"], token_height=case["side"], dynamic_mode=case["mode"], sample_gap=GAP,
        force_dense_steps=[0] if case["dense"] else None))


def _zimage_texts(case):
    """Prompt lengths of the batch: one sample, or two when the second is given."""
    return [case["text"]] + ([case["text2"]] if case["text2"] else [])


def _zimage_lens(case):
    return [case["side"] ** 2 + t for t in _zimage_texts(case)]


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    st = {"kind": kind}
    if kind in ("attention", "inner"):
        st["q"], st["k"], st["v"] = _qkv(case, g)
        m = _head_mask(case, -(-case["N"] // BLOCK), g)
        if kind == "attention":
            st["mask"] = m.unsqueeze(0).expand(case["B"], -1, -1, -1).contiguous()
            st["lse"] = case["lse"]
        else:
            cfg = sa.SinkSparseConfig(dynamic_mode=case["mode"], sample_gap=GAP)
            st["mod"] = wr.WanSinkSparseInnerAttention(0, m.cpu(), cfg)
    elif kind == "record":
        st["q"], st["k"], st["v"] = _qkv(case, g)
        st["cfg"] = sa.SinkSparseConfig(block_size=case["block"], pooling_mode=case["pooling"])
    elif kind == "package":
        st["calls"] = [_qkv(case, g) for _ in range(2)]
        st["cfg"] = sa.SinkSparseConfig(block_size=case["block"], pooling_mode="exact")
    elif kind == "mask":
        H, nb = case["H"], case["nb"]
        # a mean softmax-mass map: positive rows that sum to one, a few columns that draw more
        s = torch.randn(H, nb, nb, device="cuda", generator=g)
        s[:, :, torch.randint(0, nb, (4,), device="cuda", generator=g)] += 3.0
        st["scores"] = torch.softmax(s, dim=-1)
        st["cfg"] = sa.SinkSparseConfig()
    elif kind == "wan_calib":
        dim, dt = case["H"] * case["D"], DTYPES[case["dtype"]]
        st["attn"] = _Attn(case["H"], dim, dim, dt, g)
        st["x"] = torch.randn(case["B"], case["N"], dim, device="cuda", dtype=dt, generator=g)
        ang = _angles(case["N"], case["D"] // 2, g).repeat_interleave(2, dim=-1).view(1, case["N"], 1, case["D"])
        st["rotary"] = (ang.cos(), ang.sin())
        st["cfg"] = sa.SinkSparseConfig(pooling_mode="exact")
    else:
        dim, dt = case["H"] * case["D"], DTYPES[case["dtype"]]
        lens = _zimage_lens(case)
        n, B = -(-max(lens) // 32) * 32, len(lens)
        st["attn"] = _Attn(case["H"], dim, case["D"], dt, g)
        st["x"] = torch.randn(B, n, dim, device="cuda", dtype=dt, generator=g)
        st["valid"] = torch.arange(n, device="cuda").view(1, -1) < torch.tensor(lens, device="cuda").view(-1, 1)
        ang = _angles(n, case["D"] // 2, g)
        st["freqs"] = torch.polar(torch.ones_like(ang), ang).unsqueeze(0).expand(B, -1, -1).contiguous()
        cfg = _zimage_config(case)
        total = zr._fixed_block_shape(cfg)[2]
        m = _head_mask(dict(case, lo=case["density"], hi=case["density"], dense_heads=0), total, g)
        st["mask"] = m.cpu()
        state = zr.SinkRuntimeState()
        # a generation in its first step (forced dense when the configuration says so)
        state.current_step = 0
        st["proc"] = zr.ZImageStaticSinkProcessor(layer_idx=1, total_layers=30, sink_mask=m.cpu(), config=cfg,
                                                  runtime_state=state)
    return st


@torch.no_grad()
def run(st):
    kind = st["kind"]
    if kind == "attention":
        out, lse = sa._block_sparse_attn(st["q"], st["k"], st["v"], st["mask"], return_lse=st["lse"])
        return [out] if lse is None else [out, lse]
    if kind == "inner":
        return [st["mod"](st["q"], st["k"], st["v"])]
    if kind == "record":
        cal = sa.SinkMaskCalibrator(st["cfg"])
        cal.record(0, st["q"], st["k"], st["v"])
        return [cal.score_sums[0], cal.score_sq_sums[0]]
    if kind == "package":
        cal = sa.SinkMaskCalibrator(st["cfg"])
        for q, k, v in st["calls"]:
            cal.record(0, q, k, v)
        package = cal.build_package(include_scores=True)
        return [package["mean_scores"]["0"], cal.score_sums[0], package["sink_masks"]["0"]]
    if kind == "mask":
        return [sa._build_direct_mean_coverage_mask(st["scores"], st["cfg"])]
    if kind == "wan_calib":
        cal = sa.SinkMaskCalibrator(st["cfg"])
        out = wr.WanSinkCalibrationProcessor2_0(cal, 0)(st["attn"], st["x"], rotary_emb=st["rotary"])
        return [out, cal.score_sums[0]]
    return [st["proc"](st["attn"], st["x"], attention_mask=st["valid"], freqs_cis=st["freqs"])]


# --- work and tolerance ---------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "mask":
        n = case["H"] * case["nb"] ** 2
        return {"bytes": 5 * n, "flops": 2 * n}
    H, D, es = case["H"], case["D"], BYTES[case["dtype"]]
    if kind == "zimage":
        dim, flops, toks = H * D, 0.0, 0
        for n, t in zip(_zimage_lens(case), _zimage_texts(case)):
            nb, tb = -(-n // BLOCK), -(-t // BLOCK)
            ib = nb - tb
            share = _kept(case["density"], ib) / ib ** 2
            pairs = n * n if case["dense"] else share * (n - t) ** 2 + 2.0 * t * n - t * t
            if case["mode"] == "pooled_kv" and not case["dense"]:
                pairs += (n - t) * ((n - t) / GAP + t)
            flops += 4.0 * H * D * pairs + 8.0 * n * dim * dim
            toks += n
        return {"bytes": int(2 * toks * dim * es + 4 * dim * dim * es), "flops": int(flops)}
    B, N = case["B"], case["N"]
    elems, nb = B * H * N * D, -(-N // case.get("block", BLOCK))
    if kind in ("attention", "inner"):
        pairs = sum(_kept(d, nb) / nb ** 2 for d in _densities(case)) * N * N
        if case.get("mode") == "pooled_kv":
            pairs += H * N * (N / GAP)
        return {"bytes": 4 * elems * es + (B * H * N * es if case.get("lse") else 0),
                "flops": int(4.0 * D * B * pairs)}
    if kind == "wan_calib":
        dim = H * D
        return {"bytes": int(2 * B * N * dim * es + 4 * dim * dim * es + 4 * H * nb * nb),
                "flops": int(6.0 * B * H * N * N * D + 8.0 * B * N * dim * dim)}
    calls = 2 if kind == "package" else 1
    if case.get("pooling") == "mean":
        flops = 2.0 * B * H * nb * nb * D + 2.0 * elems
    else:
        flops = 2.0 * B * H * N * N * D
    return {"bytes": calls * 2 * elems * es + 8 * H * nb * nb, "flops": int(calls * flops)}


def tolerance(case):
    """About four times the distance of the path's results from the 64-bit ones (measured over
    the listed cases and draws): 1.6e-3 for bf16 attention (P and the output are rounded to
    16 bits), 2.1e-4 for f16, 7.7e-6 for f32 (products of split operands), 1-6e-7 for maps
    summed in 32 bits, 1.5e-4 for block maxima (16-bit roundings that flip with the order of
    a dot product's sum)."""
    kind, dtype = case["kind"], case.get("dtype")
    if kind == "mask":
        return "exact"
    if kind in ("attention", "inner"):
        return {"rel": {"bf16": 7e-3, "f16": 1e-3, "f32": 3e-5}[dtype]}
    if kind == "package":
        # masks: blocks whose mean sits on the coverage cut may go either way
        return {"rel": 3e-6, "differ": 1e-3}
    if kind == "record":
        if case["pooling"] == "triton":
            return {"rel": 1e-5 if dtype == "f32" else 1e-3}
        return {"rel": 3e-6}
    return {"rel": 1e-2 if kind == "wan_calib" else 2e-2}


# --- the results in 64 bits ---------------------------------------------------------------
def _attend64(q, k, v, mask=None, kd=None, vd=None, gap=1, comp_rows=0):
    """softmax(Q K^T / sqrt(D) + M) V and the LSE, one head at a time; the first `comp_rows` rows
    also see every key of kd/vd counted `gap` times."""
    B, H, N, D = q.shape
    Nk = k.shape[2]
    out = torch.zeros(B, H, N, D, dtype=torch.float64, device=q.device)
    lse = torch.zeros(B, H, N, 1, dtype=torch.float64, device=q.device)
    scale = 1.0 / math.sqrt(D)
    for b in range(B):
        for h in range(H):
            kt, vv = k[b, h].double().t().contiguous(), v[b, h].double().contiguous()
            if kd is not None:
                kdt, vdd = kd[b, h].double().t().contiguous(), vd[b, h].double().contiguous()
            for r0 in range(0, N, 16 * BLOCK):
                r1 = min(N, r0 + 16 * BLOCK)
                qr = q[b, h, r0:r1].double() * scale
                s = qr @ kt
                if mask is not None:
                    rows = mask[b, h, r0 // BLOCK:-(-r1 // BLOCK)]
                    keep = rows.repeat_interleave(BLOCK, 0)[:r1 - r0].repeat_interleave(BLOCK, 1)[:, :Nk]
                    s.masked_fill_(~keep, -math.inf)
                vals = vv
                c = min(max(comp_rows - r0, 0), r1 - r0)
                if kd is not None and c > 0:
                    sd = qr @ kdt + math.log(gap)
                    sd[c:] = -math.inf
                    s, vals = torch.cat([s, sd], 1), torch.cat([vv, vdd], 0)
                m = s.amax(1, keepdim=True)
                s.sub_(m).exp_()
                l = s.sum(1, keepdim=True)
                out[b, h, r0:r1] = (s @ vals) / l
                lse[b, h, r0:r1] = m + l.log()
    return out, lse


def _mean_pool64(x, gap):
    n = x.shape[2]
    x = x.double()
    pad = (-n) % gap
    if pad:
        x = torch.cat([x, x[:, :, -1:].expand(-1, -1, pad, -1)], 2)
    return x.unflatten(2, (-1, gap)).mean(3)


def _record64(q, k, block, pooling, dtype):
    """The batch mean of the block scores, [H, nb, nb]."""
    B, H, N, D = q.shape
    nb, scale = -(-N // block), 1.0 / math.sqrt(D)
    out = torch.zeros(H, nb, nb, dtype=torch.float64, device=q.device)
    step = max(1, 2048 // block)
    if pooling == "mean":
        qp, kp = _mean_pool64(q, block), _mean_pool64(k, block)
        for b in range(B):
            for h in range(H):
                out[h] += torch.softmax((qp[b, h] @ kp[b, h].t().contiguous()) * scale, -1)
        return out / B
    starts = torch.arange(nb, device=q.device) * block
    for b in range(B):
        for h in range(H):
            kt = k[b, h].double().t().contiguous()
            po = torch.zeros(nb, nb, dtype=torch.float64, device=q.device)
            for i0 in range(0, nb, step):
                i1 = min(nb, i0 + step)
                r0, r1 = i0 * block, min(N, i1 * block)
                s = q[b, h, r0:r1].double() @ kt
                fill = 0.0 if pooling == "exact" else -math.inf
                if pooling == "exact":
                    s = torch.softmax(s * scale, 1)
                s = nn.functional.pad(s, (0, nb * block - N), value=fill).unflatten(1, (nb, block))
                if pooling == "exact":
                    s = s.sum(2)
                    s = nn.functional.pad(s, (0, 0, 0, (i1 - i0) * block - (r1 - r0)))
                    rows = torch.minimum(starts[i0:i1] + block, torch.tensor(N, device=q.device)) - starts[i0:i1]
                    po[i0:i1] = s.unflatten(0, (i1 - i0, block)).sum(1) / rows.view(-1, 1)
                else:  # block maxima in the input type, relative to the row's unrounded maximum
                    s = s.amax(2) * (scale * 1.44269504)
                    m = s.amax(1, keepdim=True)
                    e = torch.exp2(s.to(DTYPES[dtype]).double() - m)
                    e = nn.functional.pad(e, (0, 0, 0, (i1 - i0) * block - (r1 - r0)))
                    po[i0:i1] = e.unflatten(0, (i1 - i0, block)).amax(1).to(DTYPES[dtype]).double()
            if pooling != "exact":
                total = po.sum(1, keepdim=True).to(DTYPES[dtype]).double()
                po = (po / total).to(DTYPES[dtype]).double()
            out[h] += po
    return out / B


def _layer_qkv64(st, x, cos, sin, per_head_norm):
    """Q, K, V [B, H, N, d] of an attention layer in 64 bits."""
    attn = st["attn"]
    H = attn.heads
    out = []
    for lin, norm in ((attn.to_q, attn.norm_q), (attn.to_k, attn.norm_k), (attn.to_v, None)):
        y = x.double() @ lin.weight.double().t().contiguous() + lin.bias.double()
        if per_head_norm:
            y = y.unflatten(-1, (H, -1))
        if norm is not None:
            y = y * torch.rsqrt(y.square().mean(-1, keepdim=True) + norm.eps) * norm.weight.double()
        if not per_head_norm:
            y = y.unflatten(-1, (H, -1))
        if norm is not None:
            a, b = y[..., 0::2], y[..., 1::2]
            y = torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)
        out.append(y.transpose(1, 2).contiguous())
    return out


def _project64(attn, o):
    lin = attn.to_out[0]
    return o.transpose(1, 2).flatten(2) @ lin.weight.double().t().contiguous() + lin.bias.double()


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind == "mask":
        return None
    st = prepare(case, seed)
    if kind in ("attention", "inner"):
        q, k, v = st["q"], st["k"], st["v"]
        if kind == "attention":
            out, lse = _attend64(q, k, v, st["mask"])
            return [out, lse] if case["lse"] else [out]
        mask = st["mod"].sink_mask.cuda().unsqueeze(0).expand(case["B"], -1, -1, -1)
        if case["mode"] == "none":
            return [_attend64(q, k, v, mask)[0]]
        return [_attend64(q, k, v, mask, _mean_pool64(k, GAP), _mean_pool64(v, GAP), GAP, case["N"])[0]]
    if kind == "record":
        s = _record64(st["q"], st["k"], case["block"], case["pooling"], case["dtype"])
        return [s, s.square()]
    if kind == "package":
        s = sum(_record64(q, k, case["block"], "exact", case["dtype"]) for q, k, _ in st["calls"])
        return [(s / 2).cpu(), s, None]
    attn = st["attn"]
    if kind == "wan_calib":
        cos, sin = (t[0, :, 0, 0::2].double().view(1, case["N"], 1, -1) for t in st["rotary"])
        q, k, v = _layer_qkv64(st, st["x"], cos, sin, False)
        return [_project64(attn, _attend64(q, k, v)[0]), _record64(q, k, BLOCK, "exact", case["dtype"])]
    f = st["freqs"].unsqueeze(2)
    q, k, v = _layer_qkv64(st, st["x"], f.real.double(), f.imag.double(), True)
    cfg, img = _zimage_config(case), case["side"] ** 2
    _, ib, total = zr._fixed_block_shape(cfg)
    o = torch.zeros_like(q)
    for b, n in enumerate(_zimage_lens(case)):
        tb = -(-(n - img) // BLOCK)
        idx = torch.cat([torch.arange(ib), torch.arange(total - tb, total)])
        m = st["mask"][:, idx][:, :, idx].cuda().unsqueeze(0)
        m[..., ib:, :] = True
        m[..., :, ib:] = True
        qs, ks, vs = (t[b:b + 1, :, :n] for t in (q, k, v))
        if case["dense"]:
            o[b:b + 1, :, :n] = _attend64(qs, ks, vs)[0]
        elif case["mode"] == "none":
            o[b:b + 1, :, :n] = _attend64(qs, ks, vs, m)[0]
        else:
            kd, vd = (torch.cat([_mean_pool64(t[:, :, :img], GAP), t[:, :, img:]], 2) for t in (ks, vs))
            o[b:b + 1, :, :n] = _attend64(qs, ks, vs, m, kd, vd, GAP, img)[0]
    return [_project64(attn, o)]
