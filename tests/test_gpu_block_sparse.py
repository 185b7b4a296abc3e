"""GPU parity of the block-sparse attention forward (sinkattn_block_sparse_fwd) against
the fp32 dense masked-softmax oracle (oracle/torch_ref.dense_masked_attention).

Tolerance: max |out - ref| <= 2e-2 and mean |out - ref| <= 1e-3.  The fp32 lse
the kernels write is held to 4e-3 + 1e-5 |ref|: the head-dim-128 kernel sums the 16-bit P
values it multiplies V with (on the matrix cores), each within 2^-8 relative of the fp32
value for bf16, so its row sum is within 2^-8 relative and its lse within log(1 + 2^-8) =
3.9e-3 of the fp32 one (the other kernels sum fp32 P and stay near 1e-5).  The drop-in's lse,
cast to q.dtype like the reference's, is held to 2e-2 plus that type's rounding.
"""
import math

import pytest
import torch

from oracle import torch_ref
from sinkattn_amd import _lib, ops
from sinkattn_amd import sparse_attention as sa

pytestmark = pytest.mark.gpu

MAX_ABS, MEAN_ABS = 2e-2, 1e-3
LSE_ABS = 4e-3


def _inputs(B, H, Nq, Nk, D, dtype, seed, sink_keys=0, sink_scale=8.0, layout="bhsd"):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(B, H, Nq, D, generator=g)
    k = torch.randn(B, H, Nk, D, generator=g)
    v = torch.randn(B, H, Nk, D, generator=g)
    if sink_keys:
        k[:, :, :sink_keys] *= sink_scale
    dev = "cuda"
    if layout == "bshd":  # [B, N, H, D] memory viewed as [B, H, N, D]
        q = q.transpose(1, 2).contiguous().transpose(1, 2)
        k = k.transpose(1, 2).contiguous().transpose(1, 2)
        v = v.transpose(1, 2).contiguous().transpose(1, 2)
    return q.to(dev, dtype), k.to(dev, dtype), v.to(dev, dtype)


def _random_mask(B, H, nqb, nkb, density, seed, diag=True, col0=True, empty_rows=0):
    g = torch.Generator().manual_seed(seed)
    m = torch.rand(B, H, nqb, nkb, generator=g) < density
    if diag:
        d = torch.arange(min(nqb, nkb))
        m[:, :, d, d] = True
    if col0:
        m[..., 0] = True
    for i in range(empty_rows):
        m[0, 0, (7 * i) % nqb, :] = False
    return m.cuda()


def _check(out, lse, q, k, v, mask, rows=None, scale=None):
    ref_o, ref_l = torch_ref.dense_masked_attention(q, k, v, mask, scale=scale, rows=rows)
    o = out.float().cpu()
    l = lse.float().cpu()
    if rows is not None:
        o = o[:, :, rows.cpu()]
        l = l[:, :, rows.cpu()]
    err = (o - ref_o).abs()
    assert err.max().item() <= MAX_ABS, err.max().item()
    assert err.mean().item() <= MEAN_ABS, err.mean().item()
    fin = torch.isfinite(ref_l)
    assert torch.equal(fin, torch.isfinite(l))
    if lse.dtype == torch.float32:
        assert ((l[fin] - ref_l[fin]).abs() <= LSE_ABS + 1e-5 * ref_l[fin].abs()).all(), \
            (l[fin] - ref_l[fin]).abs().max().item()
    else:
        # lse from the drop-in API is cast to q.dtype like the reference's; allow that rounding
        rnd = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[lse.dtype]
        assert ((l[fin] - ref_l[fin]).abs() <= 2e-2 + rnd * ref_l[fin].abs()).all()
    assert torch.equal(o[~fin.unsqueeze(-1).expand_as(o)], torch.zeros_like(o[~fin.unsqueeze(-1).expand_as(o)]))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("N", [256, 1000])
def test_small_random_masks(dtype, N):
    q, k, v = _inputs(1, 3, N, N, 128, dtype, seed=N)
    nb = math.ceil(N / 128)
    mask = _random_mask(1, 3, nb, nb, 0.4, seed=1)
    plan = ops.block_sparse_plan(mask)
    out, lse = ops.block_sparse_attention(q, k, v, plan)
    torch.cuda.synchronize()
    _check(out, lse, q, k, v, mask)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("D", [32, 64])
def test_head_dims_32_and_64(dtype, D):
    # the register-staged kernel (head dims below 128; the external kernel the reference
    # calls takes 32, 64 and 128), ragged N and Nq != Nk
    q, _, _ = _inputs(2, 3, 700, 700, D, dtype, seed=D)
    _, k, v = _inputs(2, 3, 900, 900, D, dtype, seed=D + 1, sink_keys=3)
    mask = _random_mask(2, 3, 6, 8, 0.4, seed=D)
    out, lse = ops.block_sparse_attention(q, k, v, ops.block_sparse_plan(mask))
    torch.cuda.synchronize()
    _check(out, lse, q, k, v, mask)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Nq,Nk", [(1, 1), (1, 300), (130, 1), (700, 900), (900, 129)])
def test_d128_tiny_and_unequal_lengths(dtype, Nq, Nk):
    # the DMA-staged D=128 kernel on single rows / single keys, ragged last blocks on both
    # sides and Nq != Nk; with one key the output is that key's v row and lse its logit
    q, k, v = _inputs(1, 2, Nq, Nk, 128, dtype, seed=Nq * 1000 + Nk, sink_keys=1)
    nqb, nkb = math.ceil(Nq / 128), math.ceil(Nk / 128)
    mask = _random_mask(1, 2, nqb, nkb, 0.5, seed=Nk)
    out, lse = ops.block_sparse_attention(q, k, v, ops.block_sparse_plan(mask))
    torch.cuda.synchronize()
    _check(out, lse, q, k, v, mask)
    if Nk == 1:
        assert torch.equal(out.float().cpu(), v.float().cpu().expand(-1, -1, Nq, -1))
        logit = (q.float() @ k.float().transpose(-1, -2)).squeeze(-1).cpu() / math.sqrt(128)
        assert (lse.cpu() - logit).abs().max().item() <= 1e-4


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("step", [7.5, 30.0, -12.0])
def test_running_maximum_moves_across_tiles(dtype, step):
    # Key block j gets a score offset of j * step log2 units (through channel 0: q = 1,
    # k = offset / (scale * log2 e)), so the row maximum rises slowly (the softmax reference
    # point lags it by up to 8 and P reaches ~2^7.5), rises fast (moves on every tile) or
    # falls (never moves after the first tile).
    B, H, N, D = 1, 2, 1024, 128
    g = torch.Generator().manual_seed(21)
    q = torch.randn(B, H, N, D, generator=g) * 0.5
    k = torch.randn(B, H, N, D, generator=g) * 0.5
    v = torch.randn(B, H, N, D, generator=g)
    c = (1.0 / math.sqrt(D)) * 1.4426950408889634
    q[..., 0] = 1.0
    offs = torch.arange(N) // 128 * step
    offs = offs - offs.min()
    k[..., 0] = (offs / c).round()
    q, k, v = (x.to("cuda", dtype) for x in (q, k, v))
    mask = _random_mask(B, H, 8, 8, 0.7, seed=5)
    out, lse = ops.block_sparse_attention(q, k, v, ops.block_sparse_plan(mask))
    torch.cuda.synchronize()
    _check(out, lse, q, k, v, mask)


def test_config1_shape_fp32_with_sinks():
    # B=1, H=12, N=4096, d=128, fp32, 4 sink keys scaled 8x.
    q, k, v = _inputs(1, 12, 4096, 4096, 128, torch.float32, seed=0, sink_keys=4)
    mask = _random_mask(1, 12, 32, 32, 0.25, seed=3)
    out, lse = sa._block_sparse_attn(q, k, v, mask, return_lse=True)
    torch.cuda.synchronize()
    assert lse.shape == (1, 12, 4096, 1) and lse.dtype == torch.float32
    rows = torch.randperm(4096, generator=torch.Generator().manual_seed(0))[:512].sort().values
    _check(out, lse[..., 0], q, k, v, mask, rows=rows)


def test_config1_chain_mass_mask_attention():
    """[1,12,4096,128] fp32 as one chain: exact block mass -> coverage-0.85 mask -> sparse
    attention on that mask (sparse_attention.py:145-227, 268-376, 710-776).

    fp32 [1,12,4096,128], keys 0..3 x8.  Mass within 1e-5 relative of the oracle; the mask
    bit-exact with the oracle's builder on the same pooled map; attention on that mask within
    2e-2 / 1e-3 of the dense masked softmax (1024 rows per head)."""
    q, k, v = _inputs(1, 12, 4096, 4096, 128, torch.float32, seed=0, sink_keys=4)
    cfg = sa.SinkSparseConfig(pooling_mode="exact", offline_direct_coverage=0.85)
    mass = sa._compute_block_scores(q, k, v, cfg)
    torch.cuda.synchronize()
    assert mass.shape == (1, 12, 32, 32) and mass.dtype == torch.float32
    ref = torch_ref.exact_block_mass(q, k).double()
    rel = ((mass.cpu().double() - ref).abs() / ref.abs().clamp_min(1e-30))
    assert bool(((mass.cpu().double() - ref).abs() <= 1e-5 * ref.abs() + 1e-8).all()), rel.max().item()
    mean_scores = mass.mean(dim=0)                                # batch mean, [12, 32, 32]
    mask = sa._build_direct_mean_coverage_mask(mean_scores, cfg)
    assert mask.dtype == torch.bool and mask.is_cuda
    want = torch_ref.coverage_mask(mean_scores.cpu(), coverage=0.85, keep_diagonal=True)
    assert torch.equal(mask.cpu(), want)
    density = mask.float().mean().item()
    assert 0.0 < density < 1.0, density                           # the sinks make it sparse
    block_mask = mask.unsqueeze(0).expand(1, -1, -1, -1)
    out, lse = sa._block_sparse_attn(q, k, v, block_mask, return_lse=True)
    torch.cuda.synchronize()
    rows = torch.randperm(4096, generator=torch.Generator().manual_seed(1))[:1024].sort().values
    _check(out, lse[..., 0], q, k, v, block_mask, rows=rows)


def test_full_mask_equals_dense_sdpa():
    q, k, v = _inputs(2, 4, 640, 640, 128, torch.bfloat16, seed=5)
    mask = torch.ones(2, 4, 5, 5, dtype=torch.bool, device="cuda")
    out, _ = sa._block_sparse_attn(q, k, v, mask, return_lse=False)
    ref = torch.nn.functional.scaled_dot_product_attention(q.float().cpu(), k.float().cpu(), v.float().cpu())
    err = (out.float().cpu() - ref).abs()
    assert err.max().item() <= MAX_ABS and err.mean().item() <= MEAN_ABS


def test_diagonal_mask_is_block_local_attention():
    q, k, v = _inputs(1, 2, 512, 512, 128, torch.bfloat16, seed=6)
    mask = torch.eye(4, dtype=torch.bool, device="cuda").expand(1, 2, 4, 4).contiguous()
    out, lse = sa._block_sparse_attn(q, k, v, mask)
    qs, ks, vs = (t.float().cpu().view(1, 2, 4, 128, 128) for t in (q, k, v))
    ref = torch.nn.functional.scaled_dot_product_attention(qs, ks, vs).view(1, 2, 512, 128)
    err = (out.float().cpu() - ref).abs()
    assert err.max().item() <= MAX_ABS and err.mean().item() <= MEAN_ABS


def test_empty_rows_ragged_and_strided_bshd():
    # ragged N (last block 50 keys), rows with no listed block, [B,N,H,D] memory views
    q, k, v = _inputs(2, 3, 690, 690, 128, torch.bfloat16, seed=7, layout="bshd")
    mask = _random_mask(2, 3, 6, 6, 0.3, seed=8, diag=False, col0=False, empty_rows=2)
    out, lse = sa._block_sparse_attn(q, k, v, mask)
    torch.cuda.synchronize()
    _check(out, lse[..., 0], q, k, v, mask)
    assert out.stride() == (690 * 3 * 128, 128, 3 * 128, 1)


def test_head_dim_64_and_cross_lengths():
    q, _, _ = _inputs(1, 2, 300, 300, 64, torch.bfloat16, seed=9)
    _, k, v = _inputs(1, 2, 1092, 1092, 64, torch.bfloat16, seed=10)
    mask = _random_mask(1, 2, 3, 9, 0.5, seed=11)
    out, lse = sa._block_sparse_attn(q, k, v, mask)
    torch.cuda.synchronize()
    _check(out, lse[..., 0], q, k, v, mask)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("Nq,Nk,layout", [(1, 1, "bhsd"), (31, 129, "bshd"), (130, 1, "bhsd"), (257, 1000, "bshd"),
                                          (900, 640, "bhsd")])
def test_small_head_dims_edges_and_key_strides(dtype, D, Nq, Nk, layout):
    """Remainders of the 128-row tiles at head dims 32 and 64, both layouts; and keys whose rows
    overlap (a broadcast key dim), which the buffer copies cannot address.  The row sums are
    fp32 sums of unrounded exponentials: the lse is held to 1e-4 + 1e-5 |lse|."""
    q, k, v = _inputs(2, 3, Nq, Nk, D, dtype, seed=Nq + Nk, layout=layout)
    mask = _random_mask(2, 3, -(-Nq // 128), -(-Nk // 128), 0.5, seed=3, empty_rows=1 if Nq > 128 else 0)
    plan = ops.block_sparse_plan(mask)
    out, lse = ops.block_sparse_attention(q, k, v, plan)
    _check(out, lse, q, k, v, mask)
    ref_l = torch_ref.dense_masked_attention(q, k, v, mask)[1]
    fin = torch.isfinite(ref_l)
    assert ((lse.cpu() - ref_l)[fin].abs() <= 1e-4 + 1e-5 * ref_l[fin].abs()).all()
    ke, ve = k[:, :, :1].expand(-1, -1, Nk, -1), v[:, :, :1].expand(-1, -1, Nk, -1)
    assert ke.stride(2) == 0 or Nk == 1
    oe, le = ops.block_sparse_attention(q, ke, ve, plan)
    _check(oe, le, q, ke, ve, mask)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("Nq,Nk,layout", [(1, 1, "bhsd"), (31, 65, "bshd"), (130, 64, "bhsd"), (257, 1000, "bshd"),
                                          (900, 577, "bhsd")])
def test_f32_steps_edges(D, Nq, Nk, layout):
    """fp32 operands in steps of 64 keys: last blocks of one and of two steps, ragged rows, a broadcast
    key dim.  Operands split into bf16 pairs keep 16 mantissa bits (2^-17 relative), so a logit
    is within 3 * 2^-17 * |q||k| / sqrt(D) <= 3 * 2^-17 * 2 sqrt(D) of its exact value and the
    output, an average of |v| <= 5, within 2.6e-3; 2e-4 is what random rounding leaves of it."""
    q, k, v = _inputs(1, 3, Nq, Nk, D, torch.float32, seed=Nq + Nk, layout=layout)
    mask = _random_mask(1, 3, -(-Nq // 128), -(-Nk // 128), 0.5, seed=5, empty_rows=1 if Nq > 128 else 0)
    plan = ops.block_sparse_plan(mask)
    for kk, vv in ((k, v), (k[:, :, :1].expand(-1, -1, Nk, -1), v[:, :, :1].expand(-1, -1, Nk, -1))):
        out, lse = ops.block_sparse_attention(q, kk, vv, plan)
        _check(out, lse, q, kk, vv, mask)
        ref_o, ref_l = torch_ref.dense_masked_attention(q, kk, vv, mask)
        fin = torch.isfinite(ref_l)
        assert (out.cpu() - ref_o).abs().max() <= 2e-4
        assert (lse.cpu() - ref_l)[fin].abs().max() <= 1e-4


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("inf_keys", [64, 128])
def test_f32_first_step_of_minus_infinity(D, inf_keys):
    """fp32: a first step of 64 keys (and a whole first block) whose scores overflow to -inf weighs
    nothing; rows without a finite score are NaN with an lse of -inf.  The keys are -3e38 in one
    channel, where the queries are 4 (an infinite key has no finite remainder to split).  Bars of
    test_f32_steps_edges."""
    q, k, v = _inputs(1, 2, 200, 300, D, torch.float32, seed=D)
    q[..., 0] = 4.0
    k[:, 0, :inf_keys, 0] = -3e38
    k[:, 1, :, 0] = -3e38
    mask = _random_mask(1, 2, 2, 3, 0.6, seed=9)
    ref_o, ref_l = torch_ref.dense_masked_attention(q, k, v, mask)
    assert torch.isfinite(ref_o[:, 0]).all() and torch.isnan(ref_o[:, 1]).all()
    out, lse = ops.block_sparse_attention(q, k, v, ops.block_sparse_plan(mask))
    assert torch.isnan(out[:, 1]).all() and (lse[:, 1] == -math.inf).all()
    assert (out.cpu() - ref_o)[:, 0].abs().max() <= 2e-4
    assert (lse.cpu() - ref_l)[:, 0].abs().max() <= 1e-4


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Nq,Nk,layout", [(1, 1, "bhsd"), (130, 129, "bshd"), (700, 1500, "bhsd"), (1029, 640, "bshd")])
def test_dense_forms(dtype, Nq, Nk, layout):
    """The plan-free dense kernel and the one that also returns the block-mass map: attention bars
    against the oracle, fp32 row sums (lse to 1e-4 + 1e-5 |lse|), the map at the pooling bar."""
    q, k, v = _inputs(2, 3, Nq, Nk, 128, dtype, seed=Nq + Nk, sink_keys=2, layout=layout)
    full = torch.ones(2, 3, -(-Nq // 128), -(-Nk // 128), dtype=torch.bool)
    out, lse = ops.dense_attention(q, k, v, return_lse=True)
    _check(out, lse, q, k, v, full.cuda())
    ref_l = torch_ref.dense_masked_attention(q, k, v, full)[1]
    assert ((lse.cpu() - ref_l).abs() <= 1e-4 + 1e-5 * ref_l.abs()).all()
    o2, mass = ops.dense_attention_mass(q, k, v)
    _check(o2, lse, q, k, v, full.cuda())
    ref = torch_ref.exact_block_mass(q, k)
    assert mass.shape == ref.shape and ((mass.cpu() - ref).abs() <= 1e-8 + 1e-5 * ref.abs()).all()


def test_dense_mass_reference_moves():
    # rising maxima, and first keys ~80 log2 units below the later ones: the row sums' unit
    # moves past its 2^64 limit and the earlier sums are rescaled
    g = torch.Generator().manual_seed(4)
    q = 0.5 + 0.1 * torch.randn(1, 2, 400, 128, generator=g)
    k = torch.randn(1, 2, 1500, 128, generator=g)
    k[:, :, :128] = -10.0
    k[:, :, 1200:] *= 3.0
    qq, kk = q.bfloat16().cuda(), k.bfloat16().cuda()
    out, mass = ops.dense_attention_mass(qq, kk, kk)
    ref = torch_ref.exact_block_mass(qq, kk)
    assert ((mass.cpu() - ref).abs() <= 1e-8 + 1e-5 * ref.abs()).all()
    _check(out, ops.dense_attention(qq, kk, kk, return_lse=True)[1], qq, kk, kk,
           torch.ones(1, 2, 4, 12, dtype=torch.bool).cuda())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Nq", [1, 130, 383])
def test_dense_mass_infinite_keys_and_ragged_rows(dtype, Nq):
    """Keys of -inf and a last q-block that is not full: the rows past the end add nothing to its map."""
    q, k, v = _inputs(1, 2, Nq, 500, 128, dtype, seed=Nq)
    q = q.abs() + 0.5
    k[:, :, 64:300] = -math.inf
    mass, ref = ops.dense_attention_mass(q, k, v)[1].cpu(), torch_ref.exact_block_mass(q, k)
    assert ((mass - ref).abs() <= 1e-8 + 1e-5 * ref.abs()).all()


def test_dense_mass_in_several_launches():
    # more heads than one launch's workspace holds (2 GiB of row sums): the heads at the seam
    # against the pooling kernel's own map
    B, H, N = 1, 13, 75600
    assert _lib.lib().sinkattn_dense_mass_workspace_bytes(B, H, N, N) < H * 591 * 591 * 512
    g = torch.Generator(device="cuda").manual_seed(0)
    q, k, v = (torch.randn(B, N, H, 128, device="cuda", dtype=torch.bfloat16, generator=g).transpose(1, 2)
               for _ in range(3))
    out, mass = ops.dense_attention_mass(q, k, v)
    for h in (0, 10, 11, 12):
        want = ops.block_mass_scores(q[:, h:h + 1], k[:, h:h + 1])
        assert ((mass[:, h:h + 1] - want).abs() <= 1e-8 + 1e-5 * want.abs()).all()
        assert torch.equal(out[:, h:h + 1, :256], ops.dense_attention_mass(q[:, h:h + 1, :256], k[:, h:h + 1],
                                                                           v[:, h:h + 1])[0])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D,Nq,Nk", [(128, 300, 417), (128, 33, 1000), (64, 300, 417), (32, 161, 97)])
def test_few_and_many_q_blocks(dtype, D, Nq, Nk):
    """The split kernel (few q-blocks) and the whole-q-block kernels (the same heads repeated over a
    batch past the line) on ragged lengths, an empty row and a quarter of a tile whose scores are
    all -inf: both at the attention bars, keys of -inf score without weight."""
    q, k, v = _inputs(1, 2, Nq, Nk, D, dtype, seed=D + Nq)
    q = q.abs()
    mask = _random_mask(1, 2, -(-Nq // 128), -(-Nk // 128), 0.6, seed=9, empty_rows=1 if Nq > 128 else 0)
    many = 300 // (2 * mask.shape[2]) + 1
    for inf_keys in (0, 32):
        kk = k.clone()
        kk[:, :, 32:32 + inf_keys] = -math.inf
        ref_o, ref_l = torch_ref.dense_masked_attention(q, kk, v, mask)
        fin = torch.isfinite(ref_l)
        for rep in (1, many):
            qr, kr, vr, mr = (t.expand(rep, -1, -1, -1) for t in (q, kk, v, mask.contiguous()))
            out, lse = ops.block_sparse_attention(qr, kr, vr, ops.block_sparse_plan(mr.contiguous()))
            err = (out[-1:].float().cpu() - ref_o).abs()
            assert err.max() <= MAX_ABS and err.mean() <= MEAN_ABS, (rep, inf_keys, err.max())
            assert torch.equal(torch.isfinite(lse[-1:].cpu()), fin)
            assert ((lse[-1:].cpu() - ref_l)[fin].abs() <= LSE_ABS + 1e-5 * ref_l[fin].abs()).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [32, 64, 128])
def test_first_tile_of_minus_infinity(dtype, D):
    """A first listed tile whose scores are all -inf weighs nothing, in the split kernel, the
    whole-q-block kernels, the overlapping-row kernel (broadcast keys) and the dense forms; rows
    whose every score is -inf are NaN (a softmax of them) with an lse of -inf, and 0 in the dense
    forms, as scaled_dot_product_attention gives."""
    q, k, v = _inputs(1, 2, 256, 417, D, dtype, seed=D)
    q = q.abs()
    k[:, 0, :128] = -math.inf
    k[:, 1] = -math.inf
    mask = _random_mask(1, 2, 2, 4, 0.6, seed=9)
    ref_o, ref_l = torch_ref.dense_masked_attention(q, k, v, mask)

    def close(out, lse):
        assert torch.isnan(out[:, 1]).all() and (lse[:, 1] == -math.inf).all()
        err = (out[:, 0].float().cpu() - ref_o[:, 0]).abs()
        assert err.max() <= MAX_ABS and err.mean() <= MEAN_ABS
        assert ((lse[:, 0].cpu() - ref_l[:, 0]).abs() <= LSE_ABS + 1e-5 * ref_l[:, 0].abs()).all()

    for rep in (1, 80):  # 4 and 320 q-blocks
        qr, kr, vr, mr = (t.expand(rep, -1, -1, -1) for t in (q, k, v, mask))
        out, lse = ops.block_sparse_attention(qr, kr, vr, ops.block_sparse_plan(mr.contiguous()))
        close(out[-1:], lse[-1:])
    if D < 128:
        inf = k[:, 1:, :1].expand(-1, 2, 417, -1)
        out, lse = ops.block_sparse_attention(q, inf, v[:, :, :1].expand(-1, -1, 417, -1), ops.block_sparse_plan(mask))
        assert torch.isnan(out).all() and (lse == -math.inf).all()
        return
    want = torch.nn.functional.scaled_dot_product_attention(q, k, v)
    full = torch_ref.dense_masked_attention(q[:, :1], k[:, :1], v[:, :1], torch.ones(1, 1, 2, 4, dtype=torch.bool))[0]
    for out in (ops.dense_attention(q, k, v)[0], ops.dense_attention_mass(q, k, v)[0]):
        assert torch.equal(out[:, 1], want[:, 1]) and not torch.isnan(want).any()
        err = (out[:, :1].float().cpu() - full).abs()
        assert err.max() <= MAX_ABS and err.mean() <= MEAN_ABS
    mass = ops.dense_attention_mass(q, k, v)[1]
    ref = torch_ref.exact_block_mass(q, k)
    assert torch.equal(torch.isnan(mass.cpu()), torch.isnan(ref)) and torch.isnan(ref[:, 1]).all()
    assert ((mass.cpu() - ref)[:, 0].abs() <= 1e-8 + 1e-5 * ref[:, 0].abs()).all()


@pytest.mark.parametrize("form,dtype,D,bar", [("sparse", torch.float16, 64, 5.2e-7), ("sparse", torch.bfloat16, 32, 5.2e-7),
                                              ("dense", torch.float16, 128, 5.2e-7), ("sparse", torch.float32, 128, 6.4e-7)])
def test_row_sums_of_long_rows(form, dtype, D, bar):
    """fp32 row sums of 32760 keys are taken in short chains (a tile's, then the tiles'): the spread of
    the fp32 lse around the 64-bit one.  Its own rounding is 2.8e-7 rms (values of 8 to 16 have an
    ulp of 9.5e-7), 256 additions of tile sums in each of four lanes 1.6e-7, the scores' and
    exponentials' roundings bring it to 4.4e-7 (fp32 operands, split in bf16 pairs, 5.9e-7); one chain
    over the row gave 6.2e-7 (7.0e-7)."""
    g = torch.Generator(device="cuda").manual_seed(0)
    H, N = 12, 32760
    q, k, v = (torch.randn(1, H, N, D, device="cuda", generator=g).to(dtype) for _ in range(3))
    if form == "dense":
        lse = ops.dense_attention(q, k, v, return_lse=True)[1]
    else:
        lse = ops.block_sparse_attention(q, k, v, ops.block_sparse_plan(torch.ones(1, H, 256, 256, dtype=torch.bool, device="cuda")))[1]
    d = torch.cat([lse[0, h, :1024].double()
                   - torch.logsumexp(q[0, h, :1024].double() @ k[0, h].double().t().contiguous() / D ** 0.5, -1) for h in range(4)])
    print(f"{form} {dtype} {D}: mean {d.mean():.2e} spread {d.std():.2e}", flush=True)
    assert abs(float(d.mean())) <= 1e-6 and float(d.std()) <= bar


def _whole_q_blocks(q, k, v, mask):
    """The heads repeated over a batch of more than 256 q-blocks, past which every 16-bit call takes the
    whole-q-block kernels: the outputs of its last entry."""
    rep = 256 // (q.shape[0] * q.shape[1] * mask.shape[2]) + 1
    B = q.shape[0]
    qr, kr, vr = (t.repeat(rep, 1, 1, 1) if B > 1 else t.expand(rep, -1, -1, -1) for t in (q, k, v))
    out, lse = ops.block_sparse_attention(qr, kr, vr, ops.block_sparse_plan(mask.repeat(rep, 1, 1, 1)))
    assert torch.equal(out[:B], out[-B:]) and torch.equal(lse[:B], lse[-B:])
    return out[-B:], lse[-B:]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("Nq,Nk,layout,empty", [(1, 1, "bhsd", 0), (1, 300, "bshd", 0), (31, 129, "bshd", 0), (130, 1, "bhsd", 0),
                                                (257, 1000, "bshd", 1), (690, 690, "bshd", 2), (900, 129, "bhsd", 1)])
def test_whole_q_block_kernels_edges(dtype, D, Nq, Nk, layout, empty):
    """The shapes and layouts of the tests above (single rows and keys, ragged last blocks on both sides,
    rows without a listed block), whose few q-blocks run the split kernel, on the whole-q-block
    kernels.  Head dims 64 and 32 sum fp32 exponentials: their lse is held to 1e-4 + 1e-5 |lse|."""
    q, k, v = _inputs(1, 2, Nq, Nk, D, dtype, seed=Nq * 1000 + Nk, sink_keys=1, layout=layout)
    mask = _random_mask(1, 2, -(-Nq // 128), -(-Nk // 128), 0.4, seed=Nk, empty_rows=empty)
    out, lse = _whole_q_blocks(q, k, v, mask)
    _check(out, lse, q, k, v, mask)
    if D < 128:
        ref_l = torch_ref.dense_masked_attention(q, k, v, mask)[1]
        fin = torch.isfinite(ref_l)
        assert ((lse.cpu() - ref_l)[fin].abs() <= 1e-4 + 1e-5 * ref_l[fin].abs()).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("step", [7.5, 30.0, -12.0])
def test_whole_q_block_running_maximum(dtype, D, step):
    """test_running_maximum_moves_across_tiles on the whole-q-block kernels: maxima that rise slowly
    (the reference at head dim 128 lags them by up to 8 log2 units), fast, or fall."""
    N = 1024
    g = torch.Generator().manual_seed(21)
    q, k, v = (torch.randn(1, 2, N, D, generator=g) * f for f in (0.5, 0.5, 1.0))
    q[..., 0] = 1.0
    offs = torch.arange(N) // 128 * step
    k[..., 0] = ((offs - offs.min()) / (D ** -0.5 * 1.4426950408889634)).round()
    q, k, v = (x.to("cuda", dtype) for x in (q, k, v))
    mask = _random_mask(1, 2, 8, 8, 0.7, seed=5)
    out, lse = _whole_q_blocks(q, k, v, mask)
    _check(out, lse, q, k, v, mask)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("D,B,N", [(128, 1, 300), (128, 60, 300), (64, 1, 300), (64, 100, 300), (32, 2, 129)])
def test_lse_in_the_operands_type(dtype, D, B, N):
    """The kernels' rounded lse is the fp32 lse cast to the type, bit for bit, rows without a
    listed key (+inf) included, in every 16-bit kernel (few and many q-blocks, overlapping rows)."""
    q, k, v = _inputs(1, 2, N, N, D, dtype, seed=D + B)
    nb = -(-N // 128)
    mask = _random_mask(B, 2, nb, nb, 0.6, seed=9, empty_rows=1)
    plan = ops.block_sparse_plan(mask)
    q, k, v = (t.expand(B, -1, -1, -1) for t in (q, k, v))
    forms = [(k, v)] + ([(k[:, :, :1].expand(-1, -1, N, -1),) * 2] if D < 128 else [])
    for kk, vv in forms:
        full = ops.block_sparse_attention(q, kk, vv, plan)[1]
        own = ops.block_sparse_attention(q, kk, vv, plan, lse_in_dtype=True)[1]
        assert own.dtype == dtype and torch.equal(own, full.to(dtype)) and bool(torch.isinf(own).any())


def _chunk_layout(nbh, nqb):
    """Chunking of the launch order: heads [0, nbh_w) in Cw chunks (qb mod Cw), the heads
    of the partial last round of 8 in Cs = Cw * F finer chunks."""
    from math import gcd
    Cw = max(1, nqb // 128)
    rem = (nbh * Cw) % 8
    nsplit = 0 if rem == 0 else -(-rem // Cw)
    F = 8 // gcd(nsplit * Cw, 8)
    while F > 1 and Cw * F > nqb:
        F //= 2
    Cs = Cw * F
    nbh_w = nbh - nsplit
    return dict(nbh_w=nbh_w, Cw=Cw, Sw=-(-nqb // Cw), Cs=Cs, Ss=-(-nqb // Cs),
                nw=nbh_w * Cw, ns=nsplit * Cs)


MAX_OUTLIERS = 1024  # q-blocks taken out of the chunk sequences, in the whole plan
QBLOCK_COST = 2      # fixed cost of a q-block in the launch-order model, in tiles


def _check_order(plan, counts, nbh, nqb):
    """Launch-order invariants: a permutation of the rows; slot i runs on XCD i % 8; every
    chunk (q-blocks qb = j mod C of one head) on one XCD, at most ceil(n / 8) chunks of each
    kind (whole, fine) per XCD; each XCD's slots hold, from slot 0: its outliers (cost =
    tiles + QBLOCK_COST above twice the XCD's mean; none when the plan has more than MAX_OUTLIERS) by
    cost desc, then its fine chunks, then its whole chunks (each kind in ascending chunk
    order), each chunk's other q-blocks by cost desc; LPT keeps the XCD loads within one
    chunk's cost."""
    L = _chunk_layout(nbh, nqb)
    cap_w, cap_s = -(-L["nw"] // 8), -(-L["ns"] // 8)
    slots = (cap_w * L["Sw"] + cap_s * L["Ss"]) * 8
    # the launch slots, then the plan's chunk table (32 + 2 ints per chunk)
    assert plan.order.numel() == slots + 32 + 2 * (L["nw"] + L["ns"])
    order = plan.order.cpu().tolist()[:slots]
    rows = nbh * nqb
    real = sorted(r for r in order if r >= 0)
    assert real == list(range(rows))

    def chunk_of(r):
        bh, qb = divmod(r, nqb)
        if bh < L["nbh_w"]:
            return bh * L["Cw"] + qb % L["Cw"]
        return L["nw"] + (bh - L["nbh_w"]) * L["Cs"] + qb % L["Cs"]

    cost = [int(counts[r]) + QBLOCK_COST for r in range(rows)]
    chunk_xcd = {}
    for i, r in enumerate(order):
        if r >= 0:
            assert chunk_xcd.setdefault(chunk_of(r), i % 8) == i % 8
    mine_of = [[r for r in range(rows) if chunk_xcd[chunk_of(r)] == x] for x in range(8)]
    sums = [sum(cost[r] for r in m) for m in mine_of]
    outliers = [[r for r in m if cost[r] * len(m) > 2 * sums[x]] for x, m in enumerate(mine_of)]
    if sum(len(o) for o in outliers) > MAX_OUTLIERS:
        outliers = [[] for _ in range(8)]
    load = [0] * 8
    for x in range(8):
        mine = mine_of[x]
        load[x] = sums[x]
        chs = sorted({chunk_of(r) for r in mine})
        assert len([c for c in chs if c < L["nw"]]) <= cap_w
        assert len([c for c in chs if c >= L["nw"]]) <= cap_s
        if not mine:
            assert all(order[k * 8 + x] == -1 for k in range(len(order) // 8))
            continue
        out = set(outliers[x])
        want = sorted(out, key=lambda r: (-cost[r], r))
        for ch in [c for c in chs if c >= L["nw"]] + [c for c in chs if c < L["nw"]]:
            rest = [r for r in mine if chunk_of(r) == ch and r not in out]
            want += sorted(rest, key=lambda r: (-cost[r], r))
        got = [order[k * 8 + x] for k in range(len(order) // 8)]
        assert got[: len(want)] == want
        assert all(r == -1 for r in got[len(want):])
    chunk_cost = {}
    for r in range(rows):
        chunk_cost[chunk_of(r)] = chunk_cost.get(chunk_of(r), 0) + cost[r]
    nch = L["nw"] + L["ns"]
    busy = [l for l in load if l > 0]
    assert max(busy) - min(load if nch >= 8 else busy) <= max(chunk_cost.values())


@pytest.mark.parametrize("B,H,nqb,nkb,density", [(2, 3, 7, 9, 0.35), (1, 5, 300, 40, 0.3), (2, 12, 256, 256, 0.2),
                                                 (1, 30, 132, 132, 0.15), (1, 3, 2, 2, 0.5),
                                                 (2, 40, 210, 64, 0.2)])
def test_plan_lists_and_order(B, H, nqb, nkb, density):
    mask = _random_mask(B, H, nqb, nkb, density, seed=12, diag=False, col0=False, empty_rows=1)
    plan = ops.block_sparse_plan(mask)
    counts = plan.counts.cpu()
    idx = plan.idx.cpu().view(-1, nkb)
    flat = mask.cpu().view(-1, nkb)
    for r in range(flat.shape[0]):
        want = torch.nonzero(flat[r]).flatten().to(torch.int32)
        assert counts[r].item() == want.numel()
        assert torch.equal(idx[r, : want.numel()], want)
    _check_order(plan, counts, B * H, nqb)


@pytest.mark.parametrize("B,H,nqb,full,density", [(1, 30, 132, 0.03, 0.15), (2, 12, 256, 0.1, 0.05),
                                                  (2, 12, 256, 0.4, 0.0), (1, 5, 300, 0.02, 0.1),
                                                  (2, 40, 210, 0.02, 0.1)])
def test_plan_order_long_rows_first(B, H, nqb, full, density):
    # Masks with a share of fully dense q-block rows (the text rows of Z-Image's joint
    # sequence, the prefix rows of the coverage mask): those rows lead their XCD's sequence,
    # unless the plan holds more than MAX_OUTLIERS of them (the 40% case).  The last case
    # has more q-blocks (16800) than the ordering kernel stages in LDS.
    g = torch.Generator().manual_seed(50)
    m = torch.rand(B, H, nqb, nqb, generator=g) < density
    m[torch.rand(B, H, nqb, generator=g) < full] = True
    plan = ops.block_sparse_plan(m.cuda())
    _check_order(plan, plan.counts.cpu(), B * H, nqb)


def test_plan_order_large_costs():
    # 32768 dense q-blocks of 8192 key blocks: the chunk costs add up past 2^28, where the
    # launch-order pass picks each chunk's XCD by a scalar scan instead of the packed
    # (load * 8 + XCD) minimum; the order keeps every invariant.
    mask = torch.ones(1, 128, 256, 8192, dtype=torch.bool, device="cuda")
    plan = ops.block_sparse_plan(mask)
    counts = plan.counts.cpu()
    assert int(counts.sum()) + 2 * counts.numel() >= 1 << 28
    assert bool((counts == 8192).all())
    del mask
    _check_order(plan, counts, 128, 256)


def test_plan_order_many_heads_interleaved():
    # More than 4096 chunks (here 4100 heads of 20 q-blocks): the plan falls back to the
    # interleaved order.  Slot (bh * S + k) * 8 + x (S = ceil(nqb / 8)) holds the k-th
    # q-block of head bh with qb = x mod 8, by tile count desc then qb asc, -1 past the end;
    # the forward over that order matches the oracle on sampled heads.
    B, H, nqb, D = 1, 4100, 20, 128
    N = nqb * 128
    g = torch.Generator(device="cuda").manual_seed(60)
    q, k, v = (torch.randn(B, H, N, D, device="cuda", dtype=torch.bfloat16, generator=g) for _ in range(3))
    mask = _random_mask(B, H, nqb, nqb, 0.3, seed=61)
    plan = ops.block_sparse_plan(mask)
    S = -(-nqb // 8)
    assert plan.order.numel() == B * H * S * 8
    order = plan.order.cpu().view(B * H, S, 8)
    counts = plan.counts.cpu().view(B * H, nqb)
    want = torch.full((B * H, S, 8), -1, dtype=torch.int32)
    for x in range(8):
        qbs = torch.arange(x, nqb, 8)
        c = counts[:, qbs]  # [heads, n]
        # by count desc, then qb asc: sort on count * nqb + (nqb - 1 - qb), descending
        key = c * nqb + (nqb - 1 - qbs).unsqueeze(0)
        rank = torch.argsort(key, dim=1, descending=True)
        rows = torch.arange(B * H).unsqueeze(1) * nqb + qbs[rank]
        want[:, : qbs.numel(), x] = rows.to(torch.int32)
    assert torch.equal(order, want)
    out, lse = ops.block_sparse_attention(q, k, v, plan)
    torch.cuda.synchronize()
    heads = torch.tensor([0, 1, 2047, 4096, 4099])
    sub = lambda t: t[:, heads.cuda()]  # noqa: E731
    _check(sub(out), sub(lse), sub(q), sub(k), sub(v), sub(mask))


def test_bad_mask_shape_raises():
    q, k, v = _inputs(1, 2, 256, 256, 128, torch.bfloat16, seed=1)
    with pytest.raises(ValueError):
        sa._block_sparse_attn(q, k, v, torch.ones(1, 2, 3, 2, dtype=torch.bool, device="cuda"))


@pytest.mark.slow
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_wan_config2_full_size_rows_subsampled(dtype):
    # BASELINE config 2 at full size: B=2, H=12, N=32760 (last block 120), bf16 (and f16),
    # sinks at frame-0 positions, 20% seeded mask + diagonal + column 0.  The oracle
    # evaluates 48 rows per (b, h) spread over the sequence, including the ragged last block.
    B, H, N = 2, 12, 32760
    q, k, v = _inputs(B, H, N, N, 128, dtype, seed=20)
    g = torch.Generator().manual_seed(21)
    sinks = torch.randint(0, 1560, (8,), generator=g)
    k[:, :, sinks.cuda()] *= 6.0
    mask = _random_mask(B, H, 256, 256, 0.2, seed=22)
    out, lse = sa._block_sparse_attn(q, k, v, mask)
    torch.cuda.synchronize()
    rows = torch.cat([torch.randperm(N - 120, generator=g)[:40], torch.arange(N - 8, N)]).sort().values
    _check(out, lse[..., 0], q, k, v, mask, rows=rows)
    # the kernel's own fp32 lse (the drop-in rounds it to q.dtype)
    _, lse32 = ops.block_sparse_attention(q, k, v, ops.PLAN_CACHE.get(mask))
    torch.cuda.synchronize()
    _check(out, lse32, q, k, v, mask, rows=rows)


@pytest.mark.slow
def test_zimage_config4_full_size_rows_subsampled():
    # B=1, H=30, N=16896 (16384 image + 512 text tokens), bf16, the last
    # 512 keys x4; mask [1, 30, 132, 132] with the required prefix rows/cols 0-3 (what the
    # coverage builder adds for text_length=512), the diagonal and a seeded 15% remainder.
    B, H, N = 1, 30, 16896
    q, k, v = _inputs(B, H, N, N, 128, torch.bfloat16, seed=30)
    k[:, :, N - 512:] *= 4.0
    mask = _random_mask(B, H, 132, 132, 0.15, seed=31)
    mask[..., :4] = True
    mask[..., :4, :] = True
    out, lse = sa._block_sparse_attn(q, k, v, mask)
    torch.cuda.synchronize()
    g = torch.Generator().manual_seed(32)
    rows = torch.cat([torch.arange(0, 8), torch.randperm(N, generator=g)[:40], torch.arange(N - 8, N)])
    _check(out, lse[..., 0], q, k, v, mask, rows=rows.unique())


@pytest.mark.slow
def test_config5_mixed_head_densities_rows_subsampled():
    # BASELINE config 5 shape: C2-sized calls with per-head densities drawn from [5%, 60%]
    # and one fully dense head; the launch order balances such heads across XCDs.
    B, H, N = 2, 12, 32760
    q, k, v = _inputs(B, H, N, N, 128, torch.bfloat16, seed=40)
    g = torch.Generator().manual_seed(41)
    dens = 0.05 + 0.55 * torch.rand(H, generator=g)
    m = torch.rand(B, H, 256, 256, generator=g) < dens.view(1, H, 1, 1)
    m[:, 5] = True
    d = torch.arange(256)
    m[:, :, d, d] = True
    mask = m.cuda()
    plan = ops.block_sparse_plan(mask)
    _check_order(plan, plan.counts.cpu(), B * H, 256)
    out, lse = ops.block_sparse_attention(q, k, v, plan)
    torch.cuda.synchronize()
    rows = torch.cat([torch.randperm(N - 120, generator=g)[:24], torch.arange(N - 4, N)]).sort().values
    _check(out, lse, q, k, v, mask, rows=rows)
