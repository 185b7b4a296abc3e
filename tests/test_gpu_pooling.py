"""GPU parity of the block-score kernels.

exact mode  vs oracle/torch_ref.exact_block_mass (fp32 restatement of
            sparse_attention.py:145-227): elementwise rtol 1e-5 (atol 1e-8); rows of the
            map sum to 1.
max mode    vs oracle/torch_ref.max_pool_map (the reference's four rounding points in
            q.dtype, pinned bit for bit against the reference kernel's own outputs in
            tests/test_golden_max_pool.py): `parity_bars.max_pool_bar`, i.e. entries within
            the factor 2^ulp(max |R|) plus two ulps of q.dtype, at most 0.2% of the entries
            beyond a 2-ulp ripple and 8% of the rows touched, each such entry explained by
            a row near a rounding boundary (q.k is summed in another order on the matrix
            cores than on the CPU).
mean mode   vs oracle/torch_ref.mean_pool_scores: rtol 1e-5.
"""
import math
import threading

import pytest
import torch

from oracle import torch_ref
from parity_bars import max_block_logit, max_pool_bar
from sinkattn_amd import ops
from sinkattn_amd import sparse_attention as sa

pytestmark = pytest.mark.gpu

RTOL, ATOL = 1e-5, 1e-8


def _qk(B, H, Nq, Nk, dtype, seed, sinks=0, sink_scale=8.0, sink_at_end=False):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(B, H, Nq, 128, generator=g)
    k = torch.randn(B, H, Nk, 128, generator=g)
    if sinks:
        if sink_at_end:
            k[:, :, -sinks:] *= sink_scale
        else:
            k[:, :, :sinks] *= sink_scale
    return q.to(dtype), k.to(dtype)


def _max_pool_close(ours, ref, q, k, sm, block=128, causal=False, what=""):
    max_pool_bar(ours, ref, max_block_logit(q, k, sm, block, causal), what, qk=(q, k, sm, block, causal))


def _close(ours, ref):
    ours = ours.cpu().double()
    ref = ref.cpu().double()
    bad = ~((ours - ref).abs() <= ATOL + RTOL * ref.abs())  # a NaN is bad
    assert not bad.any(), f"{bad.sum().item()} elements, max rel {((ours - ref).abs() / ref.abs().clamp_min(1e-30)).max().item():.3g}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("N", [384, 1000])
def test_exact_mass_small(dtype, N):
    q, k = _qk(1, 2, N, N, dtype, seed=N, sinks=4)
    ours = ops.block_mass_scores(q.cuda(), k.cuda())
    ref = torch_ref.exact_block_mass(q, k)
    _close(ours, ref)
    assert torch.allclose(ours.sum(-1).cpu(), torch.ones(1, 2, ours.shape[2]), atol=1e-5)


def test_exact_mass_config1_fp32():
    # [1,12,4096,128] fp32 with 4 sink keys scaled 8x -> [1,12,32,32]
    q, k = _qk(1, 12, 4096, 4096, torch.float32, seed=0, sinks=4)
    cfg = sa.SinkSparseConfig(pooling_mode="exact")
    ours = sa._compute_block_scores(q.cuda(), k.cuda(), k.cuda(), cfg)
    assert ours.shape == (1, 12, 32, 32) and ours.dtype == torch.float32
    ref = torch_ref.exact_block_mass(q, k)
    _close(ours, ref)


def test_exact_mass_rescale_path_sinks_last():
    # the running maximum keeps rising (sinks at the end, growing key norms): exercises
    # the per-row rescaling of earlier key-block sums
    g = torch.Generator().manual_seed(3)
    q = torch.randn(1, 2, 512, 128, generator=g)
    k = torch.randn(1, 2, 1500, 128, generator=g) * torch.linspace(0.2, 3.0, 1500).view(1, 1, -1, 1)
    for dt in (torch.bfloat16, torch.float32):
        qq, kk = q.to(dt), k.to(dt)
        _close(ops.block_mass_scores(qq.cuda(), kk.cuda()), torch_ref.exact_block_mass(qq, kk))


# The matrix-core exact block-mass kernel at block sizes 16, 32 and 64 (16-bit inputs, head
# dim 128; smaller head dims are zero-padded to 128): q-blocks of KB rows inside 128-row
# items, key blocks of KB keys inside 128-key tiles, ragged ends on both sides, Nq != Nk.
@pytest.mark.parametrize("bs", [16, 32, 64])
@pytest.mark.parametrize("D,Nq,Nk,dtype", [(128, 1000, 1000, torch.bfloat16), (128, 333, 1111, torch.float16),
                                           (64, 520, 260, torch.bfloat16)])
def test_exact_mass_mfma_block_sizes(bs, D, Nq, Nk, dtype):
    q, k = _qkd(2, 3, 3, Nq, Nk, D, dtype, seed=bs + Nq, sinks=3)
    ours = ops.block_mass_scores(q.cuda(), k.cuda(), block_size=bs)
    ref = torch_ref.exact_block_mass(q, k, block_size=bs)
    assert ours.shape == ref.shape == (2, 3, math.ceil(Nq / bs), math.ceil(Nk / bs))
    _close(ours, ref)
    assert torch.allclose(ours.cpu().sum(-1), torch.ones(ref.shape[:-1]), atol=1e-5)


@pytest.mark.parametrize("bs", [16, 32, 64, 128])
def test_exact_mass_mfma_rescale_and_persistent_loop(bs):
    # 96 heads x 9 items of 128 rows: more items than resident work-groups, so slots are
    # reused.  q = 0.5 + 0.1 N(0,1) and the first 128 keys all -10: those scores are about
    # -640, ~80 log2 units below the N(0,1) keys after them, so the first tile's maximum
    # (the rows' reference point) sends every row through the 2^64 rescale of its earlier
    # key-block sums on the second tile (moderate scores elsewhere keep fp32 summation-order
    # differences below the 1e-5 bar)
    g = torch.Generator().manual_seed(bs)
    q = 0.5 + 0.1 * torch.randn(1, 96, 1100, 128, generator=g)
    k = torch.randn(1, 96, 1500, 128, generator=g)
    k[:, :, :128] = -10.0
    qq, kk = q.bfloat16(), k.bfloat16()
    ours = ops.block_mass_scores(qq.cuda(), kk.cuda(), block_size=bs)
    ref = torch_ref.exact_block_mass(qq, kk, block_size=bs)
    _close(ours, ref)
    assert float(ours[..., : 128 // bs].sum(-1).max()) < 1e-20   # the first tile holds no mass


def test_exact_mass_closed_forms():
    # Q = 0: uniform softmax -> mass = |kb| / N (last block 120 of 32760 -> 120/N)
    N = 1016  # 7 full blocks + 120
    q = torch.zeros(1, 1, 256, 128, dtype=torch.bfloat16)
    k = torch.randn(1, 1, N, 128).to(torch.bfloat16)
    m = ops.block_mass_scores(q.cuda(), k.cuda()).cpu()
    want = torch.tensor([128.0] * 7 + [120.0]) / N
    assert torch.allclose(m[0, 0], want.expand(2, -1), rtol=1e-5, atol=0)
    # one dominant key: all the mass in its block
    k2 = torch.zeros(1, 1, N, 128)
    k2[0, 0, 300] = 50.0
    q2 = torch.ones(1, 1, 256, 128)
    m2 = ops.block_mass_scores(q2.cuda().bfloat16(), k2.cuda().bfloat16()).cpu()
    assert torch.allclose(m2[0, 0, :, 2], torch.ones(2), atol=1e-6)


def test_exact_mass_vs_fp64():
    q, k = _qk(2, 2, 700, 900, torch.bfloat16, seed=4, sinks=3)
    ours = ops.block_mass_scores(q.cuda(), k.cuda()).cpu().double()
    ref = torch_ref.exact_block_mass_fp64(q, k)
    assert ((ours - ref).abs() <= 2e-5 * ref.abs() + 1e-9).all()


@pytest.mark.slow
def test_exact_mass_wan_shape_one_head():
    # Wan config 2/3 shape per (b, h): N = 32760 (ragged 120), bf16 -> [256, 256]
    q, k = _qk(1, 1, 32760, 32760, torch.bfloat16, seed=5, sinks=16)
    ours = ops.block_mass_scores(q.cuda(), k.cuda()).cpu()
    assert ours.shape == (1, 1, 256, 256)
    assert torch.allclose(ours.sum(-1), torch.ones(1, 1, 256), atol=2e-5)
    rows = [0, 1, 97, 255]
    ref = torch_ref.exact_block_mass(q[:, :, [r * 128 + i for r in rows for i in range(128 if r < 255 else 120)]], k)
    # ref rows are the selected q-blocks in order
    _close(ours[:, :, rows], ref)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("causal", [False, True])
def test_max_pool_vs_closed_form(dtype, causal):
    q, k = _qk(1, 4, 1024, 1024, dtype, seed=7, sinks=2)
    sm = 1.0 / math.sqrt(128)
    ours = ops.max_pool_scores(q.cuda(), k.cuda(), sm, causal=causal).cpu()
    ref = torch_ref.max_pool_map(q, k, sm, causal=causal)
    assert ours.dtype == dtype
    _max_pool_close(ours, ref, q, k, sm, causal=causal)
    # the unrounded formula agrees up to the reference's own rounding of the log2-domain
    # block maxima to q.dtype (|R| ~ 40 -> bf16 ulp 0.25 -> up to 2^0.125 in the ratio)
    ex = torch_ref.max_pool_map(q, k, sm, causal=causal, exact=True)
    assert torch.allclose(ours.double(), ex, rtol=0.2, atol=1e-3)


def test_max_pool_persistent_loop_ragged():
    # 96 heads x 9 query blocks = 864 items: more than one item per resident work-group,
    # so the workspace slot of a group is reused; N = 1100 leaves a ragged last block.
    q, k = _qk(1, 96, 1100, 1100, torch.bfloat16, seed=12, sinks=3)
    sm = 1.0 / math.sqrt(128)
    for causal in (False, True):
        ours = ops.max_pool_scores(q.cuda(), k.cuda(), sm, causal=causal).cpu()
        ref = torch_ref.max_pool_map(q, k, sm, causal=causal)
        _max_pool_close(ours, ref, q, k, sm, causal=causal, what=f"causal={causal}")


@pytest.mark.parametrize("bs", [16, 32, 64])
def test_max_pool_small_blocks_persistent_loop_ragged(bs):
    # the matrix-core max-pool kernel at blocks 16-64: 96 heads x 9 items of 128 rows (more
    # than one item per resident work-group), N = 1100 (ragged last block), causal and not
    q, k = _qk(1, 96, 1100, 1100, torch.bfloat16, seed=40 + bs, sinks=3)
    sm = 1.0 / math.sqrt(128)
    for causal in (False, True):
        ours = ops.max_pool_scores(q.cuda(), k.cuda(), sm, block_size=bs, causal=causal).cpu()
        ref = torch_ref.max_pool_map(q, k, sm, block_size=bs, causal=causal)
        _max_pool_close(ours, ref, q, k, sm, bs, causal, what=f"bs={bs} causal={causal}")


def test_max_pool_many_key_blocks():
    # N = 40000 -> 313 key blocks per row (ragged 64); three query blocks are checked
    # against the closed form.
    q, k = _qk(1, 1, 40000, 40000, torch.bfloat16, seed=13, sinks=8)
    assert ops.max_pool_scores(q.cuda(), k.cuda(), 0.088).shape == (1, 1, 313, 313)
    sel = [0, 150, 312]
    for causal in (False, True):
        ours = ops.max_pool_scores(q.cuda(), k.cuda(), 0.088, causal=causal).cpu()
        ref = torch_ref.max_pool_map(q, k, 0.088, causal=causal, query_blocks=sel)
        rows = [r * 128 + i for r in sel for i in range(128) if r * 128 + i < 40000]
        max_pool_bar(ours[:, :, sel], ref, max_block_logit(q, k, 0.088, 128, causal, rows=rows),
                     what=f"causal={causal}", qk=(q, k, 0.088, 128, causal, sel))


def test_attn_with_pooling_api_and_gqa():
    from sinkattention.pooling_kernel import attn_with_pooling
    q, _ = _qk(1, 4, 512, 512, torch.bfloat16, seed=8)
    _, k = _qk(1, 2, 512, 512, torch.bfloat16, seed=9)
    o, po = attn_with_pooling(q.cuda(), k.cuda(), k.cuda(), False, 0.088, 128)
    assert o.shape == q.shape and not o.any()
    ref = torch_ref.max_pool_map(q, k, 0.088)
    _max_pool_close(po, ref, q, k, 0.088)


def _qkd(B, H, Hk, Nq, Nk, D, dtype, seed, sinks=0):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(B, H, Nq, D, generator=g)
    k = torch.randn(B, Hk, Nk, D, generator=g)
    if sinks:
        k[:, :, :sinks] *= 6.0
    return q.to(dtype), k.to(dtype)


# Shapes off the block-128 / head-dim-128 MFMA kernels run on the generic kernels: block
# sizes that do not divide 128 or exceed it, head dims 16..256, ragged ends, Nq != Nk, fp32
# with more than 256 key blocks.
@pytest.mark.parametrize("D,bs,Nq,Nk,dtype", [
    (64, 64, 300, 300, torch.bfloat16), (128, 32, 260, 500, torch.bfloat16),
    (32, 96, 333, 250, torch.float16), (256, 16, 200, 130, torch.float32),
    (128, 256, 600, 600, torch.bfloat16), (80, 128, 300, 300, torch.bfloat16),
    (128, 128, 200, 33000, torch.float32), (16, 7, 50, 61, torch.bfloat16),
    (20, 64, 300, 280, torch.bfloat16), (20, 50, 300, 280, torch.float32)])
def test_exact_mass_generic_shapes(D, bs, Nq, Nk, dtype):
    q, k = _qkd(1, 2, 2, Nq, Nk, D, dtype, seed=D + bs, sinks=3)
    ours = ops.block_mass_scores(q.cuda(), k.cuda(), block_size=bs)
    ref = torch_ref.exact_block_mass(q, k, block_size=bs)
    assert ours.shape == ref.shape
    _close(ours, ref)
    assert torch.allclose(ours.cpu().sum(-1), torch.ones(ref.shape[:-1]), atol=1e-5)


@pytest.mark.parametrize("D,bs,N,dtype,causal", [
    (64, 64, 500, torch.bfloat16, False), (64, 32, 333, torch.float16, True),
    (256, 16, 200, torch.bfloat16, False), (32, 128, 400, torch.float32, False),
    (128, 64, 1000, torch.bfloat16, True), (16, 16, 100, torch.bfloat16, False)])
def test_max_pool_generic_shapes(D, bs, N, dtype, causal):
    q, k = _qkd(1, 4, 2, N, N, D, dtype, seed=D * 7 + bs, sinks=2)  # GQA: 4 query heads, 2 kv
    sm = 1.0 / math.sqrt(D)
    ours = ops.max_pool_scores(q.cuda(), k.cuda(), sm, block_size=bs, causal=causal).cpu()
    ref = torch_ref.max_pool_map(q, k, sm, block_size=bs, causal=causal)
    assert ours.dtype == dtype and ours.shape == ref.shape
    if dtype == torch.float32:
        assert torch.allclose(ours, ref, rtol=1e-5, atol=1e-12)
    else:
        _max_pool_close(ours, ref, q, k, sm, bs, causal, what=f"D={D} bs={bs}")


def test_attn_with_pooling_block_64_head_dim_64():
    from sinkattention.pooling_kernel import attn_with_pooling
    q, k = _qkd(2, 3, 3, 640, 640, 64, torch.bfloat16, seed=21)
    o, po = attn_with_pooling(q.cuda(), k.cuda(), k.cuda(), False, 0.125, 64)
    assert o.shape == q.shape and not o.any() and po.shape == (2, 3, 10, 10)
    _max_pool_close(po, torch_ref.max_pool_map(q, k, 0.125, block_size=64), q, k, 0.125, 64)


@pytest.mark.parametrize("bs,D", [(64, 64), (200, 128), (16, 32), (64, 20)])
def test_mean_mode_generic_block(bs, D):
    q, k = _qkd(1, 2, 2, 700, 500, D, torch.bfloat16, seed=bs)
    ours = ops.mean_pool_scores(q.cuda(), k.cuda(), block_size=bs).cpu()
    ref = torch_ref.mean_pool_scores(q, k, block_size=bs)
    assert torch.allclose(ours, ref, rtol=1e-5, atol=1e-7)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_mean_mode(dtype):
    q, k = _qk(2, 3, 1000, 700, dtype, seed=10)
    cfg = sa.SinkSparseConfig(pooling_mode="mean")
    ours = sa._compute_block_scores(q.cuda(), k.cuda(), k.cuda(), cfg).cpu()
    ref = torch_ref.mean_pool_scores(q, k)
    assert torch.allclose(ours, ref, rtol=1e-5, atol=1e-7)


def test_pooling_mode_dispatch():
    q, k = _qk(1, 2, 256, 256, torch.bfloat16, seed=11)
    qc, kc = q.cuda(), k.cuda()
    with pytest.raises(ValueError):
        sa._compute_block_scores(qc, kc, kc, sa.SinkSparseConfig(pooling_mode="bogus"))
    t = sa._compute_block_scores(qc, kc, kc, sa.SinkSparseConfig(pooling_mode="triton"))
    assert t.dtype == torch.float32 and t.shape == (1, 2, 2, 2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bs,H,Nq,Nk", [(128, 2, 1, 2048), (128, 3, 300, 2049), (64, 2, 1100, 4200), (32, 1, 130, 2500),
                                        (16, 1, 257, 2300), (128, 85, 1200, 2100)])
def test_exact_mass_key_ranges(dtype, bs, H, Nq, Nk):
    """Items of a partial round split over key ranges: one to eight ranges, ragged ends, a round of
    items plus a few (85 heads of 10), scores that rise past 2^64 in a later range, and a first
    range whose scores are all -inf (no reference there).  The pooling bar of 1e-5."""
    g = torch.Generator().manual_seed(bs + Nk)
    # five sigma above 0, and positive: a negative channel times -inf is +inf, whose row is NaN
    q = (0.5 + 0.1 * torch.randn(1, H, Nq, 128, generator=g)).abs()
    k = torch.randn(1, H, Nk, 128, generator=g)
    for low in (None, -10.0, -math.inf):
        kk = k.clone()
        if low is not None:
            kk[:, :, : Nk // 2] = low
        qd, kd = q.to(dtype), kk.to(dtype)
        ours = ops.block_mass_scores(qd.cuda(), kd.cuda(), block_size=bs)
        heads = [0, H - 1]
        _close(ours[:, heads], torch_ref.exact_block_mass(qd[:, heads], kd[:, heads], block_size=bs))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("bs", [16, 32, 64, 128])
@pytest.mark.parametrize("H,B", [(2, 1), (4, 200)])
def test_exact_mass_first_tile_of_minus_infinity(dtype, bs, H, B):
    """A first tile (32 keys in fp32, 128 in 16 bits) whose scores are all -inf weighs nothing, in calls
    of few items and of more than a round of them (the last batch entry is compared); rows without
    a finite score are NaN, as the oracle's.  The pooling bar of 1e-5."""
    g = torch.Generator().manual_seed(bs)
    q = torch.randn(1, H, 128, 128, generator=g)
    k = torch.randn(1, H, 400, 128, generator=g)
    q[..., 0] = 4.0
    low = -3e38 if dtype == torch.float32 else -math.inf
    k[:, 0, :32 if dtype == torch.float32 else 128, 0] = low
    k[:, 1, :, 0] = low
    q, k = q.to(dtype), k.to(dtype)
    ref = torch_ref.exact_block_mass(q, k, block_size=bs)
    ours = ops.block_mass_scores(q.cuda().expand(B, -1, -1, -1), k.cuda().expand(B, -1, -1, -1), block_size=bs).cpu()[-1:]
    assert torch.isnan(ref[:, 1]).all() and torch.isnan(ours[:, 1]).all()
    rest = [h for h in range(H) if h != 1]
    assert ((ours - ref)[:, rest].abs() <= ATOL + RTOL * ref[:, rest].abs()).all()


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bs,N", [(128, 3073), (128, 3300), (64, 3100), (32, 3201), (16, 3075)])
def test_max_pool_key_ranges(dtype, bs, N, causal):
    """Few items split over key ranges: the map of the whole-item kernel bit for bit (the same
    heads repeated over a batch past the line; the tests above hold that kernel to its bar), on
    ragged lengths, causal too."""
    q, k = _qkd(1, 4, 2, N, N, 128, dtype, seed=bs + N, sinks=2)
    qc, kc = q.cuda(), k.cuda()
    few = ops.max_pool_scores(qc, kc, 0.0883, block_size=bs, causal=causal)
    rep = 600 // (4 * (-(-N // 128))) + 1
    many = ops.max_pool_scores(qc.expand(rep, -1, -1, -1), kc.expand(rep, -1, -1, -1), 0.0883, block_size=bs,
                               causal=causal)
    assert torch.equal(few, many[:1]) and torch.equal(few, many[-1:])


# The fp32 matrix-core kernels (head dim 128, blocks 16-128): items of 64 rows (two to a
# 128-row block), tiles of 32 keys (two blocks of 16 each), the last key counts whose row values
# fit LDS (511 key blocks, all 160 KB of it) and the first that take the generic kernel, keys
# whose rows overlap, and the 2^64 rescale.  Bar: the pooling bar of 1e-5 relative (fp32 products
# and sums on both sides).
@pytest.mark.parametrize("bs,Nq,Nk", [(128, 1, 1), (128, 193, 127), (128, 64, 500), (64, 65, 33), (64, 130, 2000),
                                      (32, 63, 31), (32, 300, 257), (16, 79, 49), (16, 90, 7830), (16, 90, 8161),
                                      (16, 90, 8176), (16, 90, 8177)])
def test_exact_mass_f32_tile_edges(bs, Nq, Nk):
    g = torch.Generator().manual_seed(bs + Nq)
    q = torch.randn(2, Nq, 3, 128, generator=g).transpose(1, 2)
    k = torch.randn(2, Nk, 3, 128, generator=g).transpose(1, 2)
    k[:, :, : Nk // 3] -= 4.0 * (Nq % 2)
    _close(ops.block_mass_scores(q.cuda(), k.cuda(), block_size=bs), torch_ref.exact_block_mass(q, k, block_size=bs))
    ke = k[:, :, :1].expand(-1, -1, Nk, -1)
    _close(ops.block_mass_scores(q.cuda(), k.cuda()[:, :, :1].expand(-1, -1, Nk, -1), block_size=bs),
           torch_ref.exact_block_mass(q, ke.contiguous(), block_size=bs))


@pytest.mark.parametrize("bs", [16, 32, 64, 128])
def test_exact_mass_f32_rescale(bs):
    g = torch.Generator().manual_seed(bs)
    q = 0.5 + 0.1 * torch.randn(1, 2, 200, 128, generator=g)
    k = torch.randn(1, 2, 500, 128, generator=g)
    k[:, :, :128] = -10.0  # ~80 log2 units below the keys after them
    ours = ops.block_mass_scores(q.cuda(), k.cuda(), block_size=bs)
    _close(ours, torch_ref.exact_block_mass(q, k, block_size=bs))
    assert float(ours[..., : 128 // bs].sum(-1).max()) < 1e-20


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("bs,H,Hk,N", [(128, 2, 2, 1), (128, 4, 2, 321), (64, 2, 1, 190), (32, 2, 2, 333),
                                       (16, 4, 4, 259), (16, 1, 1, 7800), (16, 1, 1, 8165), (16, 1, 1, 8176),
                                       (16, 1, 1, 8177)])
def test_max_pool_f32_tile_edges(bs, H, Hk, N, causal):
    """exp2 of fp32 scores of 128 products each: the fp32 bar below, as on the generic kernel.  A negative
    scale too: a block's raw maximum is scaled, and the row's reference is the largest of those."""
    q, k = _qkd(1, H, Hk, N, N, 128, torch.float32, seed=bs + N)
    for sm in (1.0 / 128 ** 0.5, -0.05)[: 2 if N <= 511 * bs else 1]:  # the generic kernel's scale is positive
        ours = ops.max_pool_scores(q.cuda(), k.cuda(), sm, block_size=bs, causal=causal).cpu()
        ref = torch_ref.max_pool_map(q, k, sm, block_size=bs, causal=causal)
        assert torch.allclose(ours, ref, rtol=2e-5, atol=1e-8), sm


@pytest.mark.parametrize("B,H,Nq,Nk,bs,D", [(1, 1, 1, 1, 128, 128), (1, 2, 17 * 16 + 1, 33, 16, 128),
                                            (2, 1, 40, 600, 1, 64), (1, 1, 300, 1030, 2, 256),
                                            (1, 2, 5000, 2600, 1024, 48), (1, 1, 65, 64, 4, 8)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_mean_mode_tile_edges(B, H, Nq, Nk, bs, D, dtype):
    """Remainders of the 16-row score tiles, rows past the 512 key blocks kept in registers, head
    dims that end inside a 16-byte chunk or a quarter, strided operands.  Bound: fp32 sums of
    at most 1024 rows and 256 products, each within 1024 * 2^-24 relative of its terms."""
    g = torch.Generator().manual_seed(bs + D)
    q = torch.randn(B, Nq, H, D, generator=g).to(dtype).permute(0, 2, 1, 3)
    k = torch.randn(B, Nk, H, D, generator=g).to(dtype).permute(0, 2, 1, 3)
    ours = ops.mean_pool_scores(q.cuda(), k.cuda(), block_size=bs).cpu()
    ref = torch_ref.mean_pool_scores(q, k, block_size=bs)
    assert ours.shape == ref.shape
    assert torch.allclose(ours, ref, rtol=2e-5, atol=1e-7)


def test_pooling_lds_from_two_threads():
    """Host threads whose calls need different amounts of LDS (the fp32 and the generic kernels past
    64 KB): the limit a kernel may launch with is one per process, and both get theirs."""
    g = torch.Generator(device="cuda").manual_seed(3)

    def call(fn, N, D):
        q, k = (torch.randn(1, 1, N, D, device="cuda", generator=g) for _ in range(2))
        return lambda: fn(q, k)

    def mass(q, k):
        return ops.block_mass_scores(q, k, block_size=16)

    def most(q, k):
        return ops.max_pool_scores(q, k, 0.09, block_size=16)

    for fn, D, sizes in ((mass, 128, (2400, 7000)), (most, 128, (2400, 7000)), (mass, 64, (640, 9000)), (most, 64, (640, 9000))):
        calls = [call(fn, N, D) for N in sizes]
        want = [c() for c in calls]
        bad = []

        def work(i):
            with torch.cuda.stream(torch.cuda.Stream()):
                try:
                    for _ in range(40):
                        got = calls[i]()
                    torch.cuda.current_stream().synchronize()
                    if not torch.allclose(got, want[i], rtol=1e-5, atol=1e-8):
                        bad.append(f"{sizes[i]}: other values")
                except Exception as e:  # a launch past the limit another thread set
                    bad.append(f"{sizes[i]}: {e}")

        torch.cuda.synchronize()
        threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not bad, bad
