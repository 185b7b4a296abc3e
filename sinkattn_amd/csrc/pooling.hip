// Block-score ("pooling") kernels for gfx950.
//
// block_mass_pool: the reference's exact mode, `_compute_exact_block_mass_scores`
//   (sinkattention/sparse_attention.py:145-227), in one pass over K with no N x N
//   intermediate.  A work-group owns one q-block (128 rows) at a time.  For every key tile
//   it computes S^T with the matrix cores and turns each row's scores into exp2 terms
//   relative to a per-row reference maximum.
//   * bf16/f16 (block_mass_persistent_kernel): persistent groups; the per-(row, key-block)
//     sums go to the group's slot ws[kb][row] of a global workspace.  The reference maximum
//     is the row maximum of the first tile and moves only when a tile's sum exceeds 2^64
//     (kSumLimit); then the row's earlier sums are rescaled.
//   * fp32 (block_mass_f32_kernel): one group per 64 query rows; the sums stay in LDS, the
//     reference maximum as above.
//   At the end every row is normalised by its own total and the rows are averaged per key
//   block.
//
// max_pool: `attn_with_pooling` (sinkattention/pooling_kernel.py:11-248) without the
//   [B,H,N,nd] scratch: the per-(row, key-block) maxima of the rows in flight go to the
//   group's slot ws[kb][row] of a global workspace (max_pool_persistent_kernel).
//
// mean_pool: `_compute_pooled_qk_block_scores`' mean branch
//   (sinkattention/sparse_attention.py:79-94,138-142).

#include "common.h"
#include "kernels.h"
#include "tile.h"

namespace sa {

// ------------------------------------------------------------------------------------
// Exact block mass, 16-bit inputs, head dim 128, block size KB in {16, 32, 64, 128};
// persistent work-groups (up to 3 per CU).
// Each work-group walks items of 128 query rows (128 / KB q-blocks of the map); per item it
// streams every 128-key K tile into LDS by buffer DMA (rows >= Nk read as zero and are
// masked), computes S^T for its 128 rows with the matrix cores and writes each row's sum
// of exp2(scale*log2e*s - m_ref) over every KB-key block of the tile to its private
// workspace slot ws[kb][row] (kb in KB units).  m_ref is the row maximum of the first tile;
// it only moves (and the row's earlier sums are rescaled) if a tile's sum overflows 2^64,
// i.e. when scores rise more than ~64 log2 units above it.  The item's epilogue normalises
// every row by its total and averages the rows of each q-block per key block.
// Key of register j of a lane of 32-key group t, within the group: tile_key(hl, j) =
// (j & 3) + 4 ((j >> 2) & 1) + 8 hl + 16 (j >> 3), so the KB-key block of (t, j) does not
// depend on the lane: t / (KB / 32) for KB >= 32, 2 t + (j >> 3) for KB = 16 (the lane pair
// holds its two 8-key halves).
// ------------------------------------------------------------------------------------
constexpr float kSumLimit = 1.8446744073709552e19f;  // 2^64

// A row's normalisation: 1 / total, NaN without a finite score (a total of 0).
__device__ __forceinline__ float row_factor(float total) {
  return total == 0.f ? __builtin_nanf("") : 1.f / fmaxf(total, 1e-6f);
}

template <int KB>
__device__ __forceinline__ constexpr int sub_block(int t, int j) {
  return KB == 16 ? 2 * t + (j >> 3) : (t * 32) / KB;
}

// The tiles [t0, t1) of one item: each row's block sums into ws[kb][row], its reference maximum
// and the sum of all of them in m_ref and l_tot (the same in both lanes of a row).  RANGED (t0 may
// be past the first tile): a row whose scores are all -inf so far has no reference and takes it
// from the first tile that has one.
template <int CT, int KB, bool RANGED>
__device__ __forceinline__ void mass_tiles(const PoolArgs& a, SA_LDS char* lk, int item, int t0, int t1, float* ws,
                                           float& m_ref, float& l_tot) {
  constexpr int DS = 8;
  constexpr int NS = 128 / KB;  // key blocks per 128-key tile, q-blocks per 128-row item
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hl = lane >> 5, l32 = lane & 31;
  const int nkb = a.nkb;               // key blocks of the map (KB keys each)
  const int nqi = (a.Nq + 127) >> 7;   // 128-row items per head
  const uint32_t kstride = (uint32_t)a.ks[2] * 2;
  const int drow = 4 * wave + (lane >> 4);
  const uint32_t k_off = (uint32_t)drow * kstride + (uint32_t)(((lane & 15) ^ (drow & 15)) * 16);
  const int prow = k_row_perm(l32);
  uint32_t ka[DS];
#pragma unroll
  for (int ds = 0; ds < DS; ++ds) ka[ds] = (uint32_t)(prow * 256 + (((2 * ds + hl) ^ (prow & 15)) * 16));
  const float c = a.scale * kLog2e;
  const int r = wave * 32 + l32;
  const int bh = item / nqi;
  const int qi = item - bh * nqi;
  const int b = bh / a.H, h = bh - b * a.H;
  const char* qbase = (const char*)a.q + ((int64_t)b * a.qs[0] + (int64_t)h * a.qs[1]) * 2;
  const char* kbase = (const char*)a.k + ((int64_t)b * a.ks[0] + (int64_t)h * a.ks[1]) * 2;
  const int qrow = qi * 128 + r;
  u32x4 qf[DS];
  // rows past the end repeat the last one: their factor is 0, and 0 times what zeros would make of
  // an infinite key is NaN
  load_q_operand<128>(qf, qbase, a.qs[2], min(qrow, a.Nq - 1), a.Nq, hl);
  m_ref = neg_inf();
  l_tot = 0.f;

  for (int kt = t0; kt < t1; ++kt) {
    const int key0 = kt * 128;
    __syncthreads();  // the previous tile (or item epilogue) is done with lds_k
    {
      const __amdgpu_buffer_rsrc_t rs =
          make_rsrc(kbase + (int64_t)key0 * kstride, (uint32_t)(a.Nk - key0) * kstride);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        dma16(rs, (SA_LDS void*)(lk + (256 * j + 64 * wave) * 16), k_off + (uint32_t)j * 16u * kstride);
    }
    __syncthreads();  // waits for this group's DMA
    f32x16 s[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) s[t] = f32x16{};
#pragma unroll
    for (int ds = 0; ds < DS; ++ds)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const u32x4 av = *(SA_LDS const u32x4*)(lk + ka[ds] + t * 8192);
        s[t] = mfma32x32x16<CT>(av, qf[ds], s[t]);
      }
    if (key0 + 128 > a.Nk) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int j = 0; j < 16; ++j)
          if (key0 + t * 32 + tile_key(hl, j) >= a.Nk) s[t][j] = neg_inf();
    }
    if (RANGED ? __any(m_ref == neg_inf()) : kt == 0) {  // reference maximum from the first tile
      // (the lowest float when its scores are all -inf: a later tile's sum then passes the limit)
      float mx = neg_inf();
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int j = 0; j < 16; ++j) mx = fmaxf(mx, s[t][j]);
      mx = max_xor32(mx) * c;
      m_ref = RANGED ? (m_ref != neg_inf() ? m_ref : mx) : fmaxf(mx, lowest());
    }
    float ps[NS];
    auto sums = [&]() {
      const float ref = RANGED && m_ref == neg_inf() ? 0.f : m_ref;
#pragma unroll
      for (int i = 0; i < NS; ++i) ps[i] = 0.f;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int j = 0; j < 16; ++j) ps[sub_block<KB>(t, j)] += fast_exp2(__builtin_fmaf(s[t][j], c, -ref));
#pragma unroll
      for (int i = 0; i < NS; ++i) ps[i] = sum_xor32(ps[i]);
    };
    sums();
    float tot = 0.f;
#pragma unroll
    for (int i = 0; i < NS; ++i) tot += ps[i];
    if (!(tot <= kSumLimit)) {
      // Rare: scores far above m_ref.  Move m_ref to this tile's maximum and rescale
      // the row's earlier sums (the two lanes of the row split them by parity).
      float mx = neg_inf();
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int j = 0; j < 16; ++j) mx = fmaxf(mx, s[t][j]);
      mx = max_xor32(mx) * c;
      const float f = fast_exp2(m_ref - mx);
      for (int j = t0 * NS + hl; j < kt * NS; j += 2) ws[j * 128 + r] *= f;
      l_tot *= f;
      m_ref = mx;
      sums();
      tot = 0.f;
#pragma unroll
      for (int i = 0; i < NS; ++i) tot += ps[i];
    }
    l_tot += tot;
    // the lanes of a row split the stores: lane half hl stores key blocks i = hl (mod 2)
#pragma unroll
    for (int i = 0; i < NS; ++i)
      if ((NS == 1 ? hl == 0 : (i & 1) == hl) && kt * NS + i < nkb) ws[(kt * NS + i) * 128 + r] = ps[i];
  }
}

template <int CT, int KB>
__global__ __launch_bounds__(256, 3) void block_mass_persistent_kernel(PoolArgs a, int items) {
  constexpr int NS = 128 / KB;
  __shared__ u32x4 lds_k[2048];
  __shared__ float row_inv[128];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hl = lane >> 5, l32 = lane & 31;
  const int nkb = a.nkb;
  const int ntiles = (a.Nk + 127) >> 7;  // 128-key tiles
  const int nqi = (a.Nq + 127) >> 7;
  float* ws = a.ws + (size_t)blockIdx.x * (size_t)nkb * 128;
  const int r = wave * 32 + l32;

  for (int item = blockIdx.x; item < items; item += gridDim.x) {
    const int bh = item / nqi;
    const int qi = item - bh * nqi;
    const int qrow = qi * 128 + r;
    float m_ref, l_tot;
    mass_tiles<CT, KB, false>(a, (SA_LDS char*)lds_k, item, 0, ntiles, ws, m_ref, l_tot);

    // Epilogue: out[qb][kb] = mean over the q-block's rows of ws[kb][row] / total(row); lane l
    // holds rows l and l + 64, so a q-block of KB rows is one group of KB lanes (KB < 64) or
    // a whole half (KB = 64) or both halves (KB = 128).
    if (hl == 0) row_inv[r] = (qrow < a.Nq) ? row_factor(l_tot) : 0.f;
    __syncthreads();
    const float inv0 = row_inv[lane], inv1 = row_inv[lane + 64];
    const __amdgpu_buffer_rsrc_t wrs = make_rsrc(ws, (uint32_t)nkb * 512u);
    float* out = reinterpret_cast<float*>(a.out);
    for (int kb = wave; kb < nkb; kb += 4) {
      // coherent (L1-bypassing) loads of values other waves of the group wrote
      const float x0 = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(wrs, (uint32_t)(kb * 512 + lane * 4), 0, 1));
      const float x1 = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(wrs, (uint32_t)(kb * 512 + lane * 4 + 256), 0, 1));
      float v0 = x0 * inv0, v1 = x1 * inv1;
      if constexpr (KB == 128) {
        v0 += v1;
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) v0 += __shfl_xor(v0, off, 64);
      } else {
#pragma unroll
        for (int off = (KB >= 64 ? 32 : KB / 2); off >= 1; off >>= 1) {
          v0 += __shfl_xor(v0, off, 64);
          v1 += __shfl_xor(v1, off, 64);
        }
      }
      if (lane % (KB >= 64 ? 64 : KB) == 0) {
        const int g = lane / (KB >= 64 ? 64 : KB);  // q-block of the first half
#pragma unroll
        for (int half = 0; half < (KB == 128 ? 1 : 2); ++half) {
          const int qs = half * (NS / 2 > 0 ? NS / 2 : 1) + g;  // q-block within the item
          const int qb = qi * NS + qs;
          const int rows = min(KB, a.Nq - qb * KB);
          if (qb < a.nqb && rows > 0)
            out[((int64_t)bh * a.nqb + qb) * nkb + kb] = (half == 0 ? v0 : v1) / (float)rows;
        }
      }
    }
  }
}

// The items of a partial round (all of them when they are fewer than the resident groups), whose
// groups would leave the others idle: S groups per item, each a range of its key tiles.  Group
// (item i, range s) writes its block sums to item i's slot and every row's reference and sum to
// ml[i][s][2][128]; block_mass_combine_kernel puts the ranges together.
// bf16, blocks of 128: [1,12,2048,128] 36 -> 26 us, [1,12,4096,128] 80 -> 64, [1,1,16000,128]
// 239 -> 84, [1,7,16000,128] (875 items) 593 -> 514.
template <int CT, int KB>
__global__ __launch_bounds__(256, 3) void block_mass_ranged_kernel(PoolArgs a, int first, int n, int S, float* ml) {
  __shared__ u32x4 lds_k[2048];
  const int i = (int)blockIdx.x % n, s = (int)blockIdx.x / n;
  const int ntiles = (a.Nk + 127) >> 7;
  float m_ref, l_tot;
  mass_tiles<CT, KB, true>(a, (SA_LDS char*)lds_k, first + i, s * ntiles / S, (s + 1) * ntiles / S,
                           a.ws + (size_t)i * (size_t)a.nkb * 128, m_ref, l_tot);
  const int lane = threadIdx.x & 63, r = (threadIdx.x >> 6) * 32 + (lane & 31);
  if (lane < 32) {
    float* p = ml + ((size_t)i * S + s) * 256;
    p[r] = m_ref;
    p[128 + r] = l_tot;
  }
}

constexpr int kMassMaxRanges = 8;

// Group (item, slice of the key blocks): the map entries of the item from its ranges' sums.
template <int KB>
__global__ __launch_bounds__(256) void block_mass_combine_kernel(PoolArgs a, int first, int S, const float* ml) {
  constexpr int NS = 128 / KB, G = KB >= 64 ? 64 : KB;
  __shared__ float f[kMassMaxRanges][128];  // range s, row: 2^(m_s - m) / total
  const int i = blockIdx.x, item = first + i;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nkb = a.nkb, ntiles = (a.Nk + 127) >> 7, nqi = (a.Nq + 127) >> 7;
  const int bh = item / nqi, qi = item - bh * nqi;
  const float* p = ml + (size_t)i * S * 256;
  if (tid < 128) {
    float m = neg_inf(), l = 0.f;
    for (int s = 0; s < S; ++s) m = fmaxf(m, p[s * 256 + tid]);
    for (int s = 0; s < S; ++s) {
      const float ms = p[s * 256 + tid];
      const float e = ms == neg_inf() ? 0.f : fast_exp2(ms - m);
      f[s][tid] = e;
      l += p[s * 256 + 128 + tid] * e;
    }
    // a row without a finite score: 0 / 0, as in one range
    const float inv = qi * 128 + tid >= a.Nq ? 0.f : (m == neg_inf() ? __builtin_nanf("") : 1.f / fmaxf(l, 1e-6f));
    for (int s = 0; s < S; ++s) f[s][tid] = inv == 0.f ? 0.f : f[s][tid] * inv;
  }
  __syncthreads();
  const float* ws = a.ws + (size_t)i * (size_t)nkb * 128;
  float* out = reinterpret_cast<float*>(a.out);
  for (int kb = blockIdx.y * 4 + wave; kb < nkb; kb += 4 * gridDim.y) {
    const int s = ((kb / NS + 1) * S - 1) / ntiles;  // the range that holds this block's tile
    float v0 = ws[(size_t)kb * 128 + lane] * f[s][lane], v1 = ws[(size_t)kb * 128 + 64 + lane] * f[s][lane + 64];
    if constexpr (KB == 128) {
      v0 += v1;
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) v0 += __shfl_xor(v0, off, 64);
    } else {
#pragma unroll
      for (int off = G / 2; off >= 1; off >>= 1) {
        v0 += __shfl_xor(v0, off, 64);
        v1 += __shfl_xor(v1, off, 64);
      }
    }
    if (lane % G == 0) {
#pragma unroll
      for (int half = 0; half < (KB == 128 ? 1 : 2); ++half) {
        const int qb = qi * NS + half * (NS / 2 > 0 ? NS / 2 : 1) + lane / G;
        const int rows = min(KB, a.Nq - qb * KB);
        if (qb < a.nqb && rows > 0)
          out[((int64_t)bh * a.nqb + qb) * nkb + kb] = (half == 0 ? v0 : v1) / (float)rows;
      }
    }
  }
}

// ------------------------------------------------------------------------------------
// Exact block mass, f32 inputs, head dim 128, block size KB in {16, 32, 64, 128}: fp32 matrix
// cores (v_mfma_f32_16x16x4_f32, fp32 products and sums).  Bound by the matrix cores, 256 flops
// per clock and CU in fp32.  An item is 64 query rows of one head, 16 per wave, so that a short
// sequence still gives every CU an equal share ([1,12,4096,128]: 768 items, three per CU, where
// items of 128 rows would load half the CUs twice).  K streams in tiles of 32 keys through two
// LDS buffers by DMA, the next tile's copies issued a whole tile ahead, one barrier per tile.
//     S^T[16 kt .. +16] = K Q^T   (A = 16 K rows from LDS, B = Q^T in VGPRs)
// Lane l holds query l % 16 and, of every 16 channels, the four from 4 (l / 16): one 16-byte
// read feeds four matrix instructions; its S^T registers hold keys 16 kt + 4 (l / 16) + i.  The
// 16-byte chunks of a K row are swizzled by row & 15, so a 16-lane read touches 256 distinct
// bytes.  A row's per-block sums of exp2(scale*log2e*s - m_ref) stay in LDS; m_ref is the row
// maximum of the first tile and moves (rescaling the earlier sums) only when a tile's sum passes
// 2^64.  [1,12,4096,128]: 0.45 ms,
// 115 TFLOP/s of the 153 a large fp32 matrix product reaches here (0.70 ms with 32-key tiles
// staged through registers behind two barriers); blocks of 64 at [2,10,6545,128] 2.0 ms (30.5 ms
// on the generic kernel's VALU dot products).
// XCD x (work-group i runs on XCD i % 8) takes the items [x, x + 1) * items_per_xcd, so that its
// L2 holds few heads' K at a time.  Blocks of 128 rows span two items, whose halves meet in an
// atomic add to the zeroed map (two addends: the sum does not depend on their order).
// ------------------------------------------------------------------------------------
constexpr int kF32Rows = 64;  // query rows of an item
constexpr int kF32Keys = 32;  // keys of a tile

__host__ __device__ inline int f32_sum_pitch(int nkb) { return nkb | 1; }  // floats: rows on distinct banks
constexpr size_t kF32StaticLds = 2 * kF32Keys * 512 + kF32Rows * 4;

// One item's view of the K stream: the copies of a tile and its scores.
struct F32Tiles {
  const char* kbase;
  uint32_t kstride, doff[2], ka;
  int Nk, wave;
  f32x4 qv[8];  // Q^T B operands: this lane's channels 16 j + 4 (l / 16) ..

  __device__ __forceinline__ F32Tiles(const PoolArgs& a, int b, int h, int hk, int qrow, int lane, int wave_)
      : Nk(a.Nk), wave(wave_) {
    const int g = lane >> 4, sl = lane & 15;
    kbase = (const char*)a.k + ((int64_t)b * a.ks[0] + (int64_t)hk * a.ks[1]) * 4;
    kstride = (uint32_t)a.ks[2] * 4;
    // Copy j (of 4) of wave w fills tile rows 8j + 2w + lane / 32; the swizzle of those rows
    // alternates with j.
    const int drow = 2 * wave + (lane >> 5);
    doff[0] = (uint32_t)drow * kstride + (uint32_t)(((lane & 31) ^ drow) * 16);
    doff[1] = (uint32_t)drow * kstride + (uint32_t)(((lane & 31) ^ (drow + 8)) * 16);
    ka = (uint32_t)(sl * 512 + ((g ^ sl) * 16));  // chunk 4 j + g: XOR 64 j
    // rows past the end repeat the last one (as in the 16-bit kernel)
    const float* q = (const float*)a.q +
                     ((int64_t)b * a.qs[0] + (int64_t)h * a.qs[1] + (int64_t)min(qrow, a.Nq - 1) * a.qs[2]);
#pragma unroll
    for (int j = 0; j < 8; ++j) qv[j] = *reinterpret_cast<const f32x4*>(q + 16 * j + 4 * g);
  }

  __device__ __forceinline__ void copy(SA_LDS char* dst, int t) const {
    const int key0 = t * kF32Keys;
    const int valid = min(kF32Keys, Nk - key0);
    // ends with the last valid row (rows may lie closer than 128 floats); keys past it are masked
    const __amdgpu_buffer_rsrc_t rs =
        make_rsrc(kbase + (int64_t)key0 * kstride, (uint32_t)(valid - 1) * kstride + 512u);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      dma16(rs, (SA_LDS void*)(dst + (4 * j + wave) * 1024), doff[j & 1] + (uint32_t)(8 * j) * kstride);
  }

  __device__ __forceinline__ void scores(SA_LDS const char* cur, f32x4 (&s)[2]) const {
    // four chains: the odd and even 16-channel steps apart (independent instructions, and half the
    // additions in a row)
    f32x4 acc[2][2] = {{f32x4{}, f32x4{}}, {f32x4{}, f32x4{}}};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      f32x4 kv[2];
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) kv[kt] = *(SA_LDS const f32x4*)(cur + (ka ^ (64u * j)) + kt * 8192);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
          acc[j & 1][kt] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[kt][e], qv[j][e], acc[j & 1][kt], 0, 0, 0);
    }
    s[0] = acc[0][0] + acc[1][0];
    s[1] = acc[0][1] + acc[1][1];
  }
};

template <int KB>
__global__ __launch_bounds__(256, 3) void block_mass_f32_kernel(PoolArgs a, int items, int items_per_xcd) {
  constexpr int TPB = KB > kF32Keys ? KB / kF32Keys : 1;  // tiles per key block
  constexpr int NS = KB < kF32Keys ? kF32Keys / KB : 1;   // key blocks per tile
  extern __shared__ float sums[];  // [64][f32_sum_pitch(nkb)]
  // each buffer its own variable: through one the compiler makes a tile's reads wait for the
  // next tile's copies
  __shared__ u32x4 lds_k0[kF32Keys * 32];
  __shared__ u32x4 lds_k1[kF32Keys * 32];
  __shared__ float row_inv[kF32Rows];
  const int item = (int)(blockIdx.x % kXcds) * items_per_xcd + (int)(blockIdx.x / kXcds);
  if (item >= items) return;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, sl = lane & 15;
  const int nkb = a.nkb, pitch = f32_sum_pitch(nkb);
  const int ntiles = (a.Nk + kF32Keys - 1) / kF32Keys;
  const int nqi = (a.Nq + kF32Rows - 1) / kF32Rows;
  const int bh = item / nqi, qi = item - bh * nqi;
  const int b = bh / a.H, h = bh - b * a.H;
  const int r = wave * 16 + sl;  // this lane's row of the item
  const int qrow = qi * kF32Rows + r;
  const F32Tiles tl(a, b, h, h, qrow, lane, wave);
  tl.copy((SA_LDS char*)lds_k0, 0);
  const float c = a.scale * kLog2e;
  float m_ref = 0.f, l_tot = 0.f, run = 0.f;
  float* my = sums + r * pitch;

  auto tile = [&](int t, SA_LDS char* cur, SA_LDS char* next) __attribute__((always_inline)) {
    drain_then_barrier();  // tile t has landed; every wave is done with the other buffer
    if (t + 1 < ntiles) tl.copy(next, t + 1);
    f32x4 s[2];
    tl.scores(cur, s);
    const int left = a.Nk - t * kF32Keys - 4 * g;  // key 16 kt + i of this lane exists when below it
    const bool cut = (t + 1) * kF32Keys > a.Nk;
    auto row_max = [&]() __attribute__((always_inline)) {
      float mx = neg_inf();
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (!cut || 16 * kt + i < left) mx = fmaxf(mx, s[kt][i] * c);
      return max_col16(mx);
    };
    // key 0 always exists; a first tile whose scores are all -inf leaves the lowest float, and the
    // first finite score's tile then passes the limit below
    if (t == 0) m_ref = fmaxf(row_max(), lowest());
    float ps[2];
    auto tile_sums = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        ps[kt] = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float e = fast_exp2(__builtin_fmaf(s[kt][i], c, -m_ref));
          ps[kt] += !cut || 16 * kt + i < left ? e : 0.f;
        }
        ps[kt] = sum_col16(ps[kt]);
      }
    };
    tile_sums();
    if (!(ps[0] + ps[1] <= kSumLimit)) {
      // Rare: scores far above m_ref.  Move m_ref to this tile's maximum and rescale the row's
      // earlier sums (the row's four lanes split them).
      const float mx = row_max();
      const float f = fast_exp2(m_ref - mx);
      for (int j = g; j < t * NS / TPB; j += 4) my[j] *= f;
      l_tot *= f;
      run *= f;
      m_ref = mx;
      tile_sums();
    }
    l_tot += ps[0] + ps[1];
    if constexpr (NS == 2) {
      if (g < 2 && 2 * t + g < nkb) my[2 * t + g] = g == 0 ? ps[0] : ps[1];
    } else {
      run += ps[0] + ps[1];
      if ((t + 1) % TPB == 0 || t + 1 == ntiles) {
        if (g == 0) my[t / TPB] = run;
        run = 0.f;
      }
    }
  };
  for (int t = 0; t < ntiles; t += 2) {
    tile(t, (SA_LDS char*)lds_k0, (SA_LDS char*)lds_k1);
    if (t + 1 < ntiles) tile(t + 1, (SA_LDS char*)lds_k1, (SA_LDS char*)lds_k0);
  }

  if (g == 0) row_inv[r] = qrow < a.Nq ? row_factor(l_tot) : 0.f;
  __syncthreads();
  // Map entries: the mean over a q-block's rows of sum / total.
  constexpr int RB = KB < kF32Rows ? KB : kF32Rows;  // rows of this item in one q-block
  float* out = reinterpret_cast<float*>(a.out);
  for (int qs = 0; qs < kF32Rows / RB; ++qs) {
    const int qb = (qi * kF32Rows + qs * RB) / KB;
    const int rows = min(KB, a.Nq - qb * KB);  // rows of the whole q-block
    if (qb >= a.nqb) break;
    for (int kb = tid; kb < nkb; kb += 256) {
      float acc = 0.f;
#pragma unroll 8
      for (int rr = 0; rr < RB; ++rr) acc += sums[(qs * RB + rr) * pitch + kb] * row_inv[qs * RB + rr];
      float* dst = out + ((int64_t)bh * a.nqb + qb) * nkb + kb;
      if constexpr (KB > kF32Rows) atomicAdd(dst, acc / (float)rows);
      else *dst = acc / (float)rows;
    }
  }
}

__global__ __launch_bounds__(256) void fill_zero_kernel(float* p, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) p[i] = 0.f;
}

// Whether the fp32 matrix-core kernels take a call: head dim 128, a block size they have, the
// values of an item's rows within the CU's LDS beside the K tiles (511 key blocks), a tile
// of K rows within a buffer's 32-bit offsets, and an item count within the grid.  Any other
// call runs the generic kernels (6-7 TFLOP/s against 100-125).
bool pool_f32_mfma(const PoolArgs& a) {
  return a.D == 128 && (a.bs == 16 || a.bs == 32 || a.bs == 64 || a.bs == 128) &&
         kF32StaticLds + (size_t)kF32Rows * f32_sum_pitch(a.nkb) * 4 <= kGenericPoolMaxLds &&
         a.ks[2] * 4 * kF32Keys < ((int64_t)1 << 31) &&
         (int64_t)a.B * a.H * (a.Nq / kF32Rows + 1) < ((int64_t)1 << 30);
}

// The kernel's dynamic LDS and, where two items share a map entry, the zeroed map.
static hipError_t f32_pool_setup(const void* kern, const PoolArgs& a, bool zero, size_t lds, hipStream_t stream) {
  if (kF32StaticLds + lds > 64 * 1024) {  // past what a launch gets without asking
    const hipError_t e = allow_all_lds(kern, kF32StaticLds);
    if (e != hipSuccess) return e;
  }
  if (!zero) return hipSuccess;
  const int64_t n = (int64_t)a.B * a.H * a.nqb * a.nkb;
  fill_zero_kernel<<<(int)min((int64_t)1024, (n + 255) / 256), 256, 0, stream>>>((float*)a.out, n);
  return hipGetLastError();
}

template <int KB>
static hipError_t launch_mass_f32(const PoolArgs& a, hipStream_t stream) {
  const int items = a.B * a.H * ((a.Nq + kF32Rows - 1) / kF32Rows);
  const int per = (items + kXcds - 1) / kXcds;
  const size_t lds = (size_t)kF32Rows * f32_sum_pitch(a.nkb) * 4;
  const hipError_t e =
      f32_pool_setup(reinterpret_cast<const void*>(block_mass_f32_kernel<KB>), a, KB > kF32Rows, lds, stream);
  if (e != hipSuccess) return e;
  block_mass_f32_kernel<KB><<<per * kXcds, 256, lds, stream>>>(a, items, per);
  return hipGetLastError();
}

// ------------------------------------------------------------------------------------
// Max-pool map, f32 inputs, head dim 128: the tiles and items of block_mass_f32_kernel with each
// row's block maxima R[r,kb] = max_j s * (sm_scale * log2e) in LDS (fp32, so the reference's
// rounding of R to q.dtype is the identity) and m_r the maximum of R over the row.  Po[qb,kb] =
// max over the block's rows of exp2(R - m_r); rows past the end take m = +inf, which gives 0.
// The maximum is taken over the bits (values >= 0, a NaN above them all), atomically into the
// zeroed map where a block of 128 rows spans two items; max_pool_f32_norm_kernel then divides
// each map row by its sum.  Causal: key blocks after the query block are not seen and raw scores
// above the diagonal of the diagonal block get -1e6.  [1,10,6545,128]: 1.00 ms at
// blocks of 128 and 1.04 at 64 (19.1 ms on the generic kernel).
// ------------------------------------------------------------------------------------
template <int KB>
__global__ __launch_bounds__(256, 3) void max_pool_f32_kernel(PoolArgs a, int items, int items_per_xcd) {
  constexpr int TPB = KB > kF32Keys ? KB / kF32Keys : 1;
  constexpr int NS = KB < kF32Keys ? kF32Keys / KB : 1;
  extern __shared__ float maxima[];  // [64][f32_sum_pitch(nkb)]
  __shared__ u32x4 lds_k0[kF32Keys * 32];
  __shared__ u32x4 lds_k1[kF32Keys * 32];
  __shared__ float row_m[kF32Rows];
  const int item = (int)(blockIdx.x % kXcds) * items_per_xcd + (int)(blockIdx.x / kXcds);
  if (item >= items) return;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, sl = lane & 15;
  const int nkb = a.nkb, pitch = f32_sum_pitch(nkb);
  const int nqi = (a.Nq + kF32Rows - 1) / kF32Rows;
  const int bh = item / nqi, qi = item - bh * nqi;
  const int b = bh / a.H, h = bh - b * a.H;
  const int r = wave * 16 + sl;
  const int qrow = qi * kF32Rows + r;
  const int qbr = qrow / KB;  // this row's q-block
  // keys any row of the item sees
  const int key_end = a.causal ? min(a.Nk, ((qi * kF32Rows + kF32Rows - 1) / KB + 1) * KB) : a.Nk;
  const int ntiles = (key_end + kF32Keys - 1) / kF32Keys;
  const F32Tiles tl(a, b, h, h / (a.H / a.Hk), qrow, lane, wave);
  tl.copy((SA_LDS char*)lds_k0, 0);
  // The reference forms qk_scale = fp32(sm_scale) * fp32(1.44269504).
  const float c = a.scale * 1.44269504f;
  float m = neg_inf(), run = neg_inf();
  float* my = maxima + r * pitch;

  auto tile = [&](int t, SA_LDS char* cur, SA_LDS char* next) __attribute__((always_inline)) {
    drain_then_barrier();  // tile t has landed; every wave is done with the other buffer
    if (t + 1 < ntiles) tl.copy(next, t + 1);
    f32x4 s[2];
    tl.scores(cur, s);
    const int key0 = t * kF32Keys;
    if ((t + 1) * kF32Keys > a.Nk || (a.causal && key0 + kF32Keys > qi * kF32Rows / KB * KB)) {
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = key0 + 16 * kt + 4 * g + i;
          if (a.causal) {
            if (key / KB == qbr && qrow < key) s[kt][i] += -1.0e6f;
            if (key / KB > qbr) s[kt][i] = neg_inf();
          }
          if (key >= a.Nk) s[kt][i] = neg_inf();
        }
    }
    float mx[2];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      mx[kt] = neg_inf();
#pragma unroll
      for (int i = 0; i < 4; ++i) mx[kt] = fmaxf(mx[kt], s[kt][i]);
      mx[kt] = max_col16(mx[kt]);
    }
    // a block's raw maximum first, then the scale; unseen blocks (raw maximum -inf) take no part in m
    auto block = [&](int kb, float raw, bool mine) __attribute__((always_inline)) {
      if (raw != neg_inf()) m = fmaxf(m, raw * c);
      if (mine) my[kb] = raw * c;
    };
    if constexpr (NS == 2) {
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
        if (2 * t + kt < nkb) block(2 * t + kt, mx[kt], g == kt);
    } else {
      run = fmaxf(run, fmaxf(mx[0], mx[1]));
      if ((t + 1) % TPB == 0 || t + 1 == ntiles) {
        block(t / TPB, run, g == 0);
        run = neg_inf();
      }
    }
  };
  for (int t = 0; t < ntiles; t += 2) {
    tile(t, (SA_LDS char*)lds_k0, (SA_LDS char*)lds_k1);
    if (t + 1 < ntiles) tile(t + 1, (SA_LDS char*)lds_k1, (SA_LDS char*)lds_k0);
  }

  if (g == 0) row_m[r] = qrow < a.Nq ? m : pos_inf();
  __syncthreads();
  constexpr int RB = KB < kF32Rows ? KB : kF32Rows;  // rows of this item in one q-block
  unsigned* out = reinterpret_cast<unsigned*>(a.out);
  for (int qs = 0; qs < kF32Rows / RB; ++qs) {
    const int qb = (qi * kF32Rows + qs * RB) / KB;
    if (qb >= a.nqb) break;
    const int kb_end = a.causal ? min(nkb, qb + 1) : nkb;
    for (int kb = tid; kb < kb_end; kb += 256) {
      unsigned v = 0u;
#pragma unroll 8
      for (int rr = 0; rr < RB; ++rr)
        v = max(v, __float_as_uint(fast_exp2(maxima[(qs * RB + rr) * pitch + kb] - row_m[qs * RB + rr])));
      unsigned* dst = out + ((int64_t)bh * a.nqb + qb) * nkb + kb;
      if constexpr (KB > kF32Rows) atomicMax(dst, v);
      else *dst = v;
    }
  }
}

// Map rows divided by their sums (one wave per row); entries past a causal row's end are 0.
__global__ __launch_bounds__(256) void max_pool_f32_norm_kernel(PoolArgs a) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= a.B * a.H * a.nqb) return;
  const int kb_end = a.causal ? min(a.nkb, row % a.nqb + 1) : a.nkb;
  float* p = reinterpret_cast<float*>(a.out) + (int64_t)row * a.nkb;
  float sum = 0.f;
  for (int kb = lane; kb < kb_end; kb += 64) sum += p[kb];
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) sum += __shfl_xor(sum, off, 64);
  for (int kb = lane; kb < a.nkb; kb += 64) p[kb] = kb < kb_end ? p[kb] / sum : 0.f;
}

template <int KB>
static hipError_t launch_max_f32(const PoolArgs& a, hipStream_t stream) {
  const int items = a.B * a.H * ((a.Nq + kF32Rows - 1) / kF32Rows);
  const int per = (items + kXcds - 1) / kXcds;
  const size_t lds = (size_t)kF32Rows * f32_sum_pitch(a.nkb) * 4;
  hipError_t e = f32_pool_setup(reinterpret_cast<const void*>(max_pool_f32_kernel<KB>), a, KB > kF32Rows, lds, stream);
  if (e != hipSuccess) return e;
  max_pool_f32_kernel<KB><<<per * kXcds, 256, lds, stream>>>(a, items, per);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  max_pool_f32_norm_kernel<<<(a.B * a.H * a.nqb + 3) / 4, 256, 0, stream>>>(a);
  return hipGetLastError();
}

// Rounding of an fp32 value to the 16-bit type CT (returned as fp32).
template <int CT>
__device__ __forceinline__ float round_to(float x);
template <>
__device__ __forceinline__ float round_to<kBF16>(float x) {
  return (float)(__bf16)x;
}
template <>
__device__ __forceinline__ float round_to<kF16>(float x) {
  return (float)(_Float16)x;
}

// The map rows of one item from its rows' block maxima and row maxima (row_m, complete for the
// group).
template <int CT, int KB>
__device__ __forceinline__ void max_pool_rows(const PoolArgs& a, int item, float* ws, float* cm, const float* row_m,
                                              float* colmax, float* total_sh) {
  constexpr int NS = 128 / KB;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nkb = a.nkb;
  const int nqi = (a.Nq + 127) >> 7;
  const int bh = item / nqi;
  const int qi = item - bh * nqi;
  const int kb_item = a.causal ? min(nkb, (qi + 1) * NS) : nkb;  // key blocks any row of the item sees
  const float m0 = row_m[lane], m1 = row_m[lane + 64];
  const __amdgpu_buffer_rsrc_t wrs = make_rsrc(ws, (uint32_t)nkb * 512u);
  if constexpr (KB == 128) {
    for (int kb = wave; kb < kb_item; kb += 4) {
      // coherent (L1-bypassing) loads of values other waves of the group wrote
      const float x0 = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(wrs, (uint32_t)(kb * 512 + lane * 4), 0, 1));
      const float x1 = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(wrs, (uint32_t)(kb * 512 + lane * 4 + 256), 0, 1));
      float v = fmaxf(fast_exp2(x0 - m0), fast_exp2(x1 - m1));
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
      if (lane == 0) colmax[kb] = round_to<CT>(v);
    }
    __syncthreads();
    // Row normalisation in q.dtype: sum (fp32 accumulate, rounded), then divide.
    if (wave == 0) {
      float part = 0.f;
      for (int kb = lane; kb < kb_item; kb += 64) part += colmax[kb];
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) part += __shfl_xor(part, off, 64);
      if (lane == 0) total_sh[0] = round_to<CT>(part);
    }
    __syncthreads();
    const float total = total_sh[0];
    uint16_t* out = reinterpret_cast<uint16_t*>(a.out) + ((int64_t)bh * a.nqb + qi) * nkb;
    for (int kb = tid; kb < nkb; kb += 256) {
      const float v = kb < kb_item ? colmax[kb] / total : 0.f;
      out[kb] = (uint16_t)(pack2<CT>(v, 0.f) & 0xffffu);
    }
  } else {
    // Pass 1: column maxima of every (q-block, key block) of the item into cm[qs][kb]:
    // lane l holds rows l and l + 64, so a q-block is a group of KB lanes (KB < 64) or a
    // whole half (KB = 64).
    constexpr int G = KB >= 64 ? 64 : KB;
    for (int kb = wave; kb < kb_item; kb += 4) {
      const float x0 = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(wrs, (uint32_t)(kb * 512 + lane * 4), 0, 1));
      const float x1 = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(wrs, (uint32_t)(kb * 512 + lane * 4 + 256), 0, 1));
      float v0 = fast_exp2(x0 - m0), v1 = fast_exp2(x1 - m1);
#pragma unroll
      for (int off = G / 2; off >= 1; off >>= 1) {
        v0 = fmaxf(v0, __shfl_xor(v0, off, 64));
        v1 = fmaxf(v1, __shfl_xor(v1, off, 64));
      }
      if (lane % G == 0) {
        const int g = lane / G;
        cm[(size_t)g * nkb + kb] = round_to<CT>(v0);
        cm[(size_t)(NS / 2 + g) * nkb + kb] = round_to<CT>(v1);
      }
    }
    __syncthreads();  // the column maxima are in memory (the barrier drains this group's stores)
    // Pass 2: per q-block (one wave each), the row total in q.dtype, then the division.
    const __amdgpu_buffer_rsrc_t crs = make_rsrc(cm, (uint32_t)(NS * nkb) * 4u);
    for (int qs = wave; qs < NS; qs += 4) {
      const int qb = qi * NS + qs;
      if (qb >= a.nqb) continue;
      const int kb_end = a.causal ? min(nkb, qb + 1) : nkb;
      float part = 0.f;
      for (int kb = lane; kb < kb_end; kb += 64)
        part += __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(crs, (uint32_t)((qs * nkb + kb) * 4), 0, 1));
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) part += __shfl_xor(part, off, 64);
      const float total = round_to<CT>(part);
      uint16_t* out = reinterpret_cast<uint16_t*>(a.out) + ((int64_t)bh * a.nqb + qb) * nkb;
      for (int kb = lane; kb < nkb; kb += 64) {
        const float cv = kb < kb_end ? __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                            crs, (uint32_t)((qs * nkb + kb) * 4), 0, 1))
                                     : 0.f;
        out[kb] = (uint16_t)(pack2<CT>(kb < kb_end ? cv / total : 0.f, 0.f) & 0xffffu);
      }
    }
  }
}

// ------------------------------------------------------------------------------------
// Max-pool map, persistent form (bf16/f16, head dim 128, block size KB in {16, 32, 64,
// 128}): the structure of block_mass_persistent_kernel (items of 128 query rows, K tiles of
// 128 keys by DMA, S^T on the matrix cores) with the block maxima of each row kept in the
// group's workspace slot ws[kb][row] instead of LDS, so four groups (33-37 KB of LDS, 128
// VGPRs each) fit a CU: per tile a group waits for its own copy, and the other three cover
// that wait.  Per tile: R[r,kb] = q.dtype(max_j s * sm_scale * log2e) for each KB-key block
// (raw-score maximum first, then the scale, as pooling_kernel.py:39-48 does), m_r = max
// over kb of the unrounded values.  Epilogue per q-block and kb: Po[kb] = q.dtype(max over
// the block's rows of exp2(R[r,kb] - m_r)), then the row is normalised in q.dtype
// (pooling_kernel.py:65-75, 243-244).  kv head = h / (H / Hk); causal restricts kb <= qb and
// adds -1e6 to the raw scores above the diagonal of the diagonal block.  Block 128 keeps
// the item's column maxima in LDS (nkb <= 1024); smaller blocks keep them after the
// group's slot, in (128 / KB) * nkb floats of the workspace.
// ------------------------------------------------------------------------------------
template <int CT, int KB>
__global__ __launch_bounds__(256, 4) void max_pool_persistent_kernel(PoolArgs a, int items) {
  constexpr int DS = 8;
  constexpr int NS = 128 / KB;  // key blocks per tile, q-blocks per item
  __shared__ u32x4 lds_k[2048];
  __shared__ float row_m[128];
  __shared__ float colmax[KB == 128 ? 1024 : 1];
  __shared__ float total_sh[KB == 128 ? 1 : 4];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hl = lane >> 5, l32 = lane & 31;
  const int nkb = a.nkb;
  const int ntiles = (a.Nk + 127) >> 7;
  const int nqi = (a.Nq + 127) >> 7;
  float* ws = a.ws + (size_t)blockIdx.x * (size_t)nkb * (128 + (KB == 128 ? 0 : NS));
  float* cm = ws + (size_t)nkb * 128;  // [NS][nkb] column maxima (KB < 128)
  const uint32_t kstride = (uint32_t)a.ks[2] * 2;
  const int drow = 4 * wave + (lane >> 4);
  const uint32_t k_off = (uint32_t)drow * kstride + (uint32_t)(((lane & 15) ^ (drow & 15)) * 16);
  const int prow = k_row_perm(l32);
  // chunk (2ds + hl) ^ (prow & 15) of row prow: the k-step only flips bits 5-7
  const uint32_t ka0 = (uint32_t)(prow * 256 + ((hl ^ (prow & 15)) * 16));
  SA_LDS char* lk = (SA_LDS char*)lds_k;
  // The reference forms qk_scale = fp32(sm_scale) * fp32(1.44269504).
  const float qk_scale = a.scale * 1.44269504f;
  const int r = wave * 32 + l32;

  for (int item = blockIdx.x; item < items; item += gridDim.x) {
    const int bh = item / nqi;
    const int qi = item - bh * nqi;
    const int b = bh / a.H, h = bh - b * a.H;
    const int hk = h / (a.H / a.Hk);
    const int kt_end = a.causal ? min(ntiles, qi + 1) : ntiles;
    const int kb_item = a.causal ? min(nkb, (qi + 1) * NS) : nkb;  // key blocks any row of the item sees
    const char* qbase = (const char*)a.q + ((int64_t)b * a.qs[0] + (int64_t)h * a.qs[1]) * 2;
    const char* kbase = (const char*)a.k + ((int64_t)b * a.ks[0] + (int64_t)hk * a.ks[1]) * 2;
    const int qrow = qi * 128 + r;
    const int qbr = qrow / KB;  // this row's q-block
    u32x4 qf[DS];
    load_q_operand<128>(qf, qbase, a.qs[2], qrow, a.Nq, hl);
    float m = neg_inf();

    for (int kt = 0; kt < kt_end; ++kt) {
      const int key0 = kt * 128;
      __syncthreads();  // the previous tile (or item epilogue) is done with lds_k
      {
        const __amdgpu_buffer_rsrc_t rs =
            make_rsrc(kbase + (int64_t)key0 * kstride, (uint32_t)(a.Nk - key0) * kstride);
#pragma unroll
        for (int j = 0; j < 8; ++j)
          dma16(rs, (SA_LDS void*)(lk + (256 * j + 64 * wave) * 16), k_off + (uint32_t)j * 16u * kstride);
      }
      __syncthreads();  // waits for this group's DMA
      f32x16 s[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) s[t] = f32x16{};
      {
        // Flat step i = 4 ds + t.  The read for step i + 2 is issued right after the MFMA
        // of step i (the scheduling groups pin that order), so each read has two MFMAs to
        // land; a deeper ring does not fit the 128 VGPRs of four groups per CU.
        u32x4 kr[4];
        auto kread = [&](int i) __attribute__((always_inline)) {
          return *(SA_LDS const u32x4*)(lk + (ka0 ^ (32u * (i >> 2))) + (i & 3) * 8192);
        };
        kr[0] = kread(0);
        kr[1] = kread(1);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
        for (int i = 0; i < 4 * DS; ++i) {
          s[i & 3] = mfma32x32x16<CT>(kr[i & 3], qf[i >> 2], s[i & 3]);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (i + 2 < 4 * DS) {
            kr[(i + 2) & 3] = kread(i + 2);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          }
        }
      }
      const bool diag = a.causal && kt == qi;
      if (key0 + 128 > a.Nk || diag) {
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int j = 0; j < 16; ++j) {
            const int key = key0 + t * 32 + tile_key(hl, j);
            if (diag) {
              const int kbk = key / KB;
              if (kbk == qbr && qrow < key) s[t][j] += -1.0e6f;
              if (kbk > qbr) s[t][j] = neg_inf();  // a key block past the row's own: not seen
            }
            if (key >= a.Nk) s[t][j] = neg_inf();
          }
      }
      float mx[NS];
#pragma unroll
      for (int i = 0; i < NS; ++i) mx[i] = neg_inf();
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int j = 0; j < 16; ++j) mx[sub_block<KB>(t, j)] = fmaxf(mx[sub_block<KB>(t, j)], s[t][j]);
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        mx[i] = max_xor32(mx[i]) * qk_scale;
        m = fmaxf(m, mx[i]);
        if ((NS == 1 ? hl == 0 : (i & 1) == hl) && kt * NS + i < nkb) ws[(kt * NS + i) * 128 + r] = round_to<CT>(mx[i]);
      }
    }

    // Rows past the end of the sequence take no part (m = +inf gives 0).
    if (hl == 0) row_m[r] = (qrow < a.Nq) ? m : pos_inf();
    __syncthreads();
    if constexpr (KB != 128) {
      max_pool_rows<CT, KB>(a, item, ws, cm, row_m, colmax, total_sh);
    } else {  // max_pool_rows' part for blocks of 128, here: as a call 0.3% slower at the Wan layer
      const float m0 = row_m[lane], m1 = row_m[lane + 64];
      const __amdgpu_buffer_rsrc_t wrs = make_rsrc(ws, (uint32_t)nkb * 512u);
      for (int kb = wave; kb < kb_item; kb += 4) {
        // coherent (L1-bypassing) loads of values other waves of the group wrote
        const float x0 = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(wrs, (uint32_t)(kb * 512 + lane * 4), 0, 1));
        const float x1 = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(wrs, (uint32_t)(kb * 512 + lane * 4 + 256), 0, 1));
        float v = fmaxf(fast_exp2(x0 - m0), fast_exp2(x1 - m1));
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
        if (lane == 0) colmax[kb] = round_to<CT>(v);
      }
      __syncthreads();
      // Row normalisation in q.dtype: sum (fp32 accumulate, rounded), then divide.
      if (wave == 0) {
        float part = 0.f;
        for (int kb = lane; kb < kb_item; kb += 64) part += colmax[kb];
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) part += __shfl_xor(part, off, 64);
        if (lane == 0) total_sh[0] = round_to<CT>(part);
      }
      __syncthreads();
      const float total = total_sh[0];
      uint16_t* out = reinterpret_cast<uint16_t*>(a.out) + ((int64_t)bh * a.nqb + qi) * nkb;
      for (int kb = tid; kb < nkb; kb += 256) {
        const float v = kb < kb_item ? colmax[kb] / total : 0.f;
        out[kb] = (uint16_t)(pack2<CT>(v, 0.f) & 0xffffu);
      }
    }
  }
}

// 128-key tiles that any row of item `qi` of a head sees.
__device__ __forceinline__ int max_pool_tiles(const PoolArgs& a, int qi) {
  const int ntiles = (a.Nk + 127) >> 7;
  return a.causal ? min(ntiles, qi + 1) : ntiles;
}

// The tiles [t0, t1) of one item: each row's rounded block maxima into ws[kb][row], the maximum of
// the unrounded ones in m.  The persistent kernel keeps a tile loop of its own: at its 128 VGPRs
// the spills fall otherwise when the tile is a shared function (2 x 12 heads of 32760 at blocks of
// 64: 5.9 -> 6.8 ms).  A change to one of the two loops belongs in both; their maps are compared bit
// for bit in the tests.
template <int CT, int KB>
__device__ __forceinline__ void max_pool_walk(const PoolArgs& a, SA_LDS char* lk, int item, int t0, int t1, float* ws,
                                              float& m) {
  constexpr int DS = 8;
  constexpr int NS = 128 / KB;  // key blocks per tile, q-blocks per item
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hl = lane >> 5, l32 = lane & 31;
  const int nkb = a.nkb;
  const int nqi = (a.Nq + 127) >> 7;
  const uint32_t kstride = (uint32_t)a.ks[2] * 2;
  const int drow = 4 * wave + (lane >> 4);
  const uint32_t k_off = (uint32_t)drow * kstride + (uint32_t)(((lane & 15) ^ (drow & 15)) * 16);
  const int prow = k_row_perm(l32);
  // chunk (2ds + hl) ^ (prow & 15) of row prow: the k-step only flips bits 5-7
  const uint32_t ka0 = (uint32_t)(prow * 256 + ((hl ^ (prow & 15)) * 16));
  // The reference forms qk_scale = fp32(sm_scale) * fp32(1.44269504).
  const float qk_scale = a.scale * 1.44269504f;
  const int r = wave * 32 + l32;
  const int bh = item / nqi;
  const int qi = item - bh * nqi;
  const int b = bh / a.H, h = bh - b * a.H;
  const int hk = h / (a.H / a.Hk);
  const char* qbase = (const char*)a.q + ((int64_t)b * a.qs[0] + (int64_t)h * a.qs[1]) * 2;
  const char* kbase = (const char*)a.k + ((int64_t)b * a.ks[0] + (int64_t)hk * a.ks[1]) * 2;
  const int qrow = qi * 128 + r;
  const int qbr = qrow / KB;  // this row's q-block
  u32x4 qf[DS];
  load_q_operand<128>(qf, qbase, a.qs[2], qrow, a.Nq, hl);
  m = neg_inf();

  for (int kt = t0; kt < t1; ++kt) {
    const int key0 = kt * 128;
    __syncthreads();  // the previous tile (or item epilogue) is done with lds_k
    {
      const __amdgpu_buffer_rsrc_t rs =
          make_rsrc(kbase + (int64_t)key0 * kstride, (uint32_t)(a.Nk - key0) * kstride);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        dma16(rs, (SA_LDS void*)(lk + (256 * j + 64 * wave) * 16), k_off + (uint32_t)j * 16u * kstride);
    }
    __syncthreads();  // waits for this group's DMA
    f32x16 s[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) s[t] = f32x16{};
    {
      // Flat step i = 4 ds + t.  The read for step i + 2 is issued right after the MFMA
      // of step i (the scheduling groups pin that order), so each read has two MFMAs to
      // land; a deeper ring does not fit the 128 VGPRs of four groups per CU.
      u32x4 kr[4];
      auto kread = [&](int i) __attribute__((always_inline)) {
        return *(SA_LDS const u32x4*)(lk + (ka0 ^ (32u * (i >> 2))) + (i & 3) * 8192);
      };
      kr[0] = kread(0);
      kr[1] = kread(1);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
      for (int i = 0; i < 4 * DS; ++i) {
        s[i & 3] = mfma32x32x16<CT>(kr[i & 3], qf[i >> 2], s[i & 3]);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (i + 2 < 4 * DS) {
          kr[(i + 2) & 3] = kread(i + 2);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
      }
    }
    const bool diag = a.causal && kt == qi;
    if (key0 + 128 > a.Nk || diag) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const int key = key0 + t * 32 + tile_key(hl, j);
          if (diag) {
            const int kbk = key / KB;
            if (kbk == qbr && qrow < key) s[t][j] += -1.0e6f;
            if (kbk > qbr) s[t][j] = neg_inf();  // a key block past the row's own: not seen
          }
          if (key >= a.Nk) s[t][j] = neg_inf();
        }
    }
    float mx[NS];
#pragma unroll
    for (int i = 0; i < NS; ++i) mx[i] = neg_inf();
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int j = 0; j < 16; ++j) mx[sub_block<KB>(t, j)] = fmaxf(mx[sub_block<KB>(t, j)], s[t][j]);
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      mx[i] = max_xor32(mx[i]) * qk_scale;
      m = fmaxf(m, mx[i]);
      if ((NS == 1 ? hl == 0 : (i & 1) == hl) && kt * NS + i < nkb) ws[(kt * NS + i) * 128 + r] = round_to<CT>(mx[i]);
    }
  }
}

// Items of a first, partial round, whose groups would leave the others idle: S groups per item,
// each a range of its key tiles; group (item i, range s) writes its block maxima to item i's slot
// and its rows' maxima to ml[i][s][128].  max_pool_join_kernel makes the map rows: maxima do not
// depend on the split, so the map is the same bit for bit.  bf16: [1,12,4096,128] 60 -> 56 us at
// blocks of 128 and 78 -> 64 at 64, [1,1,16000,128] 166 -> 81.
template <int CT, int KB>
__global__ __launch_bounds__(256, 4) void max_pool_ranged_kernel(PoolArgs a, int n, int S, float* ml) {
  constexpr int NS = 128 / KB;
  __shared__ u32x4 lds_k[2048];
  const int i = (int)blockIdx.x % n, s = (int)blockIdx.x / n;
  const int tiles = max_pool_tiles(a, i % ((a.Nq + 127) >> 7));
  float m;
  max_pool_walk<CT, KB>(a, (SA_LDS char*)lds_k, i, s * tiles / S, (s + 1) * tiles / S,
                        a.ws + (size_t)i * (size_t)a.nkb * (128 + (KB == 128 ? 0 : NS)), m);
  const int lane = threadIdx.x & 63;
  if (lane < 32) ml[((size_t)i * S + s) * 128 + (threadIdx.x >> 6) * 32 + lane] = m;
}

template <int CT, int KB>
__global__ __launch_bounds__(256) void max_pool_join_kernel(PoolArgs a, int S, const float* ml) {
  constexpr int NS = 128 / KB;
  __shared__ float row_m[128];
  __shared__ float colmax[KB == 128 ? 1024 : 1];
  __shared__ float total_sh[KB == 128 ? 1 : 4];
  const int i = blockIdx.x, tid = threadIdx.x;
  float* ws = a.ws + (size_t)i * (size_t)a.nkb * (128 + (KB == 128 ? 0 : NS));
  if (tid < 128) {
    float m = neg_inf();
    for (int s = 0; s < S; ++s) m = fmaxf(m, ml[((size_t)i * S + s) * 128 + tid]);
    row_m[tid] = i % ((a.Nq + 127) >> 7) * 128 + tid < a.Nq ? m : pos_inf();
  }
  __syncthreads();
  max_pool_rows<CT, KB>(a, i, ws, ws + (size_t)a.nkb * 128, row_m, colmax, total_sh);
}

// ------------------------------------------------------------------------------------
// Mean-pooled scores.  Pass 1: per-block means of Q and K (replicate-padded tail), fp32,
// into workspace rows of mean_pool_row_len(D) floats (zero past D).  Bound by the read of Q
// and K: a 256-thread group takes one block, RL threads per 16-byte chunk of the head dim
// (16 at D = 128, 16-bit), each summing every RL-th row with eight loads in flight; the RL
// partial sums meet in LDS.  Q and K go in one launch.  At [2,12,32760,128] bf16, blocks of
// 128: 77 us for 403 MB, 5.2 TB/s, the rate of a large device copy (a thread per channel with
// one 2-byte load in flight took 2 x 128 us).
// ------------------------------------------------------------------------------------
template <int IT>
__device__ __forceinline__ float pool_elem(const char* p) {
  if constexpr (IT == kF32) return *reinterpret_cast<const float*>(p);
  else if constexpr (IT == kBF16) return bf16_bits_to_f32(*reinterpret_cast<const uint16_t*>(p));
  else return f16_bits_to_f32(*reinterpret_cast<const uint16_t*>(p));
}

template <int IT>
__global__ __launch_bounds__(256) void mean_pool_rows_kernel(PoolArgs a, int D, int Dp) {
  constexpr int ES = ElemSize<IT>::value;
  constexpr int EPC = 16 / ES;
  __shared__ float part[256 * EPC];
  const int tid = threadIdx.x;
  const bool is_q = (int)blockIdx.x < a.nqb;
  const int blk = is_q ? blockIdx.x : blockIdx.x - a.nqb;
  const int bh = blockIdx.y;
  const int b = bh / a.H, h = bh - b * a.H;
  const int N = is_q ? a.Nq : a.Nk;
  const int64_t* st = is_q ? a.qs : a.ks;
  const char* base = (const char*)(is_q ? a.q : a.k) + ((int64_t)b * st[0] + (int64_t)h * st[1]) * ES;
  const int64_t rstride = st[2] * ES;
  const int chunks = (D + EPC - 1) / EPC;  // <= 256 (D <= 1024)
  const int RL = 256 / chunks;
  const int c = tid % chunks, rl = tid / chunks;
  float acc[EPC];
#pragma unroll
  for (int e = 0; e < EPC; ++e) acc[e] = 0.f;
  if (rl < RL) {
    const char* src = base + c * 16;
    const int row0 = blk * a.bs, last = N - 1;
    if ((c + 1) * EPC <= D) {
      for (int i0 = rl; i0 < a.bs; i0 += 8 * RL) {
        u32x4 w[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int i = i0 + u * RL;
          w[u] = u32x4{0, 0, 0, 0};
          if (i < a.bs) w[u] = *reinterpret_cast<const u32x4*>(src + (int64_t)min(row0 + i, last) * rstride);
        }
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            if constexpr (IT == kF32) {
              acc[j] += __uint_as_float(w[u][j]);
            } else {
              const uint32_t lo = w[u][j] & 0xffffu, hi = w[u][j] >> 16;
              acc[2 * j] += IT == kBF16 ? bf16_bits_to_f32(lo) : f16_bits_to_f32(lo);
              acc[2 * j + 1] += IT == kBF16 ? bf16_bits_to_f32(hi) : f16_bits_to_f32(hi);
            }
          }
      }
    } else {  // the head dim ends inside this chunk: element by element
      for (int i = rl; i < a.bs; i += RL) {
        const char* p = src + (int64_t)min(row0 + i, last) * rstride;
#pragma unroll
        for (int e = 0; e < EPC; ++e)
          if (c * EPC + e < D) acc[e] += pool_elem<IT>(p + e * ES);
      }
    }
#pragma unroll
    for (int e = 0; e < EPC; ++e) part[(rl * chunks + c) * EPC + e] = acc[e];
  }
  __syncthreads();
  float* dst = a.ws + ((is_q ? 0 : (int64_t)a.B * a.H * a.nqb) + (int64_t)bh * (is_q ? a.nqb : a.nkb) + blk) * Dp;
  const int w = chunks * EPC;
  for (int d = tid; d < Dp; d += 256) {
    float s = 0.f;
    if (d < D)
      for (int r = 0; r < RL; ++r) s += part[r * w + d];
    dst[d] = s / (float)a.bs;
  }
}

// Pass 2: a group of 16 waves takes 16 query blocks of one head against every key block, on
// the fp32 matrix cores (v_mfma_f32_16x16x4_f32; fp32 products and sums).  Lane l of a wave
// holds query block l % 16 (A) and key block l % 16 (B) of its tile, and of every 16 channels
// the four from 4 (l / 16), one 16-byte read, so that a read covers 64 consecutive bytes of 16
// rows; D holds key block l % 16 and query blocks 4 (l / 16) .. +3, so a store writes 16
// consecutive map entries.  Wave w takes key tiles w, w + 16, ...; then each wave softmaxes one
// row, from registers up to 512 key blocks.  Bound by latency: 24 heads of
// 256 x 256 blocks take 21 us (one wave per query row with a thread per key block, whose reads
// of a pooled row never coalesce, took 785 us; four waves per group 25 us).
constexpr int kMeanRows = 16;
typedef f32x4 f32x4_dword __attribute__((aligned(4)));  // the caller's workspace may start at any float
constexpr int kMeanWaves = 16;

__global__ __launch_bounds__(64 * kMeanWaves) void mean_pool_scores_kernel(PoolArgs a, int Dp) {
  const int bh = blockIdx.y, qb0 = blockIdx.x * kMeanRows;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane >> 4, sl = lane & 15;
  const float* qp = a.ws + ((int64_t)bh * a.nqb + min(qb0 + sl, a.nqb - 1)) * Dp + 4 * g;
  const float* kp = a.ws + ((int64_t)a.B * a.H * a.nqb + (int64_t)bh * a.nkb) * Dp + 4 * g;
  float* out = reinterpret_cast<float*>(a.out) + ((int64_t)bh * a.nqb + qb0) * a.nkb;
  for (int k0 = wave * 16; k0 < a.nkb; k0 += 16 * kMeanWaves) {
    const float* kr = kp + (int64_t)min(k0 + sl, a.nkb - 1) * Dp;
    f32x4 s = f32x4{};
    int d = 0;
    for (; d + 128 <= Dp; d += 128) {  // 16 loads in flight
      f32x4 qv[8], kv[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        qv[j] = *reinterpret_cast<const f32x4_dword*>(qp + d + 16 * j);
        kv[j] = *reinterpret_cast<const f32x4_dword*>(kr + d + 16 * j);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_16x16x4f32(qv[j][e], kv[j][e], s, 0, 0, 0);
    }
    for (; d < Dp; d += 16) {
      const f32x4 qv = *reinterpret_cast<const f32x4_dword*>(qp + d);
      const f32x4 kv = *reinterpret_cast<const f32x4_dword*>(kr + d);
#pragma unroll
      for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_16x16x4f32(qv[e], kv[e], s, 0, 0, 0);
    }
    const int kb = k0 + sl;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (qb0 + 4 * g + i < a.nqb && kb < a.nkb) out[(int64_t)(4 * g + i) * a.nkb + kb] = s[i] * a.scale;
  }
  __syncthreads();  // the group's scores are in memory
  for (int r = wave; r < kMeanRows; r += kMeanWaves) {
    if (qb0 + r >= a.nqb) break;
    float* row = out + (int64_t)r * a.nkb;
    constexpr int C = 8;
    if (a.nkb <= 64 * C) {
      float x[C];
      float mx = neg_inf();
#pragma unroll
      for (int i = 0; i < C; ++i) {
        x[i] = lane + 64 * i < a.nkb ? row[lane + 64 * i] : neg_inf();
        mx = fmaxf(mx, x[i]);
      }
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < C; ++i)
        if (lane + 64 * i < a.nkb) {
          x[i] = expf(x[i] - mx);
          sum += x[i];
        }
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) sum += __shfl_xor(sum, off, 64);
#pragma unroll
      for (int i = 0; i < C; ++i)
        if (lane + 64 * i < a.nkb) row[lane + 64 * i] = x[i] / sum;
    } else {
      float mx = neg_inf();
      for (int kb = lane; kb < a.nkb; kb += 64) mx = fmaxf(mx, row[kb]);
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
      float sum = 0.f;
      for (int kb = lane; kb < a.nkb; kb += 64) {
        const float e = expf(row[kb] - mx);
        row[kb] = e;
        sum += e;
      }
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) sum += __shfl_xor(sum, off, 64);
      for (int kb = lane; kb < a.nkb; kb += 64) row[kb] = row[kb] / sum;
    }
  }
}

// ------------------------------------------------------------------------------------
// Compute units of the current device (256, an MI355X, if the query fails).
int device_cu_count() {
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0) cus = n;
  }
  return cus;
}

// Resident work-groups of the persistent block-mass kernel on the current device.
int block_mass_groups() { return 3 * device_cu_count(); }
int max_pool_groups() { return 4 * device_cu_count(); }

// Split of a 16-bit call's last, partial round of items: `n` items in S ranges of at least
// kMassMinTiles key tiles each (n = 0: none).  Only a first or second round: after two whole
// rounds the persistent groups have drifted apart and cover a short last round themselves (items
// in rounds of 768: 990 items 175 -> 172 us, 2698 898 -> 895, 3960 2198 -> 2242).  Four tiles: at
// [1,4,2048,128] 30 -> 17 us in four ranges, 22 in the two that eight tiles would allow.
constexpr int kMassMinTiles = 4;
// Key tiles from which a call is split.  Below, the second launch costs a program that records
// call after call as much as the ranges save: max-pool at [1,9,1847,128] 28 -> 22 us on the GPU,
// but 37.5 -> 41 us per recorded call.  At the line itself a call that the program waits for, or
// that follows other GPU work, gains all of it (one recorded call, block mass [1,2,2048,128] 64 -> 53
// us, max-pool [1,2,3072,128] 67 -> 58), while calls of one to four heads back to back, which are
// bound by the host, pay 3-4 us for the launch (39.8 -> 44.2 and 45.9 -> 49.1) up to 2400 and 4300
// keys; past these both gain ([1,2,3500,128] block mass 57 -> 44, [1,2,6000,128] max-pool 70 -> 49).
constexpr int kMassSplitTiles = 16, kMaxSplitTiles = 24;

struct MassSplit {
  int n, S;
};

static MassSplit mass_split(int64_t items, int Nk) {
  const int G = block_mass_groups();
  const int n = (int)(items % G), tiles = (Nk + 127) / 128;
  if (n == 0 || items >= 2 * (int64_t)G || tiles < kMassSplitTiles) return {0, 1};
  int S = G / n;
  S = min(min(S, kMassMaxRanges), tiles / kMassMinTiles);
  return S >= 2 ? MassSplit{n, S} : MassSplit{0, 1};
}

// The resident groups' slots, then the range records of a split round: n * S <= G of 256 floats.  From
// the length that may be split on the room for a full round of them is always there, so that a
// workspace sized for a call also serves every smaller one (0.8 MB).
size_t block_mass_workspace_floats(int64_t items, int64_t nkb, int64_t Nk) {
  const int64_t G = block_mass_groups(), groups = items < G ? items : G;
  const bool may_split = items > 0 && (Nk + 127) / 128 >= kMassSplitTiles;
  return (size_t)(groups * nkb * 128 + (may_split ? G * 256 : 0));
}

template <int CT, int KB>
static hipError_t launch_mass(const PoolArgs& a, hipStream_t stream) {
  const int items = a.B * a.H * ((a.Nq + 127) / 128);
  const MassSplit sp = mass_split(items, a.Nk);
  const int whole = items - sp.n;
  if (whole > 0) {
    block_mass_persistent_kernel<CT, KB><<<min(whole, block_mass_groups()), 256, 0, stream>>>(a, whole);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || sp.n == 0) return e;
  }
  float* ml = a.ws + (size_t)min(items, block_mass_groups()) * (size_t)a.nkb * 128;
  block_mass_ranged_kernel<CT, KB><<<sp.n * sp.S, 256, 0, stream>>>(a, whole, sp.n, sp.S, ml);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int slices = min((a.nkb + 15) / 16, max(1, 1024 / sp.n));
  block_mass_combine_kernel<KB><<<dim3(sp.n, slices), 256, 0, stream>>>(a, whole, sp.S, ml);
  return hipGetLastError();
}

hipError_t launch_block_mass_pool(const PoolArgs& a, int dtype, int D, hipStream_t stream) {
  (void)D;
  if (a.B * a.H * a.nqb == 0) return hipSuccess;
  if (dtype == kF32) {
    switch (a.bs) {
      case 16: return launch_mass_f32<16>(a, stream);
      case 32: return launch_mass_f32<32>(a, stream);
      case 64: return launch_mass_f32<64>(a, stream);
      default: return launch_mass_f32<128>(a, stream);
    }
  }
  switch (a.bs) {
    case 16: return dtype == kBF16 ? launch_mass<kBF16, 16>(a, stream) : launch_mass<kF16, 16>(a, stream);
    case 32: return dtype == kBF16 ? launch_mass<kBF16, 32>(a, stream) : launch_mass<kF16, 32>(a, stream);
    case 64: return dtype == kBF16 ? launch_mass<kBF16, 64>(a, stream) : launch_mass<kF16, 64>(a, stream);
    default: return dtype == kBF16 ? launch_mass<kBF16, 128>(a, stream) : launch_mass<kF16, 128>(a, stream);
  }
}

// Key ranges per item of a 16-bit max-pool call (1: none), at least kMassMinTiles key tiles each:
// up to two fifths of a round of items at blocks of 128 (384 items 60.2 -> 56.5 us, 504 128.2 ->
// 129.2), half a round below, whose longer map rows the join spreads (504 at 64: 160 -> 143).
static int max_split(int64_t items, int Nk, int block_size) {
  const int G = max_pool_groups();
  if (items <= 0 || items > (block_size == 128 ? 2 * G / 5 : G / 2) || (Nk + 127) / 128 < kMaxSplitTiles) return 1;
  return max(1, min(min((int)(max_pool_groups() / items), kMassMaxRanges), (Nk + 127) / 128 / kMassMinTiles));
}

// Per group the rows' block maxima and, below block 128, the item's column maxima; then the ranges'
// row maxima (items * S <= G of 128 floats), with room for a full round as in the block-mass call.
size_t max_pool_workspace_floats(int64_t items, int64_t nkb, int64_t N, int block_size) {
  const int64_t G = max_pool_groups(), groups = items < G ? items : G;
  const int64_t per_kb = 128 + (block_size == 128 ? 0 : 128 / block_size);
  const bool may_split = items > 0 && (N + 127) / 128 >= kMaxSplitTiles;
  return (size_t)(groups * nkb * per_kb + (may_split ? G * 128 : 0));
}

template <int CT, int KB>
static hipError_t launch_max(const PoolArgs& a, hipStream_t stream) {
  const int items = a.B * a.H * ((a.Nq + 127) / 128);
  const int S = max_split(items, a.Nk, KB);
  if (S == 1) {
    max_pool_persistent_kernel<CT, KB><<<min(items, max_pool_groups()), 256, 0, stream>>>(a, items);
    return hipGetLastError();
  }
  float* ml = a.ws + (size_t)items * (size_t)a.nkb * (128 + (KB == 128 ? 0 : 128 / KB));
  max_pool_ranged_kernel<CT, KB><<<items * S, 256, 0, stream>>>(a, items, S, ml);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  max_pool_join_kernel<CT, KB><<<items, 256, 0, stream>>>(a, S, ml);
  return hipGetLastError();
}

hipError_t launch_max_pool(const PoolArgs& a, int dtype, int D, hipStream_t stream) {
  (void)D;
  if (a.B * a.H * a.nqb == 0) return hipSuccess;
  if (dtype == kF32) {
    switch (a.bs) {
      case 16: return launch_max_f32<16>(a, stream);
      case 32: return launch_max_f32<32>(a, stream);
      case 64: return launch_max_f32<64>(a, stream);
      default: return launch_max_f32<128>(a, stream);
    }
  }
  switch (a.bs) {
    case 16: return dtype == kBF16 ? launch_max<kBF16, 16>(a, stream) : launch_max<kF16, 16>(a, stream);
    case 32: return dtype == kBF16 ? launch_max<kBF16, 32>(a, stream) : launch_max<kF16, 32>(a, stream);
    case 64: return dtype == kBF16 ? launch_max<kBF16, 64>(a, stream) : launch_max<kF16, 64>(a, stream);
    default: return dtype == kBF16 ? launch_max<kBF16, 128>(a, stream) : launch_max<kF16, 128>(a, stream);
  }
}

// Floats of a pooled row in the workspace: whole steps of 16 channels for the scores kernel.
int mean_pool_row_len(int D) { return (D + 15) & ~15; }

hipError_t launch_mean_pool(const PoolArgs& a, int dtype, int D, hipStream_t stream) {
  if (a.B * a.H == 0) return hipSuccess;
  const int Dp = mean_pool_row_len(D);
  const dim3 grid(a.nqb + a.nkb, a.B * a.H);
  if (dtype == kF32) mean_pool_rows_kernel<kF32><<<grid, 256, 0, stream>>>(a, D, Dp);
  else if (dtype == kBF16) mean_pool_rows_kernel<kBF16><<<grid, 256, 0, stream>>>(a, D, Dp);
  else mean_pool_rows_kernel<kF16><<<grid, 256, 0, stream>>>(a, D, Dp);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  mean_pool_scores_kernel<<<dim3((a.nqb + kMeanRows - 1) / kMeanRows, a.B * a.H), 64 * kMeanWaves, 0,
                            stream>>>(a, Dp);
  return hipGetLastError();
}

}  // namespace sa
