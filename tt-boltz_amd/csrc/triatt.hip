// Triangle attention (starting / ending node) for gfx950.
//
// Replaces TriangleAttention.forward (tt_bio/reference.py:294-365 with Attention
// 33-194, _attention tt_bio/boltz2.py:790-810, chunk_layer 542-628) and the ttnn
// TriangleAttention (tt_bio/tenstorrent.py:506-650).
//
// "Frame" coordinates: the starting node attends along rows of z, the ending node
// along rows of z^T.  Frame pair (i, j) is z pair (i, j) (starting) or (j, i)
// (ending); transposition is done by addressing, never materialized.
//
//   ta_proj  LN(z) -> q (pre-scaled by log2(e)/sqrt(d)), k, v^T, per-head bias
//            (x log2(e)) and the per-(row, key) additive mask term, one pass over z.
//              Q, K    op_t [B][N(row i)][H][N(j)][D]
//              Vt      op_t [B][N(row i)][H][D][N(k)], keys stored at perm16(k) (bits 2
//                      and 3 swapped) so a P.V operand fragment is one 16-byte run
//              bias32  fp32 [B][H][N(j)][N(k)]   (shared by all rows i; x log2(e) + REF_SHIFT)
//              mask16  op_t [B][N(i)][N(k)]      0, or -inf for masked / padding keys
//   ta_attn  flash attention (see the kernel's comment): 16-wave workgroups of 4 frame rows
//            x 128 queries, LDS-DMA ring, bias / mask / reference max folded into MFMAs,
//            lazy-max softmax.  Output O (normalized, ungated) op_t [B][N(i)][N(j)][H*D].
//   ta_out   o-proj epilogue: gate recomputed from LN(z) (MFMA), o*sigmoid(g) as linear_o's B
//            operand through LDS, residual.
#include <type_traits>

#include "pf_common.h"
#include "pf_direct.h"
#include "pf_internal.h"

namespace {

// C = H * D: the attention width (q / k / v / o channels).  The pair width c_z (CC in the
// projection kernels) is 128 in the trunk and 64 in the template stack.
constexpr int C = 128, H = 4, D = 32;
constexpr float LOG2E = 1.4426950408889634f;
constexpr float RESCALE_SLACK = 8.f;   // log2 units: a rescale leaves queries whose P stay <= 2^8 as they are
// Log2 units that every stored bias is raised by.  The softmax does not see it, but rows of logits
// about 0 then pass the first tile's test for 0 as their reference (LSTEP_MIN) and their P still reach
// 1: a mean P of a lane's keys between 2^-4 and 2^8 (without the shift) is accepted.  The middle of the
// range that fp16 leaves: over random blocks at most 3 % of the tiles take the third MFMA, with 2
// 0 - 37 %, with 6 0 - 28 %, and with 4 but LSTEP_MAX = 2^14 0 - 27 %.
constexpr float REF_SHIFT = 4.f;

typedef op_t opx2 __attribute__((ext_vector_type(2)));

PF_DEV float dot2_ones(const opx2& p, float acc) {
#ifdef PF_OPERAND_BF16
  const opx2 one = {(op_t)1.f, (op_t)1.f};
  return __builtin_amdgcn_fdot2_f32_bf16(p, one, acc, false);
#else
  const opx2 one = {(op_t)1.f, (op_t)1.f};
  return __builtin_amdgcn_fdot2(p, one, acc, false);
#endif
}

// Additive mask term of one (row, key), log2 units: -inf for padding keys and for the
// reference's 1e9*(mask-1) whenever that is beyond op_t's range (a masked key).
PF_DEV op_t mask_term(bool pad, float mv) {
  const float t = 1e9f * (mv - 1.f) * LOG2E;
  return (op_t)(pad || t < -65504.f ? -INFINITY : t);
}

// ---------------------------------------------------------------------------------
// Projection (pf_direct.h): 12 waves walk groups of 64 frame positions (ip, j0 .. j0 + 63).  Wave w
// owns one head of q (w < 4), k (w < 8) or v: its 32 weight rows in registers with the LayerNorm
// affine folded in (W' = W diag(gamma) in op_t, W beta in fp32 as the accumulator start), so a
// group is only normalized, by waves 0-7.  Waves 8 and 9 also compute the triangle bias of one
// 32-position tile each, from the bias rows in LDS.  The MFMA orientation is chosen per output so
// that the outputs' LDS stage takes 8- or 16-byte writes, and every store instruction writes whole
// 128-byte lines:
//   Q, K  [j][d]:  D[d][pos]   a lane holds runs of 4 d of its position
//   V^T   [d][k]:  D[pos][d]   a lane's key runs g = 2p, 2p+1 are 8 adjacent slots (perm16)
//   bias  [hd][j]: D[hd][pos]  a lane holds the 4 heads of its position
// FAST (the fast mode's block-fp8 points): the weights come as MXFP8 and are dequantized into the
// registers; q, k and v are quantize-dequantized per head (one 32-channel block per position)
// before they are stored.  Q and K blocks are lane pairs of the D[d][pos] accumulator; V's D[pos][d]
// orientation spreads a block over 32 lanes, so a D[d][pos] copy of V gives each key's block scale,
// passed through 32 floats of LDS per wave.
// Against weights resident in LDS with one 8-wave workgroup's wave per tile (us a launch): N = 128
// 20.6 + 5.2 of statistics -> 15.1, 384 54 -> 41, 512 89 -> 65, 1024 314 -> 242.
// ---------------------------------------------------------------------------------
constexpr int TAP_WAVES = 12, TAP_LN = 8;   // waves; the first ones normalize
constexpr int TAP_SP = 40, TAP_VP = 72;     // stage pitches: [64 positions][32 d + 8], [32 d][64 keys + 8]
template <int CC>
constexpr size_t tap_lds() {
  return (size_t)(2 * DP_ROWS * (CC + 8) + 2 * H * (CC + 8)) * sizeof(op_t) +
         (size_t)TAP_WAVES * (32 * (CC + 8) > DP_ROWS * TAP_SP ? 32 * (CC + 8) : DP_ROWS * TAP_SP) * sizeof(op_t) +
         (3 * C + 32 + 32 * TAP_WAVES) * sizeof(float);
}

// W_q, W_k, W_v, W_g: op_t [C][CC], or (FAST) MXFP8 bytes with their scales in `s`.
struct TaWeights {
  const void* w[4];
  const void* s[4] = {nullptr, nullptr, nullptr, nullptr};
  const op_t *g_lo = nullptr, *o_lo = nullptr;   // the residuals of W_g and W_o (op_t, or null)
};

// offb (optional, fp32 [3 C + H]): the exact W beta of the q, k, v and bias rows (else computed
// from the op_t weights); lo: the residuals of the kernel's gamma-folded weights (W diag(gamma) -
// op_t(W16 diag(gamma)), four [rows][CC] arrays for q, k, v, bias), used as DirectLo says, with the
// stats partials for DL_MEAN.
struct TaMeanFix { const float* offb; const op_t* lo[4]; const float* stats; };

template <int CC, bool FAST, int LO>
__global__ __launch_bounds__(64 * TAP_WAVES, 1) void ta_proj_kernel(
    const float* __restrict__ z, const float* __restrict__ pair_mask,
    const float* __restrict__ lnw, const float* __restrict__ lnb, TaWeights tw,
    const op_t* __restrict__ wb, op_t* __restrict__ Q, op_t* __restrict__ K,
    op_t* __restrict__ Vt, float* __restrict__ bias32, op_t* __restrict__ mask16,
    int ngroups, int N, int n_valid, int ending, float qscale, float eps, TaMeanFix mf) {
  constexpr int LW = CC + 8, KS = CC / 16, NT = 64 * TAP_WAVES;
  constexpr int WB = 32 * LW > DP_ROWS * TAP_SP ? 32 * LW : DP_ROWS * TAP_SP;   // a wave's buffer
  extern __shared__ __attribute__((aligned(16))) op_t plds[];
  op_t* sx = plds;                                     // normalized positions [2][64][LW]
  op_t* sbw = sx + 2 * DP_ROWS * LW;                   // bias rows, then (DL_MFMA) their residuals [2][H][LW]
  op_t* wbuf = sbw + 2 * H * LW;                       // weights, then outputs, per wave
  float* soff = reinterpret_cast<float*>(wbuf + TAP_WAVES * WB);   // W beta of the q, k, v rows, the bias rows
  float* vsc = soff + 3 * C + 32;                      // FAST: a wave's per-key V block scales
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, m = lane & 31;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kind = wid >> 2, hd = wid & 3;             // 0 q, 1 k, 2 v
  op_t* stg = wbuf + wid * WB;
  vsc += 32 * wid;
  auto group = [&](int g) PF_INLINE -> PosTile { return pos_tile(2u * g, N); };
  // the z pair of frame position c of a group
  auto zpair = [&](const PosTile& pt, int c) PF_INLINE -> long {
    return ((long)pt.b * N + (ending ? pt.c0 + c : pt.r)) * N + (ending ? pt.r : pt.c0 + c);
  };
  DirectLn<CC, TAP_LN> ln;
  float mv = 1.f;
  auto fetch = [&](int g) PF_INLINE {
    const PosTile pt = group(g);
    if (wid < TAP_LN) ln.load(z, [&](int c) PF_INLINE -> long { return zpair(pt, c); }, wid, lane);
    if (pair_mask && tid < DP_ROWS) mv = pair_mask[zpair(pt, tid)];
  };
  // ---- set-up: every global load first, so that it costs about one memory round trip ----
  fetch(blockIdx.x);
  ln.load_gamma(nullptr, lane);
  DirectW<CC> w, wl;
  const long r0 = 32l * hd * CC;
  if constexpr (!FAST) w.load((const op_t*)tw.w[kind] + r0, lane);
  const int row = 32 * wid + m;   // of the 3 C projection rows
  const bool exact = !FAST && mf.offb;
  float c0 = exact ? mf.offb[row] : 0.f;
  const float gb = tid < 2 * CC ? (tid < CC ? lnw[tid] : lnb[tid - CC]) : 0.f;
  // bias rows: wave 0 (c_z = 64: half of it), 8 channels bc .. of row br a lane
  const bool bias_lane = tid < H * CC / 8;
  const int br = tid / (CC / 8), bc = 8 * (tid % (CC / 8));
  opx8 bw = zero_x8(), bl = zero_x8();
  float cb = 0.f;
  if (bias_lane) {
    bw = ld_x8(wb + br * CC + bc);
    if constexpr (LO != DL_NONE) bl = ld_x8(mf.lo[3] + br * CC + bc);
    if (exact) cb = mf.offb[3 * C + br];
  }
  float psum = 0.f;
  if constexpr (LO == DL_MEAN) {
    if (tid < 512) {
      float pv[stats_per<512>()];
      stats_load<512>(mf.stats, pv);
#pragma unroll
      for (int i = 0; i < stats_per<512>(); ++i) psum += pv[i];
    }
  }
  DirectW8<CC> w8;
  if constexpr (FAST)
    w8.load((const uint8_t*)tw.w[kind] + r0, (const uint8_t*)tw.s[kind] + 32 * hd * (CC / 32), lane);
  __builtin_amdgcn_sched_barrier(0);
  float* sgb = reinterpret_cast<float*>(sx + DP_ROWS * LW);   // gamma, beta [2][CC], mu [CC], partial sums [4][128]
  float* smu = sgb + 2 * CC;                                  // (in sx[1], free until the second group)
  if (tid < 2 * CC) sgb[tid] = gb;
  if (LO == DL_MEAN && tid < 512) smu[PS_C + tid] = psum;
  __syncthreads();
  if (LO == DL_MEAN && tid < PS_C)
    smu[tid] = (smu[PS_C + tid] + smu[2 * PS_C + tid]) + (smu[3 * PS_C + tid] + smu[4 * PS_C + tid]);
  if constexpr (FAST)
    w8.dequant(w);
  else
    w.turn(stg, lane);
  __builtin_amdgcn_sched_barrier(0);
  // (the residuals' own round trip runs beside the LayerNorm: with everything in flight at once
  // the set-up spilled.  DL_MFMA, whose residuals stay in registers, keeps 5 registers of loop-
  // invariant addresses in scratch: 24 bytes a lane, each read once a group)
  if constexpr (LO != DL_NONE) wl.load(mf.lo[kind] + r0, lane);
  if (wid < TAP_LN) ln.store(sx, eps, wid, lane);
  if (!exact) c0 = direct_wbeta<KS, f32x4>(w.v, sgb + CC, h);
  w.template fold<f32x4>(sgb, h);
  if constexpr (LO != DL_NONE) wl.turn(stg, lane);
  auto bias_sum = [&](float v) PF_INLINE -> float {   // over the CC / 8 lanes of a bias row
#pragma unroll
    for (int o = CC / 16; o >= 1; o >>= 1) v += __shfl_xor(v, o);
    return v;
  };
  if (wid == 0) {
    float d = 0.f;
    opx8 f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      d += (float)bw[e] * sgb[CC + bc + e];
      f[e] = (op_t)((float)bw[e] * sgb[bc + e]);
    }
    d = bias_sum(d);
    if (!exact) cb = d;
    if (bias_lane) {
      st_x8(sbw + br * LW + bc, f);
      if constexpr (LO == DL_MFMA) st_x8(sbw + (H + br) * LW + bc, bl);
    }
  }
  if constexpr (LO == DL_MEAN) {
    __syncthreads();
    c0 += direct_wbeta<KS, f32x4>(wl.v, smu, h);
    if (wid == 0) {
      float d = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) d += (float)bl[e] * smu[bc + e];
      cb += bias_sum(d);
    }
  }
  if (h == 0) soff[row] = c0;
  if (bias_lane && bc == 0) soff[3 * C + br] = cb;
  __syncthreads();

  int buf = 0;
  for (int gi = blockIdx.x; gi < ngroups; gi += gridDim.x, buf ^= 1) {
    const PosTile pt = group(gi);
    op_t* sxb = sx + buf * DP_ROWS * LW;
    if (gi != (int)blockIdx.x) {
      if (wid < TAP_LN) ln.store(sxb, eps, wid, lane);
      __syncthreads();   // sx[buf] is whole; every wave is done with sx[buf ^ 1]
    }
    if (tid < DP_ROWS)
      // frame key j0 + tid of row ip: padding -> excluded; otherwise inf*(mask-1) (log2 units)
      mask16[((long)pt.b * N + pt.r) * N + pt.c0 + tid] = mask_term(pt.c0 + tid >= n_valid, mv);
    if (gi + (int)gridDim.x < ngroups) fetch(gi + gridDim.x);
    const long rowh = ((long)pt.b * N + pt.r) * H + hd;   // (b, ip, head) block
    if (kind < 2) {
      // Q, K: D[d][pos]; lane (pos m, h) holds d = 8g + 4h + e in acc[4g + e]
      f32x16 acc[2];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 c4 = *reinterpret_cast<const f32x4*>(soff + 32 * wid + 8 * g + 4 * h);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[0][4 * g + e] = acc[1][4 * g + e] = c4[e];
      }
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const opx8 xf = ld_x8(sxb + (32 * t + m) * LW + 16 * s + 8 * h);
          acc[t] = mfma32(w.v[s], xf, acc[t]);
          if constexpr (LO == DL_MFMA) acc[t] = mfma32(wl.v[s], xf, acc[t]);
          if (s % 4 == 3) __builtin_amdgcn_sched_barrier(0);   // not every fragment read at once
        }
      const float sc = kind == 0 ? qscale : 1.f;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        if constexpr (FAST) mx_fake_quant16(acc[t]);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          opx4 v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = (op_t)(acc[t][4 * g + e] * sc);
          st_x4(stg + (32 * t + m) * TAP_SP + 8 * g + 4 * h, v);
        }
      }
      op_t* dst = (kind == 0 ? Q : K) + (rowh * N + pt.c0) * D;   // 64 positions of 32 d: 4 KB
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int c = lane + 64 * q;
        st_x8(dst + 8 * c, ld_x8(stg + (c >> 2) * TAP_SP + 8 * (c & 3)));
      }
    } else {
      // V^T: D[pos][d]; lane (d m, h) holds keys 8g + 4h + e of a tile in acc[4g + e]
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const op_t* xr = sxb + (32 * t + m) * LW + 8 * h;
        if constexpr (FAST) {   // block scale of key 32 t + m -> vsc[m]
          f32x16 at;
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const f32x4 c4 = *reinterpret_cast<const f32x4*>(soff + 32 * wid + 8 * g + 4 * h);
#pragma unroll
            for (int e = 0; e < 4; ++e) at[4 * g + e] = c4[e];
          }
#pragma unroll
          for (int s = 0; s < KS; ++s) at = mfma32(w.v[s], ld_x8(xr + 16 * s), at);
          float a = 0.f;
#pragma unroll
          for (int r = 0; r < 16; ++r) a = fmaxf(a, fabsf(at[r]));
          a = xor32_max(a);
          if (h == 0) vsc[m] = mx_block_scale(a);
        }
        f32x16 acc;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = c0;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          const opx8 xf = ld_x8(xr + 16 * s);
          acc = mfma32(xf, w.v[s], acc);
          if constexpr (LO == DL_MFMA) acc = mfma32(xf, wl.v[s], acc);
        }
        if constexpr (FAST) {   // same wave: its LDS accesses complete in order
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const f32x4 X4 = *reinterpret_cast<const f32x4*>(vsc + 8 * g + 4 * h);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[4 * g + e] = mx_fake_quant1(acc[4 * g + e], X4[e], 448.f * X4[e]);
          }
        }
        // keys 8g + 4h + e of runs g = 2p, 2p+1 sit at storage 16p + 8h .. +7 (perm16)
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          opx8 v;
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = (op_t)acc[8 * p + e];
          st_x8(stg + m * TAP_VP + 32 * t + 16 * p + 8 * h, v);
        }
      }
      op_t* dst = Vt + rowh * D * (long)N + pt.c0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {   // eight lanes write a d's 128 bytes
        const int d = 8 * q + (lane >> 3), chunk = lane & 7;
        st_x8(dst + (long)d * N + 8 * chunk, ld_x8(stg + d * TAP_VP + 8 * chunk));
      }
      if (hd < 2) {   // the bias of tile hd: D[head][pos]; rows 0..H-1 are acc[0..3] of the h = 0 lanes
        f32x16 acc = zero16();
        const op_t* br = sbw + (m & (H - 1)) * LW + 8 * h;   // rows past H repeat and are not stored
        const op_t* xr = sxb + (32 * hd + m) * LW + 8 * h;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          const opx8 xf = ld_x8(xr + 16 * s);
          acc = mfma32(ld_x8(br + 16 * s), xf, acc);
          if constexpr (LO == DL_MFMA) acc = mfma32(ld_x8(br + H * LW + 16 * s), xf, acc);
        }
        if (h == 0) {
#pragma unroll
          for (int r = 0; r < H; ++r)
            bias32[(((long)pt.b * H + r) * N + pt.r) * N + pt.c0 + 32 * hd + m] =
                fmaf(acc[r] + soff[3 * C + r], LOG2E, REF_SHIFT);
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------------
// Flash attention.  OUT_F32 = false: O op_t [B][N][N][H*D] (frame pair layout);
// OUT_F32 = true: O fp32 [B][N][H][N][D] (the standalone attention-core API).
//
// A workgroup is 16 waves (four per SIMD): 4 frame rows (ip0 .. ip0+3) x 4 blocks of 32 queries;
// each wave owns one row and one 32-query block and walks 4 heads x N/64 key tiles.  Per step
// the workgroup's fp32 bias tile [128 q][64 k], the four rows' K [64 k][32 d] and V^T
// [32 d][64 k] tiles and their mask entries move global -> LDS by DMA (buffer loads straight to
// LDS, no VGPR staging) through a 2-deep ring, one barrier per step.  Scores S'^T[key][query]
// come out of two or three MFMAs per 32x32 tile:
//     bias^T (fp32, the accumulator's start value, read from LDS in accumulator order)
//     + K.Q^T (2)  +  [1, mask[key]] . [-m[q], 1]^T (1: two used k-slots)
// so the bias, the key mask and the reference max cost no VALU and the bias is not rounded;
// the softmax is exp2, an fp16 pair pack and v_dot2 row sums.  The third MFMA is left out while
// it would add zeros: the reference of every query of the wave is 0 and the tile lies before the
// row's first masked or padded key (masks are mostly tails).  The reference m[q] is kept as an
// op_t value (exact as an MFMA operand).  It starts at 0, which a head's first tile accepts when
// every lane's row sum is at least LSTEP_MIN, and moves lazily: to the first tile's maximum when
// 0 is not accepted, while a query has seen no unmasked key, or when a tile's row sum exceeds
// LSTEP_MAX.  A P that would overflow op_t fails the same test before it reaches
// the P.V MFMA, and the tile is then repacked from S' with the new reference.  (Against a third
// MFMA in every tile and a reference that always moved at the first: N = 1024 1083 -> 1051 us a
// launch, 4 x N = 256 108 -> 105 us.)  A wave's two key halves of a step are processed
// one after the other (so a tile's scores always use the reference the previous tile left);
// four waves per SIMD (about 100 VGPRs each) hide each other's MFMA and LDS latencies.
// Rows whose valid keys are all masked: the fp32 reference adds -1e9 to every logit,
// which rounds them all to -1e9 (|logit| < 32), i.e. a uniform average over the keys.
// Such a row's waves skip the tiles (still taking part in every barrier and DMA) and write
// the mean of v after the loop.
// ---------------------------------------------------------------------------------
constexpr int TA_WAVES = 16;
// LDS sections (bytes), each holding stage 0 then stage 1:
//   bias fp32 [128 q][64 k]: rows of 256 B, 16-byte chunk c of row q at position c ^ (q & 15)
//   K   op_t  [4 rows][64 k][32 d]: rows of 64 B, chunk swizzle swz4
//   V^T op_t  [4 rows][32 d][64 k]: rows of 128 B, chunk swizzle swz8
//   mask op_t [4 rows][64 k] (wave 0's 1 KB DMA; the upper 512 B repeat the lower)
constexpr int TS_BIAS = 0, TB_STAGE = 32768;
constexpr int TS_K = 65536, TK_STAGE = 16384;
constexpr int TS_V = 98304, TV_STAGE = 16384;
constexpr int TS_MASK = 131072, TM_STAGE = 1024;
constexpr size_t TA_LDS = (size_t)TS_MASK + 2 * TM_STAGE;
// A lane's row sum (16 keys) of one tile that forces a rescale: every P is then still finite in fp16.
constexpr float LSTEP_MAX = 61440.f;
// A lane's row sum (16 keys) of a head's first tile from which on 0 serves as the reference: one of
// its P is then at least 1, what the first tile's maximum as the reference would give, so the smaller
// P keep as many bits in op_t.
constexpr float LSTEP_MIN = 16.f;

// 16-byte chunk swizzles: rows of 8 chunks (V^T) and of 4 chunks (K).  A fragment read takes
// one chunk from each of 32 consecutive rows; any 16 consecutive rows land in 16 distinct
// 16-byte bank groups.
PF_DEV int swz8(int r) { return ((r >> 1) & 7) ^ ((r & 1) << 2); }
PF_DEV int swz4(int r) { return (r >> 2) & 3; }
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
PF_DEV uint32_t half_bits(op_t v) { return __builtin_bit_cast(uint16_t, v); }
PF_DEV opx8 as_x8(const u32x4& v) { return __builtin_bit_cast(opx8, v); }
// LDS reads from absolute LDS byte addresses (the per-lane address registers already hold the
// allocation base, so the loop's reads need no address arithmetic beyond the immediate offset)
typedef __attribute__((address_space(3))) const char* lds_ptr;
PF_DEV lds_ptr lds_at(uint32_t a) { return (lds_ptr)(uintptr_t)a; }
PF_DEV opx8 lds_rd8(uint32_t a) { return *reinterpret_cast<__attribute__((address_space(3))) const opx8*>(lds_at(a)); }
PF_DEV f32x4 lds_rd4f(uint32_t a) {
  return *reinterpret_cast<__attribute__((address_space(3))) const f32x4*>(lds_at(a));
}
PF_DEV uint32_t lds_rd16(uint32_t a) {
  return *reinterpret_cast<__attribute__((address_space(3))) const uint16_t*>(lds_at(a));
}
// Raw buffer resource over `bytes` bytes at `p` (stride 0, reads beyond `bytes` return zero).
PF_DEV __amdgpu_buffer_rsrc_t make_rsrc(const void* p, long bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)min(bytes, 0x7fffffffl), 0x00020000);
}
// 16 bytes per lane from resource byte offset voff + soff into LDS at lds + 16 * lane.
PF_DEV void dma16(__amdgpu_buffer_rsrc_t r, char* lds, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, voff, soff, 0, 0);
}

template <bool OUT_F32>
__global__ __launch_bounds__(64 * TA_WAVES, 1) void ta_attn_kernel(
    const op_t* __restrict__ Q, const op_t* __restrict__ K, const op_t* __restrict__ Vt,
    const float* __restrict__ bias32, const op_t* __restrict__ mask16, op_t* __restrict__ O16,
    float* __restrict__ O32, int N, int n_valid, int total, int full, int split) {
  extern __shared__ __attribute__((aligned(16))) char alds[];
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, m = lane & 31;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row = wid & 3, qb = wid >> 2;   // frame row, 32-query block
  // Workgroups 0 .. full-1 take all heads of their (rows, queries) block; the blocks after them
  // (a last round that would leave at least half of the CUs idle, or a whole launch that small)
  // go to `split` (2 or 4) workgroups each, H / split heads apiece, so that round takes about
  // 1 / split as long.
  int w, h0 = 0, nh = H;
  if ((int)blockIdx.x < full) {
    w = xcd_remap(blockIdx.x, full);
  } else {
    const int hw = xcd_remap(blockIdx.x - full, split * (total - full));
    w = full + hw / split;
    nh = H / split;
    h0 = (hw % split) * nh;
  }
  const int nQP = (N + 127) >> 7, nKB = N >> 6, T = nh * nKB;
  const int per_b = (N >> 2) * nQP;
  const int b = w / per_b;
  const int rem = w - b * per_b;
  const int rg = rem / nQP;
  const int jw0 = (rem - rg * nQP) * 128;
  const int ip0 = 4 * rg, ip = ip0 + row;
  const long NN = (long)N * N;
  const int seqD = N * D;                 // elements of one (row, head) Q / K / V^T block

  // ---- DMA: buffer resources (SGPRs) over this workgroup's operands, per-lane 32-bit source
  // offsets, the step's offset as the uniform soffset; reads outside a resource return 0 ----
  // bias: wave w's instruction j fills LDS bytes 2048 w + 1024 j .. of the stage, i.e. rows
  // q = 8 w + 4 j + (lane >> 4), position lane & 15, which holds chunk (lane & 15) ^ (q & 15).
  // K and V^T: chunk tid of the 16 KB tile (one instruction each); mask: wave 0, 1 KB.
  const __amdgpu_buffer_rsrc_t rB = make_rsrc(bias32 + (long)b * H * NN, (long)H * NN * 4);
  const __amdgpu_buffer_rsrc_t rK = make_rsrc(K + ((long)b * N + ip0) * H * seqD, 4l * H * seqD * 2);
  const __amdgpu_buffer_rsrc_t rV = make_rsrc(Vt + ((long)b * N + ip0) * H * seqD, 4l * H * seqD * 2);
  const __amdgpu_buffer_rsrc_t rM = make_rsrc(mask16 + ((long)b * N + ip0) * N, 4l * N * 2);
  uint32_t offB[2], offK, offV;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int q = 8 * wid + 4 * j + (lane >> 4);
    offB[j] = 4u * ((uint32_t)min(jw0 + q, N - 1) * (uint32_t)N + 4u * (uint32_t)((lane & 15) ^ (q & 15)));
  }
  {
    const int c = tid;
    const int rk = c >> 8, kk = (c >> 2) & 63, dd = (c >> 3) & 31;
    offK = 2u * (rk * H * seqD + kk * D + 8 * ((c & 3) ^ swz4(kk)));
    offV = 2u * (rk * H * seqD + dd * N + 8 * ((c & 7) ^ swz8(dd)));
  }
  const uint32_t offM = 2u * (((lane >> 3) & 3) * N + 8 * (lane & 7));
  // stage `s` of step (hd, kb0)
  auto issue = [&](int s, int hd, int kb0) PF_INLINE {
    const uint32_t sb = 4u * ((uint32_t)hd * (uint32_t)NN + (uint32_t)kb0);
    const uint32_t skv = 2u * ((uint32_t)(hd * seqD) + (uint32_t)kb0 * D);
    const uint32_t sv = 2u * ((uint32_t)(hd * seqD) + (uint32_t)kb0);
#pragma unroll
    for (int j = 0; j < 2; ++j) dma16(rB, alds + TS_BIAS + s * TB_STAGE + 2048 * wid + 1024 * j, offB[j], sb);
    dma16(rK, alds + TS_K + s * TK_STAGE + 1024 * wid, offK, skv);
    dma16(rV, alds + TS_V + s * TV_STAGE + 1024 * wid, offV, sv);
    if (wid == 0) dma16(rM, alds + TS_MASK + s * TM_STAGE, offM, 2u * (uint32_t)kb0);
  };

  // ---- per-lane LDS read addresses (stage 0; stage 1 adds the section's stage size) ----
  const uint32_t base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)alds;
  const int qrow = 32 * qb + m;
  uint32_t aB[8], aV[4], aK[2];
#pragma unroll
  for (int u = 0; u < 2; ++u)            // key half u, accumulator register group g
#pragma unroll
    for (int g = 0; g < 4; ++g)
      aB[4 * u + g] = base + TS_BIAS + 256 * qrow + 16 * ((8 * u + 2 * g + h) ^ (qrow & 15));
#pragma unroll
  for (int c = 0; c < 4; ++c)            // c = 2 u + s: chunk 2c + h of a 64-key V^T row
    aV[c] = base + TS_V + 4096 * row + 128 * m + 16 * ((2 * c + h) ^ swz8(m));
  const int ksw = swz4(m);
#pragma unroll
  for (int s = 0; s < 2; ++s) aK[s] = base + TS_K + 4096 * row + 64 * m + 16 * ((2 * s + h) ^ ksw);
  uint32_t aM = base + TS_MASK + 128 * row + 2 * m;
  // opaque to the optimizer: each read is then one address register + an immediate offset
#pragma unroll
  for (int i = 0; i < 8; ++i) asm volatile("" : "+v"(aB[i]));
#pragma unroll
  for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(aV[i]));
  asm volatile("" : "+v"(aK[0]), "+v"(aK[1]), "+v"(aM));

  issue(0, h0, 0);   // the first stage's DMA overlaps the scan below
  // rows whose valid keys are all masked, and the row's first key with a nonzero mask term (masked
  // or padding; N when there is none): tiles of keys before it need no mask (both wave-uniform)
  bool live_l = false;
  int dirty_l = N;
  {
    const op_t* mr = mask16 + ((long)b * N + ip) * N;
    for (int k = lane; k < N; k += 64) {
      const float mv = (float)mr[k];
      live_l |= k < n_valid && mv != -INFINITY;
      if (mv != 0.f) dirty_l = min(dirty_l, k);
    }
  }
  const bool live = __ballot(live_l) != 0;
#pragma unroll
  for (int sh = 32; sh >= 1; sh >>= 1) dirty_l = min(dirty_l, __shfl_xor(dirty_l, sh));
  const int first_dirty = __builtin_amdgcn_readfirstlane(dirty_l);

  const uint32_t ONE = half_bits((op_t)1.f);
  const uint32_t lo_half = h ? 0u : ~0u;   // keeps a value in lanes 0-31, zero in 32-63
  // the rank-1 operands are 4-register tuples whose words 1..3 stay zero: only word 0 changes
  // ([-m, 1] of the block's reference in fb, [1, mask] of the key half in ra), half 1 of the
  // wave holds zero
  u32x4 fb = {0u, 0u, 0u, 0u}, ra = {0u, 0u, 0u, 0u};
  auto set_fb = [&](float mv) PF_INLINE {
    fb[0] = h ? 0u : (half_bits((op_t)(-mv)) | ONE << 16);
    asm volatile("" : "+v"(fb));
  };

  const int jq0 = jw0 + 32 * qb;   // first query of this wave's block; blocks past N idle
  const bool qvalid = jq0 < N;
  opx8 qf[2], qn[2];   // this head's Q fragments, the next head's (loaded a step ahead)
  f32x16 o;
  float mh, lsum;
  uint64_t mset;   // lane mask: the queries (lanes) that have a reference maximum
  bool useref;     // some query's reference is nonzero (wave-uniform)
  auto q_fetch = [&](int hd) PF_INLINE {
    const int jq = min(jq0, N - 32);
    const op_t* qptr = Q + ((((long)b * N + ip) * H + hd) * N + jq + m) * D + 8 * h;
#pragma unroll
    for (int s = 0; s < 2; ++s) qn[s] = ld_x8(qptr + 16 * s);
  };
  auto head_start = [&]() PF_INLINE {
    o = zero16();
    lsum = 0.f;
    mh = 0.f;
    mset = 0;
    useref = false;
    set_fb(0.f);
  };
  // P = exp2(S') packed into the two P.V operands; returns the lane's row sum
  auto exp_pack = [&](const f32x16& sc, u32x4 (&pf)[2]) PF_INLINE {
    float ls[2] = {0.f, 0.f};   // two partial sums: half as long a v_dot2 chain
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int t2 = 0; t2 < 8; t2 += 2) {
        opx2 pk;
        pk[0] = (op_t)exp2_fast(sc[8 * ks + t2]);
        pk[1] = (op_t)exp2_fast(sc[8 * ks + t2 + 1]);
        ls[ks] = dot2_ones(pk, ls[ks]);
        pf[ks][t2 >> 1] = __builtin_bit_cast(uint32_t, pk);
      }
    return ls[0] + ls[1];
  };
  // One step (stage STG) of a live row: the block's two 32x32 tiles (key halves u) one after the
  // other: scores (bias as the accumulator start, K.Q^T, the mask / reference fold), the softmax
  // against the current reference, one check, and the two P.V MFMAs.  When the check fails (a query
  // without a reference -- a head's first tile -- that does not accept 0, or a tile row sum above
  // LSTEP_MAX) the reference moves to the tile's maximum first; the next tile's scores already use the new reference.
  auto step2 = [&](auto stg, int kb0) PF_INLINE {
    constexpr int STG = decltype(stg)::value;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      f32x16 sc;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 bv = lds_rd4f(aB[4 * u + g] + STG * TB_STAGE);
#pragma unroll
        for (int e = 0; e < 4; ++e) sc[4 * g + e] = bv[e];
      }
      // every fragment of the tile is read before the first MFMA (one LDS round trip, and the
      // P.V operands are not behind the rescale branch)
      const opx8 k0 = lds_rd8(aK[0] + STG * TK_STAGE + 2048 * u), k1 = lds_rd8(aK[1] + STG * TK_STAGE + 2048 * u);
      const opx8 v0 = lds_rd8(aV[2 * u] + STG * TV_STAGE), v1 = lds_rd8(aV[2 * u + 1] + STG * TV_STAGE);
      // raised issue priority while the wave issues its score MFMAs, so a wave that has its
      // operands gets the MFMA pipe ahead of the others' exponentials (2-3 % at N = 512)
      __builtin_amdgcn_s_setprio(2);
      sc = mfma32(k0, qf[0], sc);
      sc = mfma32(k1, qf[1], sc);
      if (useref || kb0 + 32 * u + 32 > first_dirty) {
        // every lane reads its key's mask entry (an in-bounds address for all lanes; half 1
        // discards it)
        ra[0] = (ONE | lds_rd16(aM + STG * TM_STAGE + 64 * u) << 16) & lo_half;
        asm volatile("" : "+v"(ra));
        sc = mfma32(as_x8(ra), as_x8(fb), sc);
      }
      __builtin_amdgcn_s_setprio(0);
      u32x4 pf[2];
      float l = exp_pack(sc, pf);
      // the lane masks come straight from v_cmp (a bool ballot would materialize and re-test
      // each lane's predicate); every lane is active here (a live row's valid query block)
      uint64_t bad = __builtin_amdgcn_fcmpf(l, LSTEP_MAX, 2 /* ordered > */);
      if (~mset != 0) {   // a head's first tile (or no unmasked key yet): 0 will do as the reference
        bad |= ~mset & __builtin_amdgcn_fcmpf(l, LSTEP_MIN, 12 /* unordered or < */);
        if (bad == 0) mset = ~0ull;
      }
      if (bad != 0) {
        float mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sc[r]);
        mx = xor32_max(mx);
        const bool ms = (mset >> lane) & 1;
        const float d = ms ? (mx > RESCALE_SLACK ? mx : 0.f) : (mx == -INFINITY ? 0.f : mx);
        const float mnew = (float)(op_t)(mh + d);
        const float dsub = mnew - mh;
        const float alpha = ms ? exp2_fast(-dsub) : 1.f;
        lsum *= alpha;
#pragma unroll
        for (int r = 0; r < 16; ++r) o[r] *= alpha;
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[r] -= dsub;
        l = exp_pack(sc, pf);
        mset |= __builtin_amdgcn_fcmpf(mx, -INFINITY, 14 /* unordered or != */);
        mh = mnew;
        useref = __builtin_amdgcn_fcmpf(mnew, 0.f, 14 /* unordered or != */) != 0;
        set_fb(mnew);
      }
      lsum += l;
      o = mfma32(v0, as_x8(pf[0]), o);
      o = mfma32(v1, as_x8(pf[1]), o);
    }
  };
  auto finalize = [&](int hd) PF_INLINE {
    if (!qvalid) return;
    const float inv = rcp_fast(xor32_sum(lsum));
    const int j = jq0 + m;
    const long rowbase = ((long)b * N + ip) * H;
    if (OUT_F32) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = o[4 * g + e] * inv;
        *reinterpret_cast<f32x4*>(O32 + ((rowbase + hd) * N + j) * D + 8 * g + 4 * h) = v;
      }
    } else {
      store_runs16(O16 + (((long)b * N + ip) * N + j) * C + 32 * hd, o, inv, h);   // 16-byte runs
    }
  };

  // Step loop: T steps (T = 4 N / 64, even), one barrier each (the loop-top wait + barrier),
  // the DMA of the next step into the other stage; during a head's last step the next head's
  // Q is loaded (it lands by the next loop-top wait).  The barrier also tells every wave that
  // the other stage (read in the previous step) is free.
  int kbi = 0, hd = h0;  // step it = (hd - h0) * nKB + kbi
  if (qvalid && live) q_fetch(h0);
  auto one_step = [&](auto stg, int it) PF_INLINE {
    constexpr int STG = decltype(stg)::value;
    __builtin_amdgcn_s_waitcnt(vmcnt_le(0));   // this wave's part of stage STG (and Q) landed ...
    __builtin_amdgcn_s_barrier();              // ... for every wave; stage STG ^ 1 is free
    asm volatile("" ::: "memory");
    if (it + 1 < T) {
      const bool wrap = kbi + 1 == nKB;
      issue(STG ^ 1, wrap ? hd + 1 : hd, wrap ? 0 : 64 * (kbi + 1));
    }
    if (qvalid && live) {
      if (kbi == 0) {
        head_start();
        qf[0] = qn[0];
        qf[1] = qn[1];
      }
      if (kbi == nKB - 1 && hd + 1 < h0 + nh) q_fetch(hd + 1);   // lands by the next step's wait
      step2(stg, 64 * kbi);
      if (kbi == nKB - 1) finalize(hd);
    }
    if (++kbi == nKB) {
      kbi = 0;
      ++hd;
    }
  };
  for (int it = 0; it < T; it += 2) {
    one_step(ic<0>{}, it);
    one_step(ic<1>{}, it + 1);
  }

  // A dead row (every valid key masked): the reference's logits all round to -1e9, so each
  // query's output is the plain mean of v over the n_valid keys, the same for every query of
  // the row.  The row's four query-block waves split its four heads: wave qb sums head qb's
  // V^T (keys stored at perm16 positions) for d = m, the two lane halves taking alternate
  // 16-byte chunks (8 loads in flight, v_dot2 pair sums, keys past n_valid zeroed by
  // selects), and the means meet in LDS.  Every wave takes part in both barriers.
  static_assert(H == TA_WAVES / 4, "one head per query-block wave of a row");
  __syncthreads();   // the last step's stage reads are done before the LDS is reused
  float* smean = reinterpret_cast<float*>(alds);   // [4 rows][H][D]
  if (!live && qb < nh) {
    const int hd2 = h0 + qb;
    const bool all_valid = n_valid >= N;   // wave-uniform
    const op_t* vrow = Vt + ((((long)b * N + ip) * H + hd2) * D + m) * (long)N;
    float acc = 0.f;
    for (int p0 = 8 * h; p0 < N; p0 += 16 * 8) {   // 8 stored keys per 16-byte load
      opx8 v8[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v8[u] = p0 + 16 * u < N ? ld_x8(vrow + p0 + 16 * u) : zero_x8();
#pragma unroll
      for (int u = 0; u < 8; ++u)
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          opx2 pr = {v8[u][e], v8[u][e + 1]};
          if (!all_valid) {
            pr[0] = perm16(p0 + 16 * u + e) < n_valid ? pr[0] : (op_t)0.f;
            pr[1] = perm16(p0 + 16 * u + e + 1) < n_valid ? pr[1] : (op_t)0.f;
          }
          acc = dot2_ones(pr, acc);
        }
    }
    const float mean = xor32_sum(acc) / (float)n_valid;   // lanes m and m + 32 both hold d = m
    if (h == 0) smean[(row * H + hd2) * D + m] = mean;
  }
  __syncthreads();
  if (!live && qvalid) {
    const int j = jq0 + m;
    for (int hd2 = h0; hd2 < h0 + nh; ++hd2) {
      const float* mrow = smean + (row * H + hd2) * D;
      if (OUT_F32) {
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4)
          *reinterpret_cast<f32x4*>(O32 + ((((long)b * N + ip) * H + hd2) * N + j) * D + 16 * h + 4 * q4) =
              *reinterpret_cast<const f32x4*>(mrow + 16 * h + 4 * q4);
      } else {
#pragma unroll
        for (int q8 = 0; q8 < 2; ++q8) {
          opx8 v;
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = (op_t)mrow[16 * h + 8 * q8 + e];
          st_x8(O16 + (((long)b * N + ip) * N + j) * C + 32 * hd2 + 16 * h + 8 * q8, v);
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------------
// Output projection (pf_direct.h): z[pair(i, j)] (+)= linear_o(O[i, j] * sigmoid(linear_g(LN(z[pair])))).
// 8 waves walk groups of 64 frame positions (ip, j0 .. j0 + 63); wave w owns head w >> 1 of the gate
// and the output channels 32 (w >> 1) .. + 31 (c_z = 64: two of the four) of the positions
// 32 (w & 1) .. + 31, its rows of W_g and W_o in registers.  The gate comes out of
// D[channel][position] = W_g . LN(z), o * sigmoid(g) goes through LDS as the B operand of
// D[out][position] = W_o . (o * g), and the residual is loaded in the accumulator's order.
// FAST (the fast mode's block-fp8 points): W_g comes as MXFP8, and g (per head: one 32-channel
// block, a lane pair's 16 + 16 registers) and the projection's output (per 32 output channels) are
// quantize-dequantized before the sigmoid and before the residual.
// Against weights resident in LDS with one wave per tile (us a launch): N = 128 19.6 -> 12.4, 384
// 61 -> 50, 512 96 -> 87, 1024 342 -> 300.
// ---------------------------------------------------------------------------------
constexpr int TAO_WAVES = 8;
template <int CC>
constexpr size_t tao_lds() {
  return (size_t)(2 * DP_ROWS * (CC + 8) + DP_ROWS * (C + 8) + TAO_WAVES * 32 * (C + 8)) * sizeof(op_t) +
         C * sizeof(float);
}

// resid: 0 -> out = update; 1 -> out = z_in + update (out may alias z_in); 2 -> out += update
// HILO: W_g and W_o come with their residuals (rounded to op_t), and both products run on hi + lo
// (two MFMAs per fragment): weights good to ~2^-22 of their size instead of the 2^-12 of one 16-bit
// rounding.  The gate's offsets use hi + lo.
template <int CC, bool FAST, bool HILO = false>
__global__ __launch_bounds__(64 * TAO_WAVES, 1) void ta_out_kernel(
    const op_t* __restrict__ O, const float* z_in, float* out, const float* __restrict__ lnw,
    const float* __restrict__ lnb, TaWeights tw, const op_t* __restrict__ wo, int ngroups, int N, int ending,
    int resid, float eps) {
  constexpr int LW = CC + 8, LO_ = C + 8, KS = CC / 16;
  extern __shared__ __attribute__((aligned(16))) op_t tlds[];
  op_t* sx = tlds;                            // normalized positions [2][64][LW]
  op_t* sog = sx + 2 * DP_ROWS * LW;          // o * sigmoid(g) [64][C + 8]
  op_t* wbuf = sog + DP_ROWS * LO_;           // the waves' weight buffers [8][32][C + 8]
  float* soff = reinterpret_cast<float*>(wbuf + TAO_WAVES * 32 * LO_);   // W_g beta (times -log2(e) unless FAST)
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, m = lane & 31;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tile = wid & 1, cb = wid >> 1;
  const bool has_out = 32 * cb < CC;
  auto group = [&](int g) PF_INLINE -> PosTile { return pos_tile(2u * g, N); };
  auto zpair = [&](const PosTile& pt, int c) PF_INLINE -> long {
    return ((long)pt.b * N + (ending ? pt.c0 + c : pt.r)) * N + (ending ? pt.r : pt.c0 + c);
  };
  DirectLn<CC, TAO_WAVES> ln;
  opx4 ov[4];   // O of channels 32 cb + 8 g + 4 h .. + 3 of position 32 tile + m
  auto fetch = [&](int g) PF_INLINE {
    const PosTile pt = group(g);
    ln.load(z_in, [&](int c) PF_INLINE -> long { return zpair(pt, c); }, wid, lane);
    const op_t* src = O + ((long)DP_ROWS * g + 32 * tile + m) * C + 32 * cb + 4 * h;
#pragma unroll
    for (int gg = 0; gg < 4; ++gg) ov[gg] = ld_x4(src + 8 * gg);
  };
  fetch(blockIdx.x);
  ln.load_gamma(lnw, lane);
  DirectW<CC> wg, wgl;
  DirectW<C> wo_, wol;
  DirectW8<CC> wg8;
  if constexpr (FAST)
    wg8.load((const uint8_t*)tw.w[3] + 32l * cb * CC, (const uint8_t*)tw.s[3] + 32 * cb * (CC / 32), lane);
  else
    wg.load((const op_t*)tw.w[3] + 32l * cb * CC, lane);
  const long or0 = has_out ? 32l * cb * C : 0;
  wo_.load(wo + or0, lane);
  if constexpr (HILO) {
    wgl.load(tw.g_lo + 32l * cb * CC, lane);
    wol.load(tw.o_lo + or0, lane);
  }
  __builtin_amdgcn_sched_barrier(0);
  {
    op_t* wb = wbuf + wid * 32 * LO_;
    if constexpr (FAST)
      wg8.dequant(wg);
    else
      wg.turn(wb, lane);
    wo_.turn(wb, lane);
    float c0 = direct_wbeta<KS>(wg.v, lnb, h);
    if constexpr (HILO) {
      wgl.turn(wb, lane);
      wol.turn(wb, lane);
      c0 += direct_wbeta<KS>(wgl.v, lnb, h);
    }
    if (tile == 0 && h == 0) soff[32 * cb + m] = FAST ? c0 : -LOG2E * c0;
  }
  int buf = 0;
  for (int gi = blockIdx.x; gi < ngroups; gi += gridDim.x, buf ^= 1) {
    const PosTile pt = group(gi);
    op_t* sxb = sx + buf * DP_ROWS * LW;
    ln.store(sxb, eps, wid, lane);
    const long zp = zpair(pt, 32 * tile + m);
    const int oc = 32 * cb + 4 * h;   // + 8 g: this lane's output channels
    f32x4 res[4];
#pragma unroll
    for (int g = 0; g < 4; ++g)
      res[g] = resid && has_out ? *reinterpret_cast<const f32x4*>((resid == 2 ? out : z_in) + zp * CC + oc + 8 * g)
                                : f32x4{0.f, 0.f, 0.f, 0.f};
    opx4 o4[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) o4[g] = ov[g];
    __syncthreads();   // every z row of the group has been read (out may alias z_in)
    if (gi + (int)gridDim.x < ngroups) fetch(gi + gridDim.x);
    f32x16 g16 = zero16();
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const opx8 xf = ld_x8(sxb + (32 * tile + m) * LW + 16 * s + 8 * h);
      g16 = mfma32(wg.v[s], xf, g16);   // D[channel][position]
      if constexpr (HILO) g16 = mfma32(wgl.v[s], xf, g16);
    }
    if constexpr (FAST) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 cg = *reinterpret_cast<const f32x4*>(soff + 32 * cb + 8 * g + 4 * h);
#pragma unroll
        for (int e = 0; e < 4; ++e) g16[4 * g + e] += cg[e];
      }
      mx_fake_quant16(g16);
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      opx4 og;
      const f32x4 cg = *reinterpret_cast<const f32x4*>(soff + 32 * cb + 8 * g + 4 * h);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float ex = FAST ? -LOG2E * g16[4 * g + e] : fmaf(g16[4 * g + e], -LOG2E, cg[e]);
        og[e] = (op_t)((float)o4[g][e] * rcp_fast(1.f + exp2_fast(ex)));
      }
      st_x4(sog + (32 * tile + m) * LO_ + 32 * cb + 8 * g + 4 * h, og);
    }
    __syncthreads();
    if (has_out) {
      f32x16 acc = zero16();
#pragma unroll
      for (int s = 0; s < C / 16; ++s) {
        const opx8 of = ld_x8(sog + (32 * tile + m) * LO_ + 16 * s + 8 * h);
        acc = mfma32(wo_.v[s], of, acc);   // D[out][position]
        if constexpr (HILO) acc = mfma32(wol.v[s], of, acc);
      }
      if constexpr (FAST) mx_fake_quant16(acc);
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = res[g][e] + acc[4 * g + e];
        *reinterpret_cast<f32x4*>(out + zp * CC + oc + 8 * g) = v;
      }
    }
  }
}

// Layout conversion for the standalone attention core (fp32 API tensors -> kernel layout).
// A workgroup takes 64 keys of one (b, i, h) sequence: q / k as 8-value runs per thread
// (coalesced 32-byte loads, 16-byte stores), v through an LDS transpose so that every V^T row
// (d) leaves as 16-byte runs of 8 stored keys.
constexpr int PREP_KB = 64;
__global__ __launch_bounds__(256) void ta_prep_qkv_kernel(const float* __restrict__ q, const float* __restrict__ k,
                                                          const float* __restrict__ v, float qs,
                                                          op_t* __restrict__ Q, op_t* __restrict__ K,
                                                          op_t* __restrict__ Vt, int N) {
  __shared__ op_t sV[D][PREP_KB + 8];   // [d][key within the block], rows 16 bytes longer
  const int nb = N / PREP_KB;
  const long r = blockIdx.x / nb;                       // sequence (b, i, h)
  const int j0 = (int)(blockIdx.x - r * nb) * PREP_KB;
  const int tid = threadIdx.x, jl = tid >> 2, d0 = (tid & 3) * 8;
  const long e = (r * N + j0 + jl) * D + d0;           // element (key j0 + jl, d0) of q / k / v
  const f32x4 q0 = *reinterpret_cast<const f32x4*>(q + e), q1 = *reinterpret_cast<const f32x4*>(q + e + 4);
  const f32x4 k0 = *reinterpret_cast<const f32x4*>(k + e), k1 = *reinterpret_cast<const f32x4*>(k + e + 4);
  const f32x4 v0 = *reinterpret_cast<const f32x4*>(v + e), v1 = *reinterpret_cast<const f32x4*>(v + e + 4);
  opx8 oq, ok;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    oq[u] = (op_t)(q0[u] * qs);
    oq[4 + u] = (op_t)(q1[u] * qs);
    ok[u] = (op_t)k0[u];
    ok[4 + u] = (op_t)k1[u];
    sV[d0 + u][jl] = (op_t)v0[u];
    sV[d0 + 4 + u][jl] = (op_t)v1[u];
  }
  st_x8(Q + e, oq);
  st_x8(K + e, ok);
  __syncthreads();
  // V^T row d = tid / 8, stored positions 8 c .. 8 c + 7 hold keys perm16(8 c + i) (perm16 is
  // its own inverse and keeps every 16-key group in place)
  const int d = tid >> 3, c = tid & 7;
  opx8 ov;
#pragma unroll
  for (int i = 0; i < 8; ++i) ov[i] = sV[d][perm16(8 * c + i)];
  st_x8(Vt + (r * D + d) * N + j0 + 8 * c, ov);
}

__global__ void ta_prep_bias_kernel(const float* __restrict__ bias, const float* __restrict__ mask,
                                    float* __restrict__ bias32, op_t* __restrict__ mask16,
                                    long nbias, long nmask, int N, int n_valid) {
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < nbias; e += (long)gridDim.x * blockDim.x) {
    bias32[e] = fmaf(bias[e], LOG2E, REF_SHIFT);
    if (e < nmask) mask16[e] = mask_term((int)(e % N) >= n_valid, mask ? mask[e] : 1.f);
  }
}

struct TaBuffers {
  op_t *Q, *K, *Vt, *O;
  float* bias32;
  op_t* mask16;
  float* stats;   // the mean-correction partials
};

// Workspace: Q, K, V^T, O (op_t, [B][N][H][N][D] each), the fp32 bias [B][H][N][N], the op_t
// mask term [B][N][N].
size_t ta_buffers_size(int B, int N) {
  const size_t e = (size_t)B * N * H * N * D;
  const size_t bytes = 4 * e * sizeof(op_t) + (size_t)B * H * N * N * sizeof(float) + (size_t)B * N * N * sizeof(op_t);
  return (bytes + 15) / 16 * 16 + PS_PARTIAL_FLOATS * sizeof(float);   // + the mean-correction partials
}

TaBuffers ta_buffers(void* ws, int B, int N) {
  const size_t e = (size_t)B * N * H * N * D;
  TaBuffers t;
  t.Q = (op_t*)ws;
  t.K = t.Q + e;
  t.Vt = t.K + e;
  t.O = t.Vt + e;
  t.bias32 = reinterpret_cast<float*>(t.O + e);
  t.mask16 = reinterpret_cast<op_t*>(t.bias32 + (size_t)B * H * N * N);
  const size_t used = (size_t)((char*)(t.mask16 + (size_t)B * N * N) - (char*)ws);
  t.stats = reinterpret_cast<float*>((char*)ws + (used + 15) / 16 * 16);
  return t;
}

template <bool OUT_F32>
int launch_attn(const TaBuffers& t, float* o32, int B, int N, int n_valid, hipStream_t st) {
  if (const int rc = pf_reserve_lds((const void*)ta_attn_kernel<OUT_F32>, TA_LDS, "ta_attn_kernel")) return rc;
  const int total = B * (N / 4) * ((N + 127) / 128);
  // the blocks of a last round (all of them when the launch is one round or less) that would fill
  // at most half of the CUs run split over 2 or 4 workgroups, H / split heads each: the largest
  // split whose workgroups still fit on the chip
  const int cus = device_cus();
  const int rest = cus <= 0 ? 0 : total > cus ? total % cus : total;
  // (the kernel takes its H / split * N / 64 steps in pairs, one per ring stage: a single-head
  // split needs an even N / 64)
  int split = 1;
  while (split < 4 && rest > 0 && 2 * split * rest <= cus && !(split == 2 && (N / 64) % 2)) split *= 2;
  const int full = split > 1 ? total - rest : total;
  static_assert(H % 4 == 0, "head splits of 2 and 4");
  pf_attend_mark(st, 0);
  ta_attn_kernel<OUT_F32><<<full + split * (total - full), 64 * TA_WAVES, TA_LDS, st>>>(
      t.Q, t.K, t.Vt, t.bias32, t.mask16, t.O, o32, N, n_valid, total, full, split > 1 ? split : 2);
  PF_CHECK_LAUNCH("ta_attn_kernel");
  pf_attend_mark(st, 1);
  return PF_OK;
}

// The residuals of ta_proj's weights for a 16-bit call with the exact offsets and the four
// folded-weight residuals, one batch element, c_z = 128 (else the plain W16): a second MFMA up to
// four groups of 64 positions per CU when W_g and W_o come with theirs too, where the statistics
// launch costs more (whole attention, us, against the weights in LDS it replaced: N = 64 48 -> 27,
// 128 55 -> 37, 256 84 -> 81), else the mean correction (384 189 -> 168, 1024 1785 -> 1622).
template <int CC, bool FAST, int LO>
int triatt_run_lo(const pf_triatt_args* a, const TaWeights& w, const TaBuffers& t, const TaMeanFix& mf, int cus) {
  hipStream_t st = (hipStream_t)a->stream;
  const int B = a->B, N = a->N;
  const int n_valid = a->n_valid ? a->n_valid : N;
  const float qscale = LOG2E / sqrtf((float)D);
  const int ngroups = (int)((long)B * N * N / DP_ROWS), grid = min(ngroups, cus);
  {
    auto kern = ta_proj_kernel<CC, FAST, LO>;
    if (const int rc = pf_reserve_lds((const void*)kern, tap_lds<CC>(), "ta_proj_kernel")) return rc;
    kern<<<grid, 64 * TAP_WAVES, tap_lds<CC>(), st>>>(a->z_in, a->pair_mask, a->ln_w, a->ln_b, w,
                                                      (const op_t*)a->w_bias, t.Q, t.K, t.Vt, t.bias32, t.mask16,
                                                      ngroups, N, n_valid, a->ending, qscale, a->eps, mf);
    PF_CHECK_LAUNCH("ta_proj_kernel");
  }
  int rc = launch_attn<false>(t, nullptr, B, N, n_valid, st);
  if (rc) return rc;
  const int resid = !a->accumulate ? 0 : (a->out == a->z_in ? 1 : 2);
  constexpr bool CAN_HILO = !FAST && CC == 128;   // the residual weights exist for the 16-bit c_z = 128 path
  auto kern = CAN_HILO && w.g_lo && w.o_lo ? ta_out_kernel<CC, FAST, CAN_HILO> : ta_out_kernel<CC, FAST, false>;
  if (const int rc = pf_reserve_lds((const void*)kern, tao_lds<CC>(), "ta_out_kernel")) return rc;
  kern<<<grid, 64 * TAO_WAVES, tao_lds<CC>(), st>>>(t.O, a->z_in, a->out, a->ln_w, a->ln_b, w, (const op_t*)a->w_o,
                                                    ngroups, N, a->ending, resid, a->eps);
  PF_CHECK_LAUNCH("ta_out_kernel");
  return PF_OK;
}

template <int CC, bool FAST>
int triatt_run(const pf_triatt_args* a, const TaWeights& w) {
  const TaBuffers t = ta_buffers(a->workspace, a->B, a->N);
  const int cus = device_cus();
  if (cus <= 0) return pf_fail(PF_E_LAUNCH, "pf_triatt_fwd: cannot query the device");
  TaMeanFix mf{nullptr, {nullptr, nullptr, nullptr, nullptr}, nullptr};
  if constexpr (!FAST && CC == PS_C) {
    mf.offb = a->in_offsets;
    if (a->in_offsets && a->B == 1 && a->w_q_lo && a->w_k_lo && a->w_v_lo && a->w_bias_lo) {
      mf.lo[0] = (const op_t*)a->w_q_lo; mf.lo[1] = (const op_t*)a->w_k_lo;
      mf.lo[2] = (const op_t*)a->w_v_lo; mf.lo[3] = (const op_t*)a->w_bias_lo;
      if (w.g_lo && w.o_lo && (long)a->N * a->N / DP_ROWS <= 4l * cus)
        return triatt_run_lo<CC, FAST, DL_MFMA>(a, w, t, mf, cus);
      mf.stats = t.stats;
      pair_stats_kernel<<<PS_WG, 64 * PS_WAVES, 0, (hipStream_t)a->stream>>>(a->z_in, a->N, a->eps, t.stats);
      PF_CHECK_LAUNCH("pair_stats_kernel");
      return triatt_run_lo<CC, FAST, DL_MEAN>(a, w, t, mf, cus);
    }
  }
  return triatt_run_lo<CC, FAST, DL_NONE>(a, w, t, mf, cus);
}

// The attention kernel addresses a batch's bias ([H][N][N] fp32) through one raw buffer
// resource, whose range is below 2^31 bytes.
bool ta_shape_ok(int N) { return (long)H * N * N * 4 < (1l << 31); }

}  // namespace

// ---------------------------------------------------------------------------------
// C-ABI
// ---------------------------------------------------------------------------------
extern "C" size_t pf_triatt_workspace_size(int B, int N, int C_, int H_, int D_) {
  if (B <= 0 || N <= 0 || (C_ != 128 && C_ != 64) || H_ != H || D_ != D) return 0;
  return ta_buffers_size(B, N);
}

extern "C" int pf_triatt_fwd(const pf_triatt_args* a) {
  if (!a) return pf_fail(PF_E_INVALID, "pf_triatt_fwd: null args");
  if ((a->C != 128 && a->C != 64) || a->H != H || a->D != D)
    return pf_fail(PF_E_INVALID, "pf_triatt_fwd: only C = 128 or 64, H=4, D=32 supported (got C=%d H=%d D=%d)",
                   a->C, a->H, a->D);
  if (a->B <= 0 || a->N <= 0 || a->N % 64)
    return pf_fail(PF_E_INVALID, "pf_triatt_fwd: need B > 0 and N a positive multiple of 64 (B=%d N=%d)", a->B, a->N);
  if ((unsigned long long)a->B * a->N * a->N >= (1ull << 32) || !ta_shape_ok(a->N))
    return pf_fail(PF_E_INVALID, "pf_triatt_fwd: need B * N * N < 2^32 and N <= 11584 (B=%d N=%d)", a->B, a->N);
  if (!a->z_in || !a->out || !a->ln_w || !a->ln_b || !a->w_bias || !a->w_q || !a->w_k ||
      !a->w_v || !a->w_g || !a->w_o || !a->workspace)
    return pf_fail(PF_E_INVALID, "pf_triatt_fwd: null pointer argument");
  const size_t need = ta_buffers_size(a->B, a->N);
  if (a->workspace_bytes < need)
    return pf_fail(PF_E_INVALID, "pf_triatt_fwd: workspace too small (%zu < %zu bytes)", a->workspace_bytes, need);
  if (a->n_valid < 0 || a->n_valid > a->N)
    return pf_fail(PF_E_INVALID, "pf_triatt_fwd: n_valid %d outside [0, N=%d]", a->n_valid, a->N);
  if ((a->w_g_lo != nullptr) != (a->w_o_lo != nullptr) || (a->w_g_lo && a->C != 128))
    return pf_fail(PF_E_INVALID, "pf_triatt_fwd: give both weight residuals (w_g_lo, w_o_lo) or neither, C = 128 only");
  {
    const bool any_lo = a->w_q_lo || a->w_k_lo || a->w_v_lo || a->w_bias_lo;
    if ((a->in_offsets || any_lo) && a->C != 128)
      return pf_fail(PF_E_INVALID, "pf_triatt_fwd: exact offsets and the mean correction need C = 128");
    if (any_lo && !(a->in_offsets && a->w_q_lo && a->w_k_lo && a->w_v_lo && a->w_bias_lo))
      return pf_fail(PF_E_INVALID, "pf_triatt_fwd: the mean correction needs in_offsets and all four residuals "
                                   "(w_q_lo, w_k_lo, w_v_lo, w_bias_lo)");
  }
  TaWeights w = {{a->w_q, a->w_k, a->w_v, a->w_g}};
  w.g_lo = (const op_t*)a->w_g_lo;
  w.o_lo = (const op_t*)a->w_o_lo;
  return a->C == 128 ? triatt_run<128, false>(a, w) : triatt_run<64, false>(a, w);
}

// Fast mode: the 16-bit workspace (the size keeps 4 C^2 op_t more, part of the interface).
extern "C" size_t pf_triatt_mx8_workspace_size(int B, int N, int C_, int H_, int D_) {
  if (B <= 0 || N <= 0 || C_ != 128 || H_ != H || D_ != D) return 0;
  return ta_buffers_size(B, N) + 4 * (size_t)C * C * sizeof(op_t);
}

extern "C" int pf_triatt_mx8_fwd(const pf_triatt_mx8_args* m) {
  if (!m) return pf_fail(PF_E_INVALID, "pf_triatt_mx8_fwd: null args");
  if (m->C != 128 || m->H != H || m->D != D)
    return pf_fail(PF_E_INVALID, "pf_triatt_mx8_fwd: only C = 128, H=4, D=32 supported (got C=%d H=%d D=%d)", m->C,
                   m->H, m->D);
  if (m->B <= 0 || m->N <= 0 || m->N % 64)
    return pf_fail(PF_E_INVALID, "pf_triatt_mx8_fwd: need B > 0 and N a positive multiple of 64 (B=%d N=%d)", m->B,
                   m->N);
  if ((unsigned long long)m->B * m->N * m->N >= (1ull << 32) || !ta_shape_ok(m->N))
    return pf_fail(PF_E_INVALID, "pf_triatt_mx8_fwd: need B * N * N < 2^32 and N <= 11584 (B=%d N=%d)", m->B, m->N);
  if (!m->z_in || !m->out || !m->ln_w || !m->ln_b || !m->w_bias || !m->w_q_q || !m->w_q_s || !m->w_k_q ||
      !m->w_k_s || !m->w_v_q || !m->w_v_s || !m->w_g_q || !m->w_g_s || !m->w_o || !m->workspace)
    return pf_fail(PF_E_INVALID, "pf_triatt_mx8_fwd: null pointer argument");
  const size_t need = pf_triatt_mx8_workspace_size(m->B, m->N, m->C, m->H, m->D);
  if (m->workspace_bytes < need)
    return pf_fail(PF_E_INVALID, "pf_triatt_mx8_fwd: workspace too small (%zu < %zu bytes)", m->workspace_bytes, need);
  if (m->n_valid < 0 || m->n_valid > m->N)
    return pf_fail(PF_E_INVALID, "pf_triatt_mx8_fwd: n_valid %d outside [0, N=%d]", m->n_valid, m->N);
  pf_triatt_args a = {};
  a.B = m->B; a.N = m->N; a.C = m->C; a.H = m->H; a.D = m->D;
  a.ending = m->ending; a.accumulate = m->accumulate; a.n_valid = m->n_valid; a.eps = m->eps;
  a.z_in = m->z_in; a.out = m->out; a.pair_mask = m->pair_mask; a.ln_w = m->ln_w; a.ln_b = m->ln_b;
  a.w_bias = m->w_bias; a.w_o = m->w_o;
  a.workspace = m->workspace; a.workspace_bytes = m->workspace_bytes; a.stream = m->stream;
  const TaWeights w = {{m->w_q_q, m->w_k_q, m->w_v_q, m->w_g_q}, {m->w_q_s, m->w_k_s, m->w_v_s, m->w_g_s}};
  return triatt_run<128, true>(&a, w);
}

extern "C" int pf_triatt_attend_workspace(void* workspace, size_t workspace_bytes, int B, int N, int n_valid,
                                          void* stream) {
  if (!workspace) return pf_fail(PF_E_INVALID, "pf_triatt_attend_workspace: null workspace");
  if (B <= 0 || N <= 0 || N % 64)
    return pf_fail(PF_E_INVALID, "pf_triatt_attend_workspace: need B > 0 and N a positive multiple of 64");
  if ((unsigned long long)B * N * N >= (1ull << 32) || !ta_shape_ok(N))
    return pf_fail(PF_E_INVALID, "pf_triatt_attend_workspace: need B * N * N < 2^32 and N <= 11584 (B=%d N=%d)",
                   B, N);
  if (n_valid < 0 || n_valid > N)
    return pf_fail(PF_E_INVALID, "pf_triatt_attend_workspace: n_valid %d outside [0, N=%d]", n_valid, N);
  const size_t need = ta_buffers_size(B, N);
  if (workspace_bytes < need)
    return pf_fail(PF_E_INVALID, "pf_triatt_attend_workspace: workspace too small (%zu < %zu bytes)",
                   workspace_bytes, need);
  return launch_attn<false>(ta_buffers(workspace, B, N), nullptr, B, N, n_valid ? n_valid : N, (hipStream_t)stream);
}

extern "C" size_t pf_tri_attention_workspace_size(int B, int N, int H_, int D_) {
  if (B <= 0 || N <= 0 || H_ != H || D_ != D) return 0;
  return ta_buffers_size(B, N);
}

extern "C" int pf_tri_attention(const float* q, const float* k, const float* v, const float* bias,
                                const float* mask, float scale, float* o, int B, int N, int H_, int D_,
                                int n_valid, void* workspace, size_t workspace_bytes, void* stream) {
  if (H_ != H || D_ != D)
    return pf_fail(PF_E_INVALID, "pf_tri_attention: only H=4, D=32 supported (got H=%d D=%d)", H_, D_);
  if (B <= 0 || N <= 0 || N % 64)
    return pf_fail(PF_E_INVALID, "pf_tri_attention: need B > 0 and N a positive multiple of 64 (B=%d N=%d)", B, N);
  if ((unsigned long long)B * N * N >= (1ull << 32) || !ta_shape_ok(N))
    return pf_fail(PF_E_INVALID, "pf_tri_attention: need B * N * N < 2^32 and N <= 11584 (B=%d N=%d)", B, N);
  if (n_valid < 0 || n_valid > N)
    return pf_fail(PF_E_INVALID, "pf_tri_attention: n_valid %d outside [0, N=%d]", n_valid, N);
  if (n_valid == 0) n_valid = N;
  if (!q || !k || !v || !bias || !o || !workspace)
    return pf_fail(PF_E_INVALID, "pf_tri_attention: null pointer argument");
  const size_t need = ta_buffers_size(B, N);
  if (workspace_bytes < need)
    return pf_fail(PF_E_INVALID, "pf_tri_attention: workspace too small (%zu < %zu bytes)", workspace_bytes, need);
  hipStream_t st = (hipStream_t)stream;
  TaBuffers t = ta_buffers(workspace, B, N);
  const long rows = (long)B * N * H;
  ta_prep_qkv_kernel<<<(unsigned)(rows * (N / PREP_KB)), 256, 0, st>>>(q, k, v, scale * LOG2E, t.Q, t.K, t.Vt, N);
  PF_CHECK_LAUNCH("ta_prep_qkv_kernel");
  ta_prep_bias_kernel<<<1024, 256, 0, st>>>(bias, mask, t.bias32, t.mask16, (long)B * H * N * N, (long)B * N * N,
                                            N, n_valid);
  PF_CHECK_LAUNCH("ta_prep_bias_kernel");
  return launch_attn<true>(t, o, B, N, n_valid, st);
}
