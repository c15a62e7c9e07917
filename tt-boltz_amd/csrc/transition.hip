// Transition (SwiGLU MLP) and row primitives for gfx950.
//
//   tr_pair_kernel   Pair transition, C = 128: LN -> fc1|fc2 (MFMA, transposed
//                    orientation) -> silu(a)*b in registers -> fc3 (MFMA) -> residual.
//                    The 4C hidden activations never leave the CU.  fc1/fc2 rows are
//                    staged in LDS perm16-permuted so the fc1/fc2 accumulator registers
//                    come out in the natural k order of fc3's B operand.  Everything is in
//                    the output-aligned layout (pf_common.h): fc3 yields D[channel][pair],
//                    so a lane owns one pair and writes 16-byte runs, and the residual is
//                    fetched with 16-byte loads, all issued before the first store.  Weight
//                    blocks arrive by LDS DMA (layout at the kernel).  fc3's rounding
//                    residual enters as a second MFMA or through a sampled mean
//                    correction (TrMode below).
//                    Replaces Transition.forward (tt_bio/boltz2.py:1227-1258) and the ttnn
//                    Transition (tt_bio/tenstorrent.py:856-946).
//   ln_rows_kernel   LayerNorm over rows, any C (nn.LayerNorm / tt_bio/boltz2.py:738-768).
//   linear_rows_kernel  out = resid + x W^T + bias, optional SwiGLU pairing of two weight
//                    matrices (tt_bio/boltz2.py:638-731); fp32 in/out, MFMA inside.
//   pair_ln_linear_kernel  out = base + W LN(x) for C = 128 rows (trunk recycling step).
#include "pf_common.h"
#include "pf_direct.h"
#include "pf_internal.h"

namespace {

constexpr int C = 128, LDSW = 136;
PF_DEV opx8 lds_x8(const char* p) { return *reinterpret_cast<const opx8*>(p); }

// Pair transition: a workgroup is TRW waves x 32 pairs; three workgroups share a CU.
// Weight blocks of 32 hidden units move global -> LDS by DMA (global_load_lds) into a
// 2-stage ring, one barrier per block:
//   W1 / W2 block: LDS row R (0..31) holds hidden unit 32 hb + perm16(R) (so the fc1/fc2
//                  accumulator rows come out in fc3's k order); 16 chunks of 8 channels,
//                  chunk c at slot c ^ (R & 15)
//   W3 block:      row R (output channel 0..127) holds hidden 32 hb .. 32 hb + 31; 4
//                  chunks, chunk c at slot c ^ swz4(R)
// so every fragment read (one 16-byte chunk from each of 32 consecutive rows) is free of
// bank conflicts.
// The output projection fc3 comes in four forms (TrMode):
//   TR_PLAIN    fc3_16 only.
//   TR_HILO     fc3 also comes with its rounding residual w3_lo = fc3 - fc3_16 (op_t), staged
//               as a fourth block beside W3 and multiplied in as a second MFMA per fragment, so
//               the projection runs on weights good to ~2^-22 of their size; the larger ring
//               leaves room for two workgroups per CU instead of three.
//   TR_MEANFIX  fc3_16, plus corr = w3_lo . mean(h) on every output row: the part of the
//               residual's error that every position shares, h the hidden activation
//               silu(fc1 x) * fc2 x averaged over sampled positions (below).
//   TR_STATS    the sampling pass behind corr: a workgroup of 4 waves takes 4 sampled tiles of
//               32 pairs (Fibonacci hashing, as pair_stats_kernel) and two of the hidden blocks
//               (both fetched at once, before the LayerNorm: the pass is latency-bound),
//               multiplies their h by w3_lo (given as w3) and sums over its pairs into one
//               partial per workgroup (already divided by the sample size).
enum TrMode { TR_PLAIN = 0, TR_HILO = 1, TR_MEANFIX = 2, TR_STATS = 3 };
constexpr int TRW = 4;                       // waves of a workgroup
constexpr int TR_BLK = 8192;                 // bytes of one fp16 weight block
#ifndef PF_TRS_TILES
#define PF_TRS_TILES 256
#endif
constexpr int TRS_TILES = PF_TRS_TILES;      // sampled tiles of the TR_STATS pass
constexpr int TRS_MAX_HIDDEN = 512;          // its hidden sizes: multiples of 64 up to this
constexpr int TRS_PARTIALS = TRS_TILES / TRW * (TRS_MAX_HIDDEN / 64);   // its workgroups (at most)
template <int MODE>
constexpr int tr_stage() { return (MODE == TR_HILO ? 4 : 3) * TR_BLK; }
PF_DEV int tr_swz4(int r) { return (r >> 2) & 3; }

template <bool ZBIAS, int MODE>
__global__ __launch_bounds__(64 * TRW, MODE == TR_HILO || MODE == TR_STATS ? 2 : 3) void tr_pair_kernel(
    const float* x_in, float* out, const float* __restrict__ lnw, const float* __restrict__ lnb,
    const op_t* __restrict__ w1, const op_t* __restrict__ w2, const op_t* __restrict__ w3,
    const op_t* __restrict__ w3_lo, long rows, int hidden, int accumulate, float eps, ZBiasArgs zb,
    const float* __restrict__ corr, float* __restrict__ partials) {
  constexpr bool HILO = MODE == TR_HILO, STATS = MODE == TR_STATS;
  constexpr int STAGE = tr_stage<MODE>();
  __shared__ __attribute__((aligned(16))) char tl[2 * STAGE];
  __shared__ float red[STATS ? 2 * TRW * C : 1];   // the sampling pass's sums
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, m = lane & 31;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nhb = hidden / 32;
  long pos0;
  int hb_lo = 0, hb_hi = nhb;
  bool live = true;
  uint32_t ns = 0;
  if constexpr (STATS) {   // hidden blocks 2 hbg, 2 hbg + 1 of sampled tiles 4 g .. 4 g + 3
    const uint32_t ntiles = (uint32_t)(rows / 32);
    ns = ntiles < (uint32_t)TRS_TILES ? ntiles : (uint32_t)TRS_TILES;
    const int ngroups = nhb / 2, hbg = blockIdx.x % ngroups;
    const uint32_t k = blockIdx.x / ngroups * TRW + wid;
    live = k < ns;   // a dead wave still takes its part in the weight DMA and the barriers
    const uint32_t kk = live ? k : 0;
    pos0 = 32l * (ns == ntiles ? kk : (uint32_t)(((uint64_t)kk * 2654435761ull) % ntiles));
    hb_lo = 2 * hbg;
    hb_hi = hb_lo + 2;
  } else {
    pos0 = ((long)blockIdx.x * TRW + wid) * 32;
  }


  // DMA: chunk e = tid + 256 i (i = 0, 1) of each block; chunk tid + 256 is row R + 16
  // (W1 / W2: same slot, perm16(R + 16) = perm16(R) + 16) or R + 64 (W3: same slot)
  const int R = tid >> 4, R3 = tid >> 2;
  const uint32_t o12 = 2u * (perm16(R) * C + 8 * ((tid & 15) ^ (R & 15)));
  const uint32_t o3 = 2u * (R3 * hidden + 8 * ((tid & 3) ^ tr_swz4(R3)));
  const uint32_t o3b = 2u * 64 * hidden;
  auto issue = [&](int hb, int buf) {
    char* st = tl + buf * STAGE + 1024 * wid;
    const char* b1 = (const char*)(w1 + (long)32 * hb * C);
    const char* b2 = (const char*)(w2 + (long)32 * hb * C);
    const char* b3 = (const char*)(w3 + 32 * hb);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      __builtin_amdgcn_global_load_lds(b1 + o12 + 4096 * i, st + 4096 * i, 16, 0, 0);
      __builtin_amdgcn_global_load_lds(b2 + o12 + 4096 * i, st + TR_BLK + 4096 * i, 16, 0, 0);
      __builtin_amdgcn_global_load_lds(b3 + o3 + o3b * i, st + 2 * TR_BLK + 4096 * i, 16, 0, 0);
      if constexpr (HILO)
        __builtin_amdgcn_global_load_lds((const char*)(w3_lo + 32 * hb) + o3 + o3b * i, st + 3 * TR_BLK + 4096 * i,
                                         16, 0, 0);
    }
  };
  // fragment read addresses: fc1 / fc2 k-step s of row m; fc3 k-step ks of row 32 ob + m
  int a12[8], a3[2];
#pragma unroll
  for (int s2 = 0; s2 < 8; ++s2) a12[s2] = 256 * m + 16 * ((2 * s2 + h) ^ (m & 15));
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) a3[ks] = 2 * TR_BLK + 64 * m + 16 * ((2 * ks + h) ^ tr_swz4(m));

  // the first block (TR_STATS: both) is on its way during the LayerNorm
  issue(hb_lo, 0);
  if constexpr (STATS) issue(hb_lo + 1, 1);
  // rows past the end are clamped on load and skipped on store
  opx8 xf[8];
  {
    float x[64];
    load_row128_frag(x_in + min(pos0 + m, rows - 1) * C, h, x);
    ln128_to_frag(x, h, lnw, lnb, eps, xf);
  }
  f32x16 acc[4];
#pragma unroll
  for (int ob = 0; ob < 4; ++ob) acc[ob] = zero16();
  float cm[4];   // TR_MEANFIX: corr of channels 32 ob + m
  if constexpr (MODE == TR_MEANFIX)
#pragma unroll
    for (int ob = 0; ob < 4; ++ob) cm[ob] = corr[32 * ob + m];

  for (int hb = hb_lo; hb < hb_hi; ++hb) {
    const int buf = (hb - hb_lo) & 1;
    __builtin_amdgcn_s_waitcnt(vmcnt_le(0));   // block hb landed ...
    __builtin_amdgcn_s_barrier();              // ... for every wave; the other stage is free
    asm volatile("" ::: "memory");
    if (!STATS && hb + 1 < hb_hi) issue(hb + 1, buf ^ 1);
    const char* st = tl + buf * STAGE;
    f32x16 a1 = zero16(), a2 = zero16();
#pragma unroll
    for (int s2 = 0; s2 < 8; ++s2) {
      a1 = mfma32(lds_x8(st + a12[s2]), xf[s2], a1);            // rows = hidden (perm16), cols = pairs
      a2 = mfma32(lds_x8(st + TR_BLK + a12[s2]), xf[s2], a2);
    }
    opx8 hf[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int t = 0; t < 8; ++t) hf[ks][t] = (op_t)(siluf(a1[8 * ks + t]) * a2[8 * ks + t]);
#pragma unroll
    for (int ob = 0; ob < 4; ++ob)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        acc[ob] = mfma32(lds_x8(st + a3[ks] + 2048 * ob), hf[ks], acc[ob]);
        if constexpr (HILO) acc[ob] = mfma32(lds_x8(st + TR_BLK + a3[ks] + 2048 * ob), hf[ks], acc[ob]);
      }
  }
  if constexpr (STATS) {
    // sums over each row of 16 lanes (16 pairs) for all 64 values first (independent DPP chains),
    // then one store per row: red[2 wid + row16 parity][channel], the 8 rows summed below
#pragma unroll
    for (int ob = 0; ob < 4; ++ob)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[ob][i] = row16_sum(acc[ob][i]);
    if ((lane & 15) == 0) {
      float* r = red + (2 * wid + ((lane >> 4) & 1)) * C + 4 * h;
#pragma unroll
      for (int ob = 0; ob < 4; ++ob)
#pragma unroll
        for (int i = 0; i < 16; ++i) r[32 * ob + 8 * (i >> 2) + (i & 3)] = live ? acc[ob][i] : 0.f;
    }
    __syncthreads();
    if (tid < C) {
      float sum = 0.f;
#pragma unroll
      for (int w = 0; w < 2 * TRW; ++w) sum += red[w * C + tid];
      partials[blockIdx.x * C + tid] = sum / (32.f * (float)ns);
    }
  } else {
    if constexpr (MODE == TR_MEANFIX) {
      // acc[ob] += corr on every pair, as one more MFMA: A = corr as a 16-bit hi + lo pair in
      // columns k = 0, 1 (row m = channel 32 ob + m, as for W3), B = 1; below the 16-bit
      // normal range the pair keeps corr to ~1e-8 absolute, far under the outputs' scale.
      // Accumulators that started from corr instead would keep a second copy of all 64 across
      // the loop.
      opx8 ones;
#pragma unroll
      for (int t = 0; t < 8; ++t) ones[t] = (op_t)1.f;
#pragma unroll
      for (int ob = 0; ob < 4; ++ob) {
        opx8 a;
#pragma unroll
        for (int t = 0; t < 8; ++t) a[t] = (op_t)0.f;
        const op_t hi = (op_t)(h == 0 ? cm[ob] : 0.f);
        a[0] = hi;
        a[1] = (op_t)(h == 0 ? cm[ob] - (float)hi : 0.f);
        acc[ob] = mfma32(a, ones, acc[ob]);
      }
    }
    pair_update_epilogue<ZBIAS>(acc, out, rows, pos0, m, h, accumulate, zb);
  }
}

// TR_HILO for small grids: a workgroup is 2 tiles of 32 pairs x 2 halves of the hidden units, so the
// serial chain over weight blocks is half as long and there are twice as many workgroups; every half
// has a ring of its own (128 KB in all).  The second half's partial sums meet the first's in LDS.
// us (with the fused pair bias) against the one-chain kernel: N = 64 27.5 -> 22, N = 128 30.5 -> 26.
constexpr size_t TRSP_LDS = 2 * 2 * (size_t)tr_stage<TR_HILO>();
template <bool ZBIAS>
__global__ __launch_bounds__(64 * TRW, 1) void tr_pair_split_kernel(
    const float* x_in, float* out, const float* __restrict__ lnw, const float* __restrict__ lnb,
    const op_t* __restrict__ w1, const op_t* __restrict__ w2, const op_t* __restrict__ w3,
    const op_t* __restrict__ w3_lo, long rows, int hidden, int accumulate, float eps, ZBiasArgs zb) {
  constexpr int STAGE = tr_stage<TR_HILO>();
  extern __shared__ __attribute__((aligned(16))) char tsl[];
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, m = lane & 31;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = wid & 1, tile = wid >> 1;
  const int nhb = hidden / 64, hb0 = half * nhb;   // blocks of this half
  const long pos0 = ((long)blockIdx.x * 2 + tile) * 32;
  char* ring = tsl + half * 2 * STAGE;
  // DMA: chunk e = 64 tile + lane + 128 i (i = 0..3) of each 8 KB block; layout as tr_pair_kernel
  const int e0 = 64 * tile + lane, R3 = e0 >> 2;
  uint32_t o12[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int R = (e0 >> 4) + 8 * i;
    o12[i] = 2u * (perm16(R) * C + 8 * ((e0 & 15) ^ (R & 15)));
  }
  const uint32_t o3 = 2u * (R3 * hidden + 8 * ((e0 & 3) ^ tr_swz4(R3)));   // row R3 + 32 i: same slot
  const uint32_t o3b = 2u * 32 * hidden;
  auto issue = [&](int hb, int buf) {
    char* st = ring + buf * STAGE + 1024 * tile;
    const char* b1 = (const char*)(w1 + (long)32 * hb * C);
    const char* b2 = (const char*)(w2 + (long)32 * hb * C);
    const char* b3 = (const char*)(w3 + 32 * hb);
    const char* b4 = (const char*)(w3_lo + 32 * hb);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      __builtin_amdgcn_global_load_lds(b1 + o12[i], st + 2048 * i, 16, 0, 0);
      __builtin_amdgcn_global_load_lds(b2 + o12[i], st + TR_BLK + 2048 * i, 16, 0, 0);
      __builtin_amdgcn_global_load_lds(b3 + o3 + o3b * i, st + 2 * TR_BLK + 2048 * i, 16, 0, 0);
      __builtin_amdgcn_global_load_lds(b4 + o3 + o3b * i, st + 3 * TR_BLK + 2048 * i, 16, 0, 0);
    }
  };
  int a12[8], a3[2];
#pragma unroll
  for (int s2 = 0; s2 < 8; ++s2) a12[s2] = 256 * m + 16 * ((2 * s2 + h) ^ (m & 15));
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) a3[ks] = 2 * TR_BLK + 64 * m + 16 * ((2 * ks + h) ^ tr_swz4(m));
  issue(hb0, 0);
  opx8 xf[8];
  {   // rows past the end are clamped on load and skipped on store
    float x[64];
    load_row128_frag(x_in + min(pos0 + m, rows - 1) * C, h, x);
    ln128_to_frag(x, h, lnw, lnb, eps, xf);
  }
  f32x16 acc[4];
#pragma unroll
  for (int ob = 0; ob < 4; ++ob) acc[ob] = zero16();
  for (int k = 0; k < nhb; ++k) {
    const int buf = k & 1;
    __builtin_amdgcn_s_waitcnt(vmcnt_le(0));   // the block landed ...
    __builtin_amdgcn_s_barrier();              // ... for every wave; the other stage is free
    asm volatile("" ::: "memory");
    if (k + 1 < nhb) issue(hb0 + k + 1, buf ^ 1);
    const char* st = ring + buf * STAGE;
    f32x16 a1 = zero16(), a2 = zero16();
#pragma unroll
    for (int s2 = 0; s2 < 8; ++s2) {
      a1 = mfma32(lds_x8(st + a12[s2]), xf[s2], a1);            // rows = hidden (perm16), cols = pairs
      a2 = mfma32(lds_x8(st + TR_BLK + a12[s2]), xf[s2], a2);
    }
    opx8 hf[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int t = 0; t < 8; ++t) hf[ks][t] = (op_t)(siluf(a1[8 * ks + t]) * a2[8 * ks + t]);
#pragma unroll
    for (int ob = 0; ob < 4; ++ob)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        acc[ob] = mfma32(lds_x8(st + a3[ks] + 2048 * ob), hf[ks], acc[ob]);
        acc[ob] = mfma32(lds_x8(st + TR_BLK + a3[ks] + 2048 * ob), hf[ks], acc[ob]);
      }
  }
  __syncthreads();   // the rings are read out
  f32x4* part = reinterpret_cast<f32x4*>(tsl) + tile * 16 * 64 + lane;   // [tile][16][64 lanes]
  if (half == 1) {
#pragma unroll
    for (int q = 0; q < 16; ++q)
      part[64 * q] = f32x4{acc[q >> 2][4 * (q & 3)], acc[q >> 2][4 * (q & 3) + 1], acc[q >> 2][4 * (q & 3) + 2],
                           acc[q >> 2][4 * (q & 3) + 3]};
  }
  __syncthreads();
  if (half == 0) {
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const f32x4 v = part[64 * q];
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[q >> 2][4 * (q & 3) + e] += v[e];
    }
    // (both halves have long read their rows: x_in may alias out)
    if (pos0 < rows) pair_update_epilogue<ZBIAS>(acc, out, rows, pos0, m, h, accumulate, zb);
  }
}

// The pair transition with its weights in registers (pf_direct.h): 8 waves (one workgroup per CU) walk
// groups of 64 rows.  Wave w owns hidden units (HID / 8) w .. of fc1 and fc2, and the output channels
// 32 (w & 3) .. + 31 of half w >> 2 of the hidden units of fc3: at HID = 512 three times 64 registers.
// A group is normalized once into LDS; the hidden activations (op_t) go through LDS; the two halves
// of each output meet in LDS, each wave finishing one 32-row tile; and the finished rows leave from
// LDS whole, 16 lanes a row, with the residual and corr (TR_MEANFIX: added in fp32).  ZBIAS: the
// workgroup then normalizes the rows it has just written and waves 0 and 1 project them.
// Against weight blocks streamed through an LDS ring by four-wave workgroups (one LDS read per MFMA,
// here three for four; the residual re-read from HBM), us, plain weights: hidden 256, N = 128 17.1 ->
// 10.3, 450 94 -> 83, 1024 434 -> 370; hidden 512, N = 128 24.4 -> 15.5, 1024 602 -> 546; with the
// mean correction and the pair bias N = 384 111 -> 105, 768 350 -> 338, 1024 601 -> 572.  MFMAs, SwiGLU and LDS traffic take about 3.5, 2.5 and
// 3.3 us of a group's 8.5 at hidden 512 and hardly overlap with one workgroup per CU: every wave is
// in the same phase (raising the priority of one wave per SIMD in the first phase changed nothing).
constexpr int TRD_WAVES = 8, TRD_ZP = 132;
template <int HID>
struct TrdLds {   // byte offsets
  static constexpr int K3L = HID == 512 ? 8 : 0;   // fc3 k-steps of a wave that stay in LDS
  static constexpr size_t SX = 0;                                            // normalized rows [64][136] op_t
  static constexpr size_t SH = SX + (size_t)DP_ROWS * LDSW * sizeof(op_t);   // hidden [64][HID + 8] op_t, then rows [64][132] fp32
  static constexpr size_t SHB = (size_t)DP_ROWS * (HID + 8) * sizeof(op_t);
  static constexpr size_t ROWB = (size_t)DP_ROWS * TRD_ZP * 4;
  static constexpr size_t WBUF = (size_t)TRD_WAVES * 32 * LDSW * sizeof(op_t);   // set-up: the weight buffers
  static_assert(ROWB + (size_t)DP_ROWS * LDSW * sizeof(op_t) <= WBUF, "ZBIAS: normalized rows behind the rows");
  static constexpr size_t VEC = SH + (SHB > WBUF ? SHB : WBUF > ROWB ? WBUF : ROWB);
  static constexpr size_t WZ = VEC + 5 * C * 4;                              // norm w, b, corr, zb norm w, b [128] fp32 each
  static constexpr size_t F3 = WZ + (size_t)16 * LDSW * sizeof(op_t);        // W_z [16][136] op_t
  static constexpr size_t BYTES = F3 + (size_t)TRD_WAVES * K3L * 64 * 16;    // fragments [8][K3L][64 lanes]
};
template <int HID, bool ZBIAS, bool CORR>
__global__ __launch_bounds__(64 * TRD_WAVES, 1) void tr_direct_kernel(
    const float* x_in, float* out, const float* __restrict__ lnw, const float* __restrict__ lnb,
    const op_t* __restrict__ w1, const op_t* __restrict__ w2, const op_t* __restrict__ w3, long rows, int accumulate,
    float eps, ZBiasArgs zb, const float* __restrict__ corr, int ngroups) {
  typedef TrdLds<HID> L;
  constexpr int NB = HID / 256;                  // 32-unit hidden blocks of a wave
  constexpr int K3 = HID / 32, K3R = K3 - L::K3L;   // fc3 k-steps of a wave, in registers
  constexpr int LH = HID + 8, ZP = TRD_ZP;
  extern __shared__ __attribute__((aligned(16))) char dl[];
  op_t* sx = reinterpret_cast<op_t*>(dl + L::SX);
  op_t* sh = reinterpret_cast<op_t*>(dl + L::SH);
  float* zrow = reinterpret_cast<float*>(sh);
  op_t* sz = reinterpret_cast<op_t*>(dl + L::SH + L::ROWB);
  float* vec = reinterpret_cast<float*>(dl + L::VEC);
  op_t* swz = reinterpret_cast<op_t*>(dl + L::WZ);
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, m = lane & 31;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  opx8* f3l = reinterpret_cast<opx8*>(dl + L::F3) + wid * L::K3L * 64 + lane;
  const int ob = wid & 3, kh = wid >> 2;
  const int g4 = lane >> 4, q4 = lane & 15;
  // rows 8 wid + 4 it + g4 of a group, channels 4 q4 .. and 64 + 4 q4 ..: loads clamped at the end
  // (uniform base + 32-bit lane offset: 64-bit lane addresses cost the registers the weights need)
  f32x4 x[2][2];
  auto fetch = [&](const float* src, int g, f32x4 (&v)[2][2]) PF_INLINE {
    const char* base = reinterpret_cast<const char*>(src + (long)DP_ROWS * g * C);
    const uint32_t last = (uint32_t)min((long)DP_ROWS, rows - (long)DP_ROWS * g) - 1;
#pragma unroll
    for (int it = 0; it < 2; ++it) {
      const uint32_t off = 4u * (min((uint32_t)(8 * wid + 4 * it + g4), last) * C + 4 * q4);
      v[it][0] = *reinterpret_cast<const f32x4*>(base + off);
      v[it][1] = *reinterpret_cast<const f32x4*>(base + off + 256);
    }
  };
  // LayerNorm with affine parameters w, b (LDS) of the wave's 8 rows -> op_t rows of dst
  auto norm_row = [&](const f32x4 (&v)[2], const float* w, const float* b, float e_, op_t* dst, int r, int q4) PF_INLINE {
    const float mean = row16_sum((v[0][0] + v[0][1]) + (v[0][2] + v[0][3]) + (v[1][0] + v[1][1]) +
                                 (v[1][2] + v[1][3])) * (1.f / C);
    float var = 0.f;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) { const float d = v[u][e] - mean; var += d * d; }
    const float rstd = rsqrtf(row16_sum(var) * (1.f / C) + e_);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const f32x4 gw = *reinterpret_cast<const f32x4*>(w + 64 * u + 4 * q4);
      const f32x4 gb = *reinterpret_cast<const f32x4*>(b + 64 * u + 4 * q4);
      opx4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (op_t)((v[u][e] - mean) * rstd * gw[e] + gb[e]);
      st_x4(dst + r * LDSW + 64 * u + 4 * q4, o);
    }
  };
  fetch(x_in, blockIdx.x, x);
  DirectW<C> f1[NB], f2[NB];
  opx8 f3[K3R];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    f1[b].load(w1 + (long)32 * (NB * wid + b) * C, lane);
    f2[b].load(w2 + (long)32 * (NB * wid + b) * C, lane);
  }
  if (tid < C) {
    vec[tid] = lnw[tid];
    vec[C + tid] = lnb[tid];
    if constexpr (CORR) vec[2 * C + tid] = corr[tid];
    if constexpr (ZBIAS) {
      vec[3 * C + tid] = zb.lnw[tid];
      vec[4 * C + tid] = zb.lnb[tid];
    }
  }
  if constexpr (ZBIAS)
    if (tid < 16 * 16)
      st_x8(swz + (tid >> 4) * LDSW + 8 * (tid & 15), ld_x8(zb.wz + min(tid >> 4, zb.H - 1) * C + 8 * (tid & 15)));
  {   // fc3 rows 32 ob + m, columns (HID / 2) kh ..: 128-byte pieces of 8 rows an instruction, turned
      // 64 columns at a time
    op_t* wb = sh + wid * 32 * LDSW;   // the waves' buffers (8 x 8.5 KB)
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      f1[b].turn(wb, lane);
      f2[b].turn(wb, lane);
    }
    const op_t* src = w3 + (long)32 * ob * HID + (HID / 2) * kh;
#pragma unroll
    for (int c = 0; c < K3 / 4; ++c) {
      opx8 v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = ld_x8(src + (long)(8 * i + (lane >> 3)) * HID + 64 * c + 8 * (lane & 7));
#pragma unroll
      for (int i = 0; i < 4; ++i) st_x8(wb + (8 * i + (lane >> 3)) * LDSW + 8 * (lane & 7), v[i]);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const opx8 f = ld_x8(wb + m * LDSW + 16 * s + 8 * h);
        if (4 * c + s < K3R)
          f3[4 * c + s < K3R ? 4 * c + s : 0] = f;
        else
          f3l[64 * (4 * c + s - K3R)] = f;
      }
    }
  }
  __syncthreads();   // the weight buffers are read out
  for (int gi = blockIdx.x; gi < ngroups; gi += gridDim.x) {
#pragma unroll
    for (int it = 0; it < 2; ++it) norm_row(x[it], vec, vec + C, eps, sx, 8 * wid + 4 * it + g4, q4);
    __syncthreads();   // sx is whole; sh and the last rows are free
    // the next group's rows as early as the registers allow
    const bool more = gi + (int)gridDim.x < ngroups;
    if (HID == 256 && more) fetch(x_in, gi + gridDim.x, x);
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        f32x16 a1 = zero16(), a2 = zero16();
        const op_t* xr = sx + (32 * t + m) * LDSW + 8 * h;
        opx8 c0 = ld_x8(xr), c1 = ld_x8(xr + 16);
#pragma unroll
        for (int s = 0; s < 8; s += 2) {   // the next two fragments are read beside these four MFMAs
          const opx8 n0 = ld_x8(xr + 16 * ((s + 2) & 7)), n1 = ld_x8(xr + 16 * ((s + 3) & 7));
          a1 = mfma32(f1[b].v[s], c0, a1);   // rows = hidden unit, cols = row of x
          a2 = mfma32(f2[b].v[s], c0, a2);
          a1 = mfma32(f1[b].v[s + 1], c1, a1);
          a2 = mfma32(f2[b].v[s + 1], c1, a2);
          c0 = n0;
          c1 = n1;
          __builtin_amdgcn_sched_barrier(0);
        }
        op_t* dst = sh + (32 * t + m) * LH + 32 * (NB * wid + b) + 4 * h;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          opx4 v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = (op_t)(siluf(a1[4 * g + e]) * a2[4 * g + e]);
          st_x4(dst + 8 * g, v);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    __syncthreads();
    if (HID != 256 && more) fetch(x_in, gi + gridDim.x, x);
    f32x4 res[2][2];   // the residual, in the rows' final layout
    if (HID == 256 && accumulate) fetch(out, gi, res);
    f32x16 acc[2] = {zero16(), zero16()};
    const op_t* hr = sh + m * LH + (HID / 2) * kh + 8 * h;
#pragma unroll
    for (int s = 0; s < K3; ++s) {
      const opx8 wf = s < K3R ? f3[s < K3R ? s : 0] : f3l[64 * (s - K3R)];
#pragma unroll
      for (int t = 0; t < 2; ++t) acc[t] = mfma32(wf, ld_x8(hr + 32 * t * LH + 16 * s), acc[t]);
      if (s % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();   // sh is read out: the rows go over it, one half's sums, then the other's added
    if (HID != 256 && accumulate) fetch(out, gi, res);
    float* zr = zrow + m * ZP + 32 * ob + 4 * h;
    if (kh == 0) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *reinterpret_cast<f32x4*>(zr + 32 * t * ZP + 8 * g) =
              f32x4{acc[t][4 * g], acc[t][4 * g + 1], acc[t][4 * g + 2], acc[t][4 * g + 3]};
    }
    __syncthreads();
    if (kh == 1) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          f32x4 v = *reinterpret_cast<f32x4*>(zr + 32 * t * ZP + 8 * g);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += acc[t][4 * g + e];
          *reinterpret_cast<f32x4*>(zr + 32 * t * ZP + 8 * g) = v;
        }
    }
    __syncthreads();
    char* obase = reinterpret_cast<char*>(out + (long)DP_ROWS * gi * C);
    const int left = (int)min((long)DP_ROWS, rows - (long)DP_ROWS * gi);
    int fl = lane;
    asm volatile("" : "+v"(fl));   // the addresses are formed here, not kept across the loop
    const int q4 = fl & 15;
#pragma unroll
    for (int it = 0; it < 2; ++it) {
      const int r = 8 * wid + 4 * it + (fl >> 4);
      f32x4 z[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        z[u] = *reinterpret_cast<const f32x4*>(zrow + r * ZP + 64 * u + 4 * q4);
        if constexpr (CORR) {
          const f32x4 c = *reinterpret_cast<const f32x4*>(vec + 2 * C + 64 * u + 4 * q4);
#pragma unroll
          for (int e = 0; e < 4; ++e) z[u][e] += c[e];
        }
        if (accumulate)
#pragma unroll
          for (int e = 0; e < 4; ++e) z[u][e] += res[it][u][e];
        if (r < left) *reinterpret_cast<f32x4*>(obase + 4u * (r * C + 64 * u + 4 * q4)) = z[u];
      }
      // ZBIAS: the updated row normalized, behind the rows in sh
      if constexpr (ZBIAS) norm_row(z, vec + 3 * C, vec + 4 * C, zb.eps, sz, r, q4);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (ZBIAS) {
      __syncthreads();
      if (wid < 2) {   // D[head][row] of tile wid (N * N is a multiple of 32)
        int zl = lane;
        asm volatile("" : "+v"(zl));   // the addresses are formed here, not kept across the loop
        const int zm = zl & 31, zh = zl >> 5;
        f32x16 hb = zero16();
#pragma unroll
        for (int s = 0; s < 8; ++s) {
          hb = mfma32(ld_x8(swz + (zm & 15) * LDSW + 16 * s + 8 * zh), ld_x8(sz + (32 * wid + zm) * LDSW + 16 * s + 8 * zh), hb);
          if (s % 2) __builtin_amdgcn_sched_barrier(0);
        }
        const long p0 = (long)DP_ROWS * gi + 32 * wid;
        if (p0 < rows) {
          const long b = p0 / zb.NN;
          char* brow = reinterpret_cast<char*>(zb.bias + b * zb.H * zb.NN + (p0 - b * zb.NN));
          const uint32_t boff = 4u * (4u * zh * (uint32_t)zb.NN + zm);
#pragma unroll
          for (int r = 0; r < 8; ++r) {   // heads 0..15: registers 0..7
            if (acc_row(r, zh) < zb.H)
              *reinterpret_cast<float*>(brow + 4 * acc_row(r, 0) * zb.NN + boff) = hb[r] * 1.4426950408889634f;
          }
        }
      }
    }
  }
}

// corr[c] = the sum of np partial rows [np][128]: one workgroup of 1024 threads, thread
// (quad q of 4 channels, group g of 32) summing rows g, g + 32, ... with all its loads in
// flight (np <= TRS_PARTIALS), then the 32 groups through LDS.
__global__ __launch_bounds__(1024) void tr_corr_kernel(const float* __restrict__ partials, int np,
                                                       float* __restrict__ corr) {
  constexpr int G = 32, PER = TRS_PARTIALS / G;
  __shared__ f32x4 part[G][C / 4 + 1];
  const int q = threadIdx.x & (C / 4 - 1), g = threadIdx.x >> 5;
  f32x4 v[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int p = g + G * i;
    v[i] = p < np ? *reinterpret_cast<const f32x4*>(partials + (size_t)p * C + 4 * q) : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < PER; ++i) sum += v[i];
  part[g][q] = sum;
  __syncthreads();
  if (threadIdx.x < C) {
    const int c = threadIdx.x;
    float t = 0.f;
#pragma unroll
    for (int j = 0; j < G; ++j) t += part[j][c >> 2][c & 3];
    corr[c] = t;
  }
}

// Workspace of the C = 128 pair transition: the TR_STATS partials and corr (fp32).
constexpr size_t TR_WS_BYTES = ((size_t)TRS_PARTIALS + 1) * C * sizeof(float);

// Checks of the fc3 residual options: C = 128 only; the mean correction needs the residual and
// the workspace for its sums.
int tr_check_fc3(const pf_transition_args* a, const char* fn) {
  if (a->fc3_lo && a->C != C)
    return pf_fail(PF_E_INVALID, "%s: the fc3 residual (fc3_lo) is supported for C = 128 only", fn);
  if (a->fc3_mean_fix && !a->fc3_lo)
    return pf_fail(PF_E_INVALID, "%s: fc3_mean_fix needs the fc3 residual (fc3_lo)", fn);
  if (a->fc3_mean_fix && (a->hidden % 64 || a->hidden > TRS_MAX_HIDDEN))
    return pf_fail(PF_E_INVALID, "%s: fc3_mean_fix needs hidden a multiple of 64 up to %d (got %d)", fn,
                   TRS_MAX_HIDDEN, a->hidden);
  if (a->fc3_mean_fix && (!a->workspace || a->workspace_bytes < TR_WS_BYTES))
    return pf_fail(PF_E_INVALID, "%s: fc3_mean_fix needs a workspace of %zu bytes (got %zu)", fn, TR_WS_BYTES,
                   a->workspace ? a->workspace_bytes : (size_t)0);
  return PF_OK;
}

// The register-weight transition where it applies (hidden 256 or 512, at most 16 heads); false: not.
template <bool ZBIAS, bool CORR>
bool launch_tr_direct(const pf_transition_args* a, const ZBiasArgs& zb, const float* corr, int* rc) {
  const long groups = (a->rows + DP_ROWS - 1) / DP_ROWS;
  if ((a->hidden != 256 && a->hidden != 512) || (ZBIAS && zb.H > 16) || groups > 0x3fffffff) return false;
  const int cus = device_cus();
  if (cus <= 0) {
    *rc = pf_fail(PF_E_LAUNCH, "tr_direct_kernel: cannot query the device");
    return true;
  }
  auto kern = a->hidden == 256 ? tr_direct_kernel<256, ZBIAS, CORR> : tr_direct_kernel<512, ZBIAS, CORR>;
  const size_t lds = a->hidden == 256 ? TrdLds<256>::BYTES : TrdLds<512>::BYTES;
  if ((*rc = pf_reserve_lds((const void*)kern, lds, "tr_direct_kernel"))) return true;
  kern<<<(unsigned)min(groups, (long)cus), 64 * TRD_WAVES, lds, (hipStream_t)a->stream>>>(
      a->x_in, a->out, a->norm_w, a->norm_b, (const op_t*)a->fc1_w, (const op_t*)a->fc2_w, (const op_t*)a->fc3_w,
      a->rows, a->accumulate, a->eps, zb, corr, (int)groups);
  const hipError_t e = hipGetLastError();
  *rc = e == hipSuccess ? PF_OK : pf_fail(PF_E_LAUNCH, "tr_direct_kernel launch failed: %s", hipGetErrorString(e));
  return true;
}

// The pair transition's launch over workgroups of TRW tiles of 32 pairs (the last one clamped):
// plain, hi + lo, or the mean-corrected form after its sampling pass.
template <bool ZBIAS>
int launch_tr_pair(const pf_transition_args* a, const ZBiasArgs& zb) {
  hipStream_t st = (hipStream_t)a->stream;
  const unsigned grid = (unsigned)((a->rows + 32 * TRW - 1) / (32 * TRW));
  const op_t *w1 = (const op_t*)a->fc1_w, *w2 = (const op_t*)a->fc2_w, *w3 = (const op_t*)a->fc3_w;
  const op_t* lo = (const op_t*)a->fc3_lo;
  int rc = PF_OK;
  if (lo && a->fc3_mean_fix) {
    float* partials = (float*)a->workspace;
    float* corr = partials + (size_t)TRS_PARTIALS * C;
    const long ntiles = a->rows / 32, ns = ntiles < TRS_TILES ? ntiles : TRS_TILES;
    const int np = (int)((ns + TRW - 1) / TRW) * (a->hidden / 64);
    if (ns > 0) {
      tr_pair_kernel<false, TR_STATS><<<np, 64 * TRW, 0, st>>>(a->x_in, nullptr, a->norm_w, a->norm_b, w1, w2, lo,
                                                              nullptr, a->rows, a->hidden, 0, a->eps, ZBiasArgs{},
                                                              nullptr, partials);
      PF_CHECK_LAUNCH("tr_pair_kernel (sampling pass)");
    }
    tr_corr_kernel<<<1, 1024, 0, st>>>(partials, ns > 0 ? np : 0, corr);   // no sample: corr = 0
    PF_CHECK_LAUNCH("tr_corr_kernel");
    if (launch_tr_direct<ZBIAS, true>(a, zb, corr, &rc)) return rc;
    tr_pair_kernel<ZBIAS, TR_MEANFIX><<<grid, 64 * TRW, 0, st>>>(a->x_in, a->out, a->norm_w, a->norm_b, w1, w2, w3,
                                                                nullptr, a->rows, a->hidden, a->accumulate, a->eps,
                                                                zb, corr, nullptr);
  } else if (lo && a->hidden % 64 == 0 && (a->rows + 63) / 64 <= device_cus()) {
    // one workgroup fills a CU: up to one round of the chip (N = 128), where the chain is the time
    const void* fn = (const void*)tr_pair_split_kernel<ZBIAS>;
    if (const int rc = pf_reserve_lds(fn, TRSP_LDS, "tr_pair_split_kernel")) return rc;
    tr_pair_split_kernel<ZBIAS><<<(unsigned)((a->rows + 63) / 64), 64 * TRW, TRSP_LDS, st>>>(
        a->x_in, a->out, a->norm_w, a->norm_b, w1, w2, w3, lo, a->rows, a->hidden, a->accumulate, a->eps, zb);
  } else if (lo) {
    tr_pair_kernel<ZBIAS, TR_HILO><<<grid, 64 * TRW, 0, st>>>(a->x_in, a->out, a->norm_w, a->norm_b, w1, w2, w3, lo,
                                                             a->rows, a->hidden, a->accumulate, a->eps, zb, nullptr,
                                                             nullptr);
  } else if (launch_tr_direct<ZBIAS, false>(a, zb, nullptr, &rc)) {
    return rc;
  } else {
    tr_pair_kernel<ZBIAS, TR_PLAIN><<<grid, 64 * TRW, 0, st>>>(a->x_in, a->out, a->norm_w, a->norm_b, w1, w2, w3,
                                                              nullptr, a->rows, a->hidden, a->accumulate, a->eps, zb,
                                                              nullptr, nullptr);
  }
  PF_CHECK_LAUNCH("tr_pair_kernel");
  return PF_OK;
}

// Transition with C = 64, hidden = 256 (the MSA transition, tt_bio/reference.py:1333,
// boltz2.py:1188-1258), fused like the pair transition.  Persistent: one workgroup of
// 8 waves per CU keeps fc1, fc2 ([256][64]) and fc3 ([64][256]) in LDS (96 KB); a wave
// walks tiles of 32 rows: LN -> fc1|fc2 as D[hidden][row] (rows of fc1/fc2 in perm16
// order within each 32-block, so the accumulators come out in fc3's k order) ->
// silu(a)*b -> fc3 as D[channel][row] -> residual in the output-aligned layout.
// LDS rows are unpadded with XOR-swizzled 16-byte chunks (conflict-free fragment reads).
constexpr int T64_WAVES = 8;

__global__ __launch_bounds__(64 * T64_WAVES, 1) void tr64_kernel(
    const float* x_in, float* out, const float* __restrict__ lnw, const float* __restrict__ lnb,
    const op_t* __restrict__ w1, const op_t* __restrict__ w2, const op_t* __restrict__ w3, long rows,
    int accumulate, float eps) {
  __shared__ __attribute__((aligned(16))) op_t s1[256 * 64];
  __shared__ __attribute__((aligned(16))) op_t s2[256 * 64];
  __shared__ __attribute__((aligned(16))) op_t s3[64 * 256];
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, m = lane & 31;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  for (int c = tid; c < 256 * 8; c += 64 * T64_WAVES) {   // fc1 / fc2: 256 rows of 8 chunks
    const int R = c >> 3, k = c & 7;
    const int src = (32 * (R >> 5) + perm16(R & 31)) * 64 + 8 * k;
    const int dst = R * 64 + 8 * (k ^ swz8r(R));
    st_x8(s1 + dst, ld_x8(w1 + src));
    st_x8(s2 + dst, ld_x8(w2 + src));
  }
  for (int c = tid; c < 64 * 32; c += 64 * T64_WAVES) {   // fc3: 64 rows of 32 chunks
    const int R = c >> 5, k = c & 31;
    st_x8(s3 + R * 256 + 8 * (k ^ (R & 15)), ld_x8(w3 + R * 256 + 8 * k));
  }
  __syncthreads();
  const int sw = swz8r(m);
  const long ntiles = (rows + 31) / 32;
  for (long t = (long)blockIdx.x * T64_WAVES + wid; t < ntiles; t += (long)gridDim.x * T64_WAVES) {
    const long r0 = 32 * t;
    const long row = min(r0 + m, rows - 1);
    opx8 xf[4];
    ln64_to_frag(x_in + row * 64, h, lnw, lnb, eps, xf);
    f32x16 acc[2] = {zero16(), zero16()};
#pragma unroll 1
    for (int blk = 0; blk < 8; ++blk) {
      f32x16 a1 = zero16(), a2 = zero16();
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        const int off = (32 * blk + m) * 64 + 8 * ((2 * st + h) ^ sw);
        a1 = mfma32(ld_x8(s1 + off), xf[st], a1);   // rows = hidden (perm16), cols = row
        a2 = mfma32(ld_x8(s2 + off), xf[st], a2);
      }
#pragma unroll
      for (int sp = 0; sp < 2; ++sp) {
        opx8 hf;
#pragma unroll
        for (int u = 0; u < 8; ++u) hf[u] = (op_t)(siluf(a1[8 * sp + u]) * a2[8 * sp + u]);
        const int kc = 2 * (2 * blk + sp) + h;   // fc3 row chunk: hidden 32 blk + 16 sp + 8 h
#pragma unroll
        for (int ob = 0; ob < 2; ++ob) {
          const int R = 32 * ob + m;
          acc[ob] = mfma32(ld_x8(s3 + R * 256 + 8 * (kc ^ (R & 15))), hf, acc[ob]);   // rows = channel
        }
      }
    }
    if (r0 + m >= rows) continue;
    // lane (row m, h): acc[ob][4 g + e] is channel 32 ob + 8 g + 4 h + e; x_in may alias out
    const float* src = x_in + (r0 + m) * 64;
    float* dst = out + (r0 + m) * 64;
    f32x4 res[8];
#pragma unroll
    for (int q = 0; q < 8; ++q)
      res[q] = accumulate ? *reinterpret_cast<const f32x4*>(src + oa_channel(q, h)) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = acc[q >> 2][4 * (q & 3) + e] + res[q][e];
      *reinterpret_cast<f32x4*>(dst + oa_channel(q, h)) = v;
    }
  }
}

// One wave per row.
// One wave per row.  Rows of up to 64 * LN_REG values are read once into registers (all of a
// lane's loads in flight together); longer rows are read three times.
constexpr int LN_REG = 8;
__global__ __launch_bounds__(256) void ln_rows_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                      const float* __restrict__ b, float* __restrict__ out,
                                                      long rows, int C_, float eps) {
  const long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= rows) return;
  const float* xr = x + row * C_;
  float* orow = out + row * C_;
  if (C_ <= 64 * LN_REG) {
    float xv[LN_REG];
#pragma unroll
    for (int u = 0; u < LN_REG; ++u) xv[u] = lane + 64 * u < C_ ? xr[lane + 64 * u] : 0.f;
    float s = 0.f;
#pragma unroll
    for (int u = 0; u < LN_REG; ++u) s += xv[u];
    const float mean = wave_sum(s) / C_;
    float v = 0.f;
#pragma unroll
    for (int u = 0; u < LN_REG; ++u) {
      const float d = lane + 64 * u < C_ ? xv[u] - mean : 0.f;
      v += d * d;
    }
    const float rstd = rsqrtf(wave_sum(v) / C_ + eps);
#pragma unroll
    for (int u = 0; u < LN_REG; ++u) {
      const int c = lane + 64 * u;
      if (c < C_) orow[c] = (xv[u] - mean) * rstd * w[c] + b[c];
    }
    return;
  }
  float s = 0.f;
  for (int c = lane; c < C_; c += 64) s += xr[c];
  const float mean = wave_sum(s) / C_;
  float v = 0.f;
  for (int c = lane; c < C_; c += 64) { const float d = xr[c] - mean; v += d * d; }
  const float rstd = rsqrtf(wave_sum(v) / C_ + eps);
  for (int c = lane; c < C_; c += 64) orow[c] = (xr[c] - mean) * rstd * w[c] + b[c];
}

// A workgroup = one 32-row x 32-column output tile of one job; its 4 waves split the K
// steps (contiguous quarters), each wave issuing up to 8 steps of loads before their
// MFMAs, so a tile pays about one memory round trip per 8 steps of its quarter.  The
// partial accumulators meet in LDS and all 256 threads run the epilogue (4 outputs each,
// 32 consecutive columns per row).  blockIdx.z selects the job (several projections of
// the same shape in one launch).  SWIGLU: out[:, n] = silu(x W[n]) * (x W2[n]).
constexpr int LIN_SPLIT = 4;
struct LinJobs { pf_lin_job j[PF_LIN_MAX_JOBS]; };

template <bool SWIGLU>
__global__ __launch_bounds__(256) void linear_rows_kernel(LinJobs jobs, long rows, int K, int Nout) {
  __shared__ float red[LIN_SPLIT][SWIGLU ? 2 : 1][16][64];
  const pf_lin_job& jb = jobs.j[blockIdx.z];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, h = lane >> 5, m = lane & 31;
  const int n0 = blockIdx.y * 32;
  const long r0 = (long)blockIdx.x * 32;
  const float* xr = jb.x + min(r0 + m, rows - 1) * K;
  const op_t* wr = (const op_t*)jb.W + (long)(n0 + m) * K;
  const op_t* wr2 = SWIGLU ? (const op_t*)jb.W2 + (long)(n0 + m) * K : nullptr;
  const int nsteps = K >> 4, per = (nsteps + LIN_SPLIT - 1) / LIN_SPLIT;
  const int s0 = min(nsteps, wid * per), s1 = min(nsteps, s0 + per);
  f32x16 acc = zero16(), acc2 = zero16();
  for (int sg = s0; sg < s1; sg += 8) {
    opx8 af[8], wf[8], wf2[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int kk = 16 * (sg + u);
      if (sg + u < s1) {
        const f32x4 a0 = *reinterpret_cast<const f32x4*>(xr + kk + 8 * h);
        const f32x4 a1 = *reinterpret_cast<const f32x4*>(xr + kk + 8 * h + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          af[u][e] = (op_t)a0[e];
          af[u][4 + e] = (op_t)a1[e];
        }
        wf[u] = ld_x8(wr + kk + 8 * h);
        if (SWIGLU) wf2[u] = ld_x8(wr2 + kk + 8 * h);
      } else {
        af[u] = zero_x8();
        wf[u] = zero_x8();
        if (SWIGLU) wf2[u] = zero_x8();
      }
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      acc = mfma32(af[u], wf[u], acc);
      if (SWIGLU) acc2 = mfma32(af[u], wf2[u], acc2);
    }
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    red[wid][0][r][lane] = acc[r];
    if (SWIGLU) red[wid][1][r][lane] = acc2[r];
  }
  __syncthreads();
  // thread (wid, lane) finishes accumulator registers 4 wid .. 4 wid + 3 of lane
  const int n = n0 + m;
  const float bn = jb.bias ? jb.bias[n] : 0.f;
  float v[4], res[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 4 * wid + i;
    float a = 0.f, a2 = 0.f;
#pragma unroll
    for (int w = 0; w < LIN_SPLIT; ++w) {
      a += red[w][0][r][lane];
      if (SWIGLU) a2 += red[w][1][r][lane];
    }
    v[i] = SWIGLU ? siluf(a) * a2 : a + bn;
    // resid may alias out: all loads ahead of the stores, so they overlap
    res[i] = !SWIGLU && jb.resid ? jb.resid[min(r0 + acc_row(r, h), rows - 1) * Nout + n] : 0.f;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const long row = r0 + acc_row(4 * wid + i, h);
    if (row < rows) jb.out[row * Nout + n] = v[i] + res[i];
  }
}

// out[p, :] = base[p, :] + W . LN(x[p, :]),  C = 128; W resident in LDS.  HILO: W = W + W_lo and
// LN(x) = hi + lo (16-bit each), products hi.W + lo.W + hi.W_lo (the lo.W_lo term is below
// fp32's resolution of the sum).
template <bool HILO>
__global__ __launch_bounds__(256) void pair_ln_linear_kernel(
    const float* x, const float* base, const float* __restrict__ lnw, const float* __restrict__ lnb,
    const op_t* __restrict__ W, const op_t* __restrict__ W_lo, float* out, long rows, float eps) {
  __shared__ __attribute__((aligned(16))) op_t sW[(HILO ? 2 : 1) * C * LDSW];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, h = lane >> 5, m = lane & 31;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int c = tid + 256 * q;
    st_x8(&sW[(c >> 4) * LDSW + (c & 15) * 8], ld_x8(W + (c >> 4) * C + (c & 15) * 8));
    if constexpr (HILO) st_x8(&sW[C * LDSW + (c >> 4) * LDSW + (c & 15) * 8], ld_x8(W_lo + (c >> 4) * C + (c & 15) * 8));
  }
  __syncthreads();
  const long pos0 = ((long)blockIdx.x * 4 + wid) * 32;
  if (pos0 >= rows) return;
  float xv[64];
  opx8 xf[8], xl[8];
  load_row128_frag(x + min(pos0 + m, rows - 1) * C, h, xv);
  if constexpr (HILO) {
    float sm = 0.f;
#pragma unroll
    for (int i = 0; i < 64; ++i) sm += xv[i];
    const float mean = xor32_sum(sm) * (1.f / C);
    float var = 0.f;
#pragma unroll
    for (int i = 0; i < 64; ++i) { const float d = xv[i] - mean; var += d * d; }
    const float rstd = rsqrtf(xor32_sum(var) * (1.f / C) + eps);
#pragma unroll
    for (int s = 0; s < 8; ++s)
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const int c = 16 * s + 8 * h + t;
        const float y = (xv[8 * s + t] - mean) * rstd * lnw[c] + lnb[c];
        xf[s][t] = (op_t)y;
        xl[s][t] = (op_t)(y - (float)xf[s][t]);
      }
  } else {
    ln128_to_frag(xv, h, lnw, lnb, eps, xf);
  }
#pragma unroll
  for (int ob = 0; ob < 4; ++ob) {
    f32x16 acc = zero16();
#pragma unroll
    for (int s = 0; s < 8; ++s) acc = mfma32(xf[s], ld_x8(&sW[(32 * ob + m) * LDSW + 16 * s + 8 * h]), acc);
    if constexpr (HILO) {
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        acc = mfma32(xl[s], ld_x8(&sW[(32 * ob + m) * LDSW + 16 * s + 8 * h]), acc);
        acc = mfma32(xf[s], ld_x8(&sW[C * LDSW + (32 * ob + m) * LDSW + 16 * s + 8 * h]), acc);
      }
    }
    // base may alias out: all loads ahead of the stores, so they overlap
    float res[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) res[r] = base[min(pos0 + acc_row(r, h), rows - 1) * C + 32 * ob + m];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const long p = pos0 + acc_row(r, h);
      if (p < rows) out[p * C + 32 * ob + m] = res[r] + acc[r];
    }
  }
}

}  // namespace

// ---------------------------------------------------------------------------------
// C-ABI
// ---------------------------------------------------------------------------------
extern "C" int pf_layernorm_fwd(const float* x, const float* w, const float* b, float* out, long rows,
                                int C_, float eps, void* stream) {
  if (!x || !w || !b || !out) return pf_fail(PF_E_INVALID, "pf_layernorm_fwd: null pointer");
  if (rows <= 0 || C_ <= 0 || C_ > 4096) return pf_fail(PF_E_INVALID, "pf_layernorm_fwd: bad shape rows=%ld C=%d", rows, C_);
  ln_rows_kernel<<<(unsigned)((rows + 3) / 4), 256, 0, (hipStream_t)stream>>>(x, w, b, out, rows, C_, eps);
  PF_CHECK_LAUNCH("ln_rows_kernel");
  return PF_OK;
}

int pf_linear_batch(const pf_lin_job* jobs, int njobs, long rows, int K, int Nout, hipStream_t st) {
  if (njobs < 1 || njobs > PF_LIN_MAX_JOBS) return pf_fail(PF_E_INVALID, "pf_linear_fwd: %d jobs", njobs);
  if (rows <= 0 || K <= 0 || K % 16 || Nout <= 0 || Nout % 32)
    return pf_fail(PF_E_INVALID, "pf_linear_fwd: need rows > 0, K %% 16 == 0, Nout %% 32 == 0 (rows=%ld K=%d Nout=%d)",
                   rows, K, Nout);
  LinJobs J{};
  const bool swiglu = jobs[0].W2 != nullptr;
  for (int i = 0; i < njobs; ++i) {
    if (!jobs[i].x || !jobs[i].W || !jobs[i].out) return pf_fail(PF_E_INVALID, "pf_linear_fwd: null pointer");
    if ((jobs[i].W2 != nullptr) != swiglu) return pf_fail(PF_E_INVALID, "pf_linear_fwd: mixed SwiGLU jobs");
    J.j[i] = jobs[i];
  }
  dim3 grid((unsigned)((rows + 31) / 32), (unsigned)(Nout / 32), (unsigned)njobs);
  if (swiglu)
    linear_rows_kernel<true><<<grid, 256, 0, st>>>(J, rows, K, Nout);
  else
    linear_rows_kernel<false><<<grid, 256, 0, st>>>(J, rows, K, Nout);
  PF_CHECK_LAUNCH("linear_rows_kernel");
  return PF_OK;
}

static int launch_linear(const float* x, const void* W, const void* W2, const float* bias, const float* resid,
                         float* out, long rows, int K, int Nout, hipStream_t st) {
  const pf_lin_job job{x, W, W2, bias, resid, out};
  return pf_linear_batch(&job, 1, rows, K, Nout, st);
}

extern "C" int pf_linear_fwd(const float* x, const void* W, const float* bias, const float* resid, float* out,
                             long rows, int K, int Nout, void* stream) {
  return launch_linear(x, W, nullptr, bias, resid, out, rows, K, Nout, (hipStream_t)stream);
}

extern "C" size_t pf_transition_workspace_size(long rows, int C_, int hidden) {
  if (rows <= 0 || C_ <= 0 || hidden <= 0) return 0;
  if (C_ == C && hidden % 32 == 0) return TR_WS_BYTES;   // fused pair kernel: the mean-correction sums
  if (C_ == 64 && hidden == 256) return 0;      // fused C = 64 kernel: no scratch
  return (size_t)rows * (C_ + hidden) * sizeof(float);
}

extern "C" int pf_transition_fwd(const pf_transition_args* a) {
  if (!a) return pf_fail(PF_E_INVALID, "pf_transition_fwd: null args");
  if (a->rows <= 0 || a->C <= 0 || a->hidden <= 0 || a->hidden % 32 || a->C % 32)
    return pf_fail(PF_E_INVALID, "pf_transition_fwd: need rows > 0 and C, hidden multiples of 32 (C=%d hidden=%d)",
                   a->C, a->hidden);
  if (!a->x_in || !a->out || !a->norm_w || !a->norm_b || !a->fc1_w || !a->fc2_w || !a->fc3_w)
    return pf_fail(PF_E_INVALID, "pf_transition_fwd: null pointer argument");
  hipStream_t st = (hipStream_t)a->stream;
  if (const int rc = tr_check_fc3(a, "pf_transition_fwd")) return rc;
  if (a->C == C) return launch_tr_pair<false>(a, ZBiasArgs{});
  if (a->C == 64 && a->hidden == 256) {
    const int cus = device_cus();
    if (cus <= 0) return pf_fail(PF_E_LAUNCH, "tr64_kernel: cannot query the device");
    const long tiles = (a->rows + 31) / 32;
    const int grid = (int)min((long)cus, (tiles + T64_WAVES - 1) / T64_WAVES);
    tr64_kernel<<<grid, 64 * T64_WAVES, 0, st>>>(a->x_in, a->out, a->norm_w, a->norm_b, (const op_t*)a->fc1_w,
                                                 (const op_t*)a->fc2_w, (const op_t*)a->fc3_w, a->rows,
                                                 a->accumulate, a->eps);
    PF_CHECK_LAUNCH("tr64_kernel");
    return PF_OK;
  }
  const size_t need = pf_transition_workspace_size(a->rows, a->C, a->hidden);
  if (!a->workspace || a->workspace_bytes < need)
    return pf_fail(PF_E_INVALID, "pf_transition_fwd: workspace too small (%zu < %zu bytes)", a->workspace_bytes, need);
  float* xn = (float*)a->workspace;
  float* hid = xn + (size_t)a->rows * a->C;
  int rc = pf_layernorm_fwd(a->x_in, a->norm_w, a->norm_b, xn, a->rows, a->C, a->eps, a->stream);
  if (rc) return rc;
  rc = launch_linear(xn, a->fc1_w, a->fc2_w, nullptr, nullptr, hid, a->rows, a->C, a->hidden, st);
  if (rc) return rc;
  return launch_linear(hid, a->fc3_w, nullptr, nullptr, a->accumulate ? a->out : nullptr, a->out, a->rows,
                       a->hidden, a->C, st);
}

extern "C" int pf_pair_ln_linear_fwd(const float* x, const float* base, const float* ln_w, const float* ln_b,
                                     const void* W, const void* W_lo, float* out, long rows, int C_, float eps,
                                     void* stream) {
  if (!x || !base || !ln_w || !ln_b || !W || !out) return pf_fail(PF_E_INVALID, "pf_pair_ln_linear_fwd: null pointer");
  if (C_ != C || rows <= 0) return pf_fail(PF_E_INVALID, "pf_pair_ln_linear_fwd: only C = 128 (got %d)", C_);
  if (W_lo)
    pair_ln_linear_kernel<true><<<(unsigned)((rows + 127) / 128), 256, 0, (hipStream_t)stream>>>(
        x, base, ln_w, ln_b, (const op_t*)W, (const op_t*)W_lo, out, rows, eps);
  else
    pair_ln_linear_kernel<false><<<(unsigned)((rows + 127) / 128), 256, 0, (hipStream_t)stream>>>(
        x, base, ln_w, ln_b, (const op_t*)W, nullptr, out, rows, eps);
  PF_CHECK_LAUNCH("pair_ln_linear_kernel");
  return PF_OK;
}

__global__ __launch_bounds__(256) void add_kernel(const float* a, const float* b, float* out, long n) {
  const long n4 = n / 4, stride = (long)gridDim.x * blockDim.x;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += stride) {
    const f32x4 u = reinterpret_cast<const f32x4*>(a)[i], v = reinterpret_cast<const f32x4*>(b)[i];
    reinterpret_cast<f32x4*>(out)[i] = u + v;
  }
  for (long i = 4 * n4 + (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) out[i] = a[i] + b[i];
}

extern "C" int pf_add_fwd(const float* a, const float* b, float* out, long n, void* stream) {
  if (!a || !b || !out) return pf_fail(PF_E_INVALID, "pf_add_fwd: null pointer");
  if (n <= 0) return pf_fail(PF_E_INVALID, "pf_add_fwd: n = %ld", n);
  if (((uintptr_t)a | (uintptr_t)b | (uintptr_t)out) & 15)
    return pf_fail(PF_E_INVALID, "pf_add_fwd: pointers must be 16-byte aligned");
  const int cus = device_cus();
  if (cus <= 0) return pf_fail(PF_E_LAUNCH, "pf_add_fwd: cannot query the device");
  const long blocks = min((long)cus * 8, (n / 4 + 255) / 256 + 1);
  add_kernel<<<(unsigned)blocks, 256, 0, (hipStream_t)stream>>>(a, b, out, n);
  PF_CHECK_LAUNCH("add_kernel");
  return PF_OK;
}

extern "C" int pf_transition_pair_bias_fwd(const pf_transition_args* a, const pf_apb_args* apb) {
  if (!a || !apb) return pf_fail(PF_E_INVALID, "pf_transition_pair_bias_fwd: null args");
  if (a->C != C || a->hidden <= 0 || a->hidden % 32)
    return pf_fail(PF_E_INVALID, "pf_transition_pair_bias_fwd: need C = 128 and hidden a multiple of 32 (C=%d hidden=%d)",
                   a->C, a->hidden);
  if (!a->x_in || !a->out || !a->norm_w || !a->norm_b || !a->fc1_w || !a->fc2_w || !a->fc3_w)
    return pf_fail(PF_E_INVALID, "pf_transition_pair_bias_fwd: null pointer argument");
  pf_apb_args chk = *apb;
  chk.z = a->out;   // the bias is computed from the transition's output
  int rc = pf_apb_check(&chk, "pf_transition_pair_bias_fwd", true);
  if (rc) return rc;
  if ((rc = tr_check_fc3(a, "pf_transition_pair_bias_fwd"))) return rc;
  if (a->fc3_mean_fix) {   // the sums must survive the bias writes of the same launch
    const char *t0 = (const char*)a->workspace, *b0 = (const char*)apb->workspace;
    if (t0 < b0 + apb->workspace_bytes && b0 < t0 + TR_WS_BYTES)
      return pf_fail(PF_E_INVALID, "pf_transition_pair_bias_fwd: the transition workspace overlaps the attention's");
  }
  const long NN = (long)apb->N * apb->N;
  if (a->rows != (long)apb->B * NN)
    return pf_fail(PF_E_INVALID, "pf_transition_pair_bias_fwd: rows %ld != B*N*N = %ld", a->rows, (long)apb->B * NN);
  const ZBiasArgs zb{apb->zln_w, apb->zln_b, (const op_t*)apb->w_z, pf_apb_bias_ptr(apb), NN, apb->H, apb->eps};
  return launch_tr_pair<true>(a, zb);   // N % 32 == 0: whole 32-pair tiles
}
