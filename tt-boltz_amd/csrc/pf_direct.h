// Device helpers of the "direct" pair kernels.
//
// A workgroup (one per CU, 8 waves at c_z = 128) walks groups of 64 consecutive positions.  The
// output channels are split over its waves, and each wave keeps its own 32-channel blocks of the
// weights in registers as MFMA fragments for the whole launch; the workgroup normalizes a group's
// positions into LDS once, fully coalesced, and every wave reads its activation fragments from
// there.  Against weights resident in LDS with one wave per 32-position tile (the form these
// kernels replaced: 128 KB staged per workgroup, every tile re-reading all of it, LayerNorms on
// rows strided over lanes) the set-up falls from ~14 to ~6 us, small grids use four times as many
// CUs, and LDS reads per output fall to a quarter.  Whole trimul, us: N = 64 49 -> 25, N = 128
// 56 -> 34, N = 512 230 -> 206, N = 1024 968 -> 839.
#pragma once
#include "pf_common.h"

namespace {

constexpr int DP_ROWS = 64;   // positions of a workgroup

// LayerNorm (without beta) of DP_ROWS rows of CC channels by NW waves into LDS rows of CC + 8
// op_t: wave wid takes 64 / NW rows, 16 lanes a row.  Loads and arithmetic are separate so that
// a caller can issue its weight loads between them.
template <int CC, int NW>
struct DirectLn {
  static constexpr int RPW = DP_ROWS / NW, IT = RPW / 4, NV = CC / 64;
  f32x4 x[IT][NV], gm[NV];
  template <class PairOf>
  PF_DEV void load(const float* z, PairOf pair_of, int wid, int lane) {
    const int g = lane >> 4, q = lane & 15;
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const float* p = z + pair_of(wid * RPW + 4 * it + g) * CC + 4 * q;
#pragma unroll
      for (int v = 0; v < NV; ++v) x[it][v] = *reinterpret_cast<const f32x4*>(p + 64 * v);
    }
  }
  PF_DEV void load_gamma(const float* __restrict__ gamma, int lane) {   // null: none
    const int q = lane & 15;
#pragma unroll
    for (int v = 0; v < NV; ++v)
      gm[v] = gamma ? *reinterpret_cast<const f32x4_any*>(gamma + 64 * v + 4 * q) : f32x4{1.f, 1.f, 1.f, 1.f};
  }
  PF_DEV void store(op_t* dst, float eps, int wid, int lane) const {
    const int g = lane >> 4, q = lane & 15;
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      float s = 0.f;
#pragma unroll
      for (int v = 0; v < NV; ++v) s += (x[it][v][0] + x[it][v][1]) + (x[it][v][2] + x[it][v][3]);
      const float mean = row16_sum(s) * (1.f / CC);
      float var = 0.f;
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int e = 0; e < 4; ++e) { const float d = x[it][v][e] - mean; var += d * d; }
      const float rstd = rsqrtf(row16_sum(var) * (1.f / CC) + eps);
      op_t* row = dst + (wid * RPW + 4 * it + g) * (CC + 8) + 4 * q;
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        opx4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = (op_t)((x[it][v][e] - mean) * (rstd * gm[v][e]));
        st_x4(row + 64 * v, o);
      }
    }
  }
};

// The MFMA fragments of a wave's 32 weight rows (CC op_t each, contiguous at `rows`): loaded as
// whole 1 KB runs (reading fragments straight from global memory would touch 32 cache lines an
// instruction and cost twice the L1 time), then turned through the wave's own LDS buffer of
// [32][CC + 8] op_t.  A wave's LDS accesses complete in order, so the buffer needs no barrier.
template <int CC>
struct DirectW {
  opx8 v[CC / 16];
  PF_DEV void load(const op_t* __restrict__ rows, int lane) {
#pragma unroll
    for (int i = 0; i < CC / 16; ++i) v[i] = ld_x8(rows + 8 * (lane + 64 * i));
  }
  PF_DEV void turn(op_t* buf, int lane) {   // -> v[s]: row lane & 31, k-step s
#pragma unroll
    for (int i = 0; i < CC / 16; ++i) {
      const int c = lane + 64 * i;
      st_x8(buf + (c / (CC / 8)) * (CC + 8) + 8 * (c % (CC / 8)), v[i]);
    }
#pragma unroll
    for (int s = 0; s < CC / 16; ++s) v[s] = ld_x8(buf + (lane & 31) * (CC + 8) + 16 * s + 8 * (lane >> 5));
  }
  // W diag(gamma), rounded to op_t again.  V: f32x4 for a gamma in LDS.
  template <class V = f32x4_any>
  PF_DEV void fold(const float* gamma, int h) {
    // (opaque: the 64 float conversions that an earlier W . beta took are not kept for this)
#pragma unroll
    for (int s = 0; s < CC / 16; ++s) asm volatile("" : "+v"(v[s]));
#pragma unroll
    for (int s = 0; s < CC / 16; ++s) {
      const f32x4 g0 = *reinterpret_cast<const V*>(gamma + 16 * s + 8 * h);
      const f32x4 g1 = *reinterpret_cast<const V*>(gamma + 16 * s + 8 * h + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[s][e] = (op_t)((float)v[s][e] * g0[e]);
        v[s][4 + e] = (op_t)((float)v[s][4 + e] * g1[e]);
      }
      asm volatile("" : "+v"(v[s]));   // done here, not sunk to its use with gamma kept until then
    }
  }
};

// The fragments of a wave's 32 MXFP8 rows (e4m3 bytes [32][CC] at `q`, E8M0 scales [32][CC / 32] at
// `sc`), loaded, then rounded to op_t (exact for scales in its range; a scale byte 0, an all-zero
// block, gives zeros).
template <int CC>
struct DirectW8 {
  typedef int i32x2_t __attribute__((ext_vector_type(2)));
  typedef int i32x2_any __attribute__((ext_vector_type(2), aligned(4)));   // the caller's bytes, in dwords
  i32x2_t w[CC / 16];
  uint32_t e[CC / 32];
  PF_DEV void load(const uint8_t* __restrict__ q, const uint8_t* __restrict__ sc, int lane) {
    const int m = lane & 31, h = lane >> 5;
#pragma unroll
    for (int s = 0; s < CC / 16; ++s) w[s] = *reinterpret_cast<const i32x2_any*>(q + m * CC + 16 * s + 8 * h);
#pragma unroll
    for (int k = 0; k < CC / 32; ++k) e[k] = sc[m * (CC / 32) + k];
  }
  PF_DEV void dequant(DirectW<CC>& o) const {
#pragma unroll
    for (int s = 0; s < CC / 16; ++s) {
      const float X = __uint_as_float(e[s >> 1] << 23);
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        const auto lo = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(w[s][d], X, false);
        const auto hi = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(w[s][d], X, true);
        o.v[s][4 * d + 0] = (op_t)lo[0];
        o.v[s][4 * d + 1] = (op_t)lo[1];
        o.v[s][4 * d + 2] = (op_t)hi[0];
        o.v[s][4 * d + 3] = (op_t)hi[1];
      }
    }
  }
};

// A wave's own tile of 32 rows of 128 channels: read fully coalesced (16 lanes a row, as DirectLn),
// normalized with the affine part, and turned through the wave's own LDS rows of 136 op_t into the
// 8 MFMA fragments (row lane & 31).  The next tile's loads run beside this tile's use.  No barriers.
struct DirectTile {
  f32x4 x[8][2], gm[2], bt[2];
  template <class RowOf>
  PF_DEV void load(const float* __restrict__ z, RowOf row_of, int lane) {   // row_of(r): row r of the tile
    const int g = lane >> 4, q = lane & 15;
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      const float* p = z + row_of(4 * it + g) * 128 + 4 * q;
      x[it][0] = *reinterpret_cast<const f32x4_any*>(p);
      x[it][1] = *reinterpret_cast<const f32x4_any*>(p + 64);
    }
  }
  PF_DEV void affine(const float* __restrict__ gamma, const float* __restrict__ beta, int lane) {   // null: none
    const int q = lane & 15;
#pragma unroll
    for (int v = 0; v < 2; ++v) {
      gm[v] = gamma ? *reinterpret_cast<const f32x4_any*>(gamma + 64 * v + 4 * q) : f32x4{1.f, 1.f, 1.f, 1.f};
      bt[v] = beta ? *reinterpret_cast<const f32x4_any*>(beta + 64 * v + 4 * q) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }
  PF_DEV void normalize(op_t* buf, float eps, int lane) const {
    const int g = lane >> 4, q = lane & 15;
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      const f32x4 a = x[it][0], b = x[it][1];
      const float mean = row16_sum((a[0] + a[1]) + (a[2] + a[3]) + (b[0] + b[1]) + (b[2] + b[3])) * (1.f / 128.f);
      float var = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float d = a[e] - mean, f = b[e] - mean;
        var += d * d + f * f;
      }
      const float rstd = rsqrtf(row16_sum(var) * (1.f / 128.f) + eps);
      opx4 o0, o1;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o0[e] = (op_t)((a[e] - mean) * rstd * gm[0][e] + bt[0][e]);
        o1[e] = (op_t)((b[e] - mean) * rstd * gm[1][e] + bt[1][e]);
      }
      op_t* row = buf + (4 * it + g) * 136 + 4 * q;
      st_x4(row, o0);
      st_x4(row + 64, o1);
    }
  }
  static PF_DEV void fragments(const op_t* buf, int lane, opx8 (&f)[8]) {
#pragma unroll
    for (int s = 0; s < 8; ++s) f[s] = ld_x8(buf + (lane & 31) * 136 + 16 * s + 8 * (lane >> 5));
  }
};

// How a direct kernel uses the rounding residuals of its weights: not at all, as a second MFMA per
// fragment, or through the mean correction (pair_stats_kernel) in the rows' offsets.
enum DirectLo { DL_NONE = 0, DL_MFMA = 1, DL_MEAN = 2 };

// gm[c] (LDS, 128 floats) = gamma[c] * mu[c] of the statistics partials, by a workgroup of NT threads;
// `scratch`: NT floats of LDS.  The caller synchronizes before reading gm.
template <int NT>
PF_DEV void direct_gmu(const float* __restrict__ stats, const float* __restrict__ gamma, float* gm, float* scratch) {
  float pv[stats_per<NT>()];
  stats_load<NT>(stats, pv);
  const float g = gamma && threadIdx.x < PS_C ? gamma[threadIdx.x] : 1.f;
  stats_reduce<NT>(pv, gm, scratch);
  if (threadIdx.x < PS_C) gm[threadIdx.x] *= g;   // written by the same thread
}

// W row . beta in fp32 from the row's fragments (both lane halves get the sum).  V: f32x4 for a
// beta in LDS.
template <int KS, class V = f32x4_any>
PF_DEV float direct_wbeta(const opx8 (&w)[KS], const float* beta, int h) {
  float acc = 0.f;
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const f32x4 b0 = *reinterpret_cast<const V*>(beta + 16 * s + 8 * h);
    const f32x4 b1 = *reinterpret_cast<const V*>(beta + 16 * s + 8 * h + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc += (float)w[s][e] * b0[e] + (float)w[s][4 + e] * b1[e];
    asm volatile("" : "+v"(acc));   // not all of beta in registers at once
  }
  return xor32_sum(acc);
}

}  // namespace
