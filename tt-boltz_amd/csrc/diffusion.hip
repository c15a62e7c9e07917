// Diffusion conditioning, pair side, for gfx950: the two N^2-sized steps that run once
// per trunk output and stay fixed for every sampling step.
//
//   cond_proj_kernel   PairwiseConditioning's input projection (tt_bio/boltz2.py:1318-1355):
//                      out = W . LN(cat(z_trunk, rel_pos)) over 256 channels (LayerNorm with
//                      affine, folded into W as below; LinearNoBias 256 -> 128).  The two
//                      transitions that follow run on the pair transition kernel
//                      (transition.hip).
//   token_bias_kernel  DiffusionConditioning's token-transformer pair bias
//                      (tt_bio/boltz2.py:2434-2441, 2472-2475; the ttnn compute_bias of
//                      tt_bio/tenstorrent.py:714-728): for each of L layers,
//                      LN_l(z) . W_l^T (H heads, no bias), concatenated over layers.  All
//                      layers normalise the same z, so the statistics are computed once and
//                      each layer's affine is folded into its weights when they are staged:
//                      W'_l = W_l diag(gamma_l), b'_l = W_l beta_l.
//
// Both kernels are persistent (one workgroup per CU) with their weights in registers (pf_direct.h):
// groups of 64 pairs are normalized once into LDS, 16 lanes a row, every wave multiplies them by its
// own 32 output rows, and the outputs leave through LDS as whole 128-byte lines.
#include "pf_common.h"
#include "pf_direct.h"
#include "pf_internal.h"

namespace {

constexpr int C = 128;       // c_z
constexpr int CP_WAVES = 8;
constexpr int TB_MAX_OUT = 512, TB_WAVES = 12;

// rows 64 g + r of a [rows][128] tensor, clamped to the last: uniform base + 32-bit lane offset
PF_DEV f32x4 group_row4(const float* t, int g, long rows, int r, int c) {
  const char* base = reinterpret_cast<const char*>(t + (long)DP_ROWS * g * C);
  const uint32_t last = (uint32_t)min((long)DP_ROWS, rows - (long)DP_ROWS * g) - 1;
  return *reinterpret_cast<const f32x4_any*>(base + 4u * (min((uint32_t)r, last) * C + c));
}

// -------------------------------------------------------------------------------------
// out[p, :] = W . LN(cat(z[p, :], r[p, :]))  (W [128][256], LN over 256 with affine)
//          = W' . LNhat(cat(z, r)) + b',  W' = W diag(gamma) in op_t, b' = W beta
// Wave w: output channels 32 (w >> 1) .. + 31 of the pairs 32 (w & 1) .. + 31, all 256 inputs.
// Bound by HBM (z and r read, out written once: 61 us at the copy rate for N = 450).  Against W in LDS
// with a lane per row: N = 37 19.2 -> 8.8 us, 128 20.4 -> 10.5, 450 80 -> 60, 512 96 -> 83.
// -------------------------------------------------------------------------------------
constexpr int CP_LW = 264, CP_ZP = 132;
struct CpLds {   // byte offsets: normalized pairs [64][264] op_t, outputs [64][132] fp32 / weight buffers, offsets
  static constexpr size_t ROW = (size_t)DP_ROWS * CP_LW * sizeof(op_t);
  static constexpr size_t WB = (size_t)CP_WAVES * 32 * (C + 8) * sizeof(op_t);
  static constexpr size_t OFF = ROW + WB, BYTES = OFF + C * sizeof(float);
  static_assert(WB >= (size_t)DP_ROWS * CP_ZP * sizeof(float), "outputs over the weight buffers");
};
__global__ __launch_bounds__(64 * CP_WAVES, 1) void cond_proj_kernel(
    const float* __restrict__ z, const float* __restrict__ r, const float* __restrict__ lnw,
    const float* __restrict__ lnb, const op_t* __restrict__ W, float* __restrict__ out, long rows, int ngroups,
    float eps) {
  extern __shared__ __attribute__((aligned(16))) char cl[];
  op_t* sx = reinterpret_cast<op_t*>(cl);
  float* so = reinterpret_cast<float*>(cl + CpLds::ROW);
  float* soff = reinterpret_cast<float*>(cl + CpLds::OFF);
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, m = lane & 31;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tile = wid & 1, ob = wid >> 1, g4 = lane >> 4, q4 = lane & 15;
  f32x4 x[2][4];   // rows 8 wid + 4 it + g4: z channels 4 q4 .., 64 + 4 q4 .., then r's
  auto fetch = [&](int g) PF_INLINE {
#pragma unroll
    for (int it = 0; it < 2; ++it)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        x[it][v] = group_row4(v < 2 ? z : r, g, rows, 8 * wid + 4 * it + g4, 64 * (v & 1) + 4 * q4);
  };
  fetch(blockIdx.x);
  DirectW<C> w[2];   // input halves: z channels, r channels
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int i = 0; i < C / 16; ++i) {
      const int c = lane + 64 * i;
      w[u].v[i] = ld_x8(W + (long)(32 * ob + (c >> 4)) * 2 * C + C * u + 8 * (c & 15));
    }
  {
    op_t* wb = reinterpret_cast<op_t*>(so) + wid * 32 * (C + 8);
    float off = 0.f;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      w[u].turn(wb, lane);
      off += direct_wbeta<C / 16>(w[u].v, lnb + C * u, h);
      w[u].fold(lnw + C * u, h);
    }
    if (tile == 0 && h == 0) soff[32 * ob + m] = off;
  }
  for (int gi = blockIdx.x; gi < ngroups; gi += gridDim.x) {
#pragma unroll
    for (int it = 0; it < 2; ++it) {
      float s = 0.f, var = 0.f;
#pragma unroll
      for (int v = 0; v < 4; ++v) s += (x[it][v][0] + x[it][v][1]) + (x[it][v][2] + x[it][v][3]);
      const float mean = row16_sum(s) * (1.f / 256.f);
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int e = 0; e < 4; ++e) { const float d = x[it][v][e] - mean; var += d * d; }
      const float rstd = rsqrtf(row16_sum(var) * (1.f / 256.f) + eps);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        opx4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = (op_t)((x[it][v][e] - mean) * rstd);
        st_x4(sx + (8 * wid + 4 * it + g4) * CP_LW + 64 * v + 4 * q4, o);
      }
    }
    __syncthreads();   // sx is whole; the outputs of the last group are read out
    if (gi + (int)gridDim.x < ngroups) fetch(gi + gridDim.x);
    f32x16 acc;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 c4 = *reinterpret_cast<const f32x4*>(soff + 32 * ob + 8 * g + 4 * h);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[4 * g + e] = c4[e];
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int s = 0; s < C / 16; ++s)
        acc = mfma32(w[u].v[s], ld_x8(sx + (32 * tile + m) * CP_LW + C * u + 16 * s + 8 * h), acc);
#pragma unroll
    for (int g = 0; g < 4; ++g)   // D[channel][pair]
      *reinterpret_cast<f32x4*>(so + (32 * tile + m) * CP_ZP + 32 * ob + 8 * g + 4 * h) =
          f32x4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
    __syncthreads();
    char* obase = reinterpret_cast<char*>(out + (long)DP_ROWS * gi * C);
    const int left = (int)min((long)DP_ROWS, rows - (long)DP_ROWS * gi);
#pragma unroll
    for (int it = 0; it < 2; ++it) {
      const int rr = 8 * wid + 4 * it + g4;
#pragma unroll
      for (int v = 0; v < 2; ++v)
        if (rr < left)
          *reinterpret_cast<f32x4*>(obase + 4u * (rr * C + 64 * v + 4 * q4)) =
              *reinterpret_cast<const f32x4*>(so + rr * CP_ZP + 64 * v + 4 * q4);
    }
  }
}

// -------------------------------------------------------------------------------------
// bias[p, o] = scale * (W'[o] . LNhat(z[p]) + b'[o]),  o = l * H + hd < M
//   layout 0: out [rows][M]        (the reference's torch.cat(..., dim=-1) layout)
//   layout 1: out [M][rows]        (one contiguous [B][N][N] plane per (layer, head))
// Wave w: output blocks w and w + 12 (M <= 512: at most 16 blocks); waves 0-7 normalize.  Layout 0
// goes through the wave's LDS stage of [64 pairs][32 outputs], so that every store instruction
// writes eight whole 128-byte runs.  Bound by HBM (M fp32 written per pair: 81 us at the copy rate for
// N = 450, M = 384).  Against W in LDS with a lane per row and 4-byte stores: N = 37 33.9 -> 7.8 us,
// 128 38.7 -> 11.8, 450 130 -> 89, 512 142 -> 113 (layout 1: 450 156 -> 137, 512 138 -> 115).
// -------------------------------------------------------------------------------------
constexpr int TB_SP = 36;   // stage pitch (floats)
struct TbLds {
  static constexpr size_t ST = (size_t)2 * DP_ROWS * (C + 8) * sizeof(op_t);   // normalized pairs, two buffers
  static constexpr size_t OFF = ST + (size_t)TB_WAVES * DP_ROWS * TB_SP * sizeof(float);
  static constexpr size_t BYTES = OFF + TB_MAX_OUT * sizeof(float);
};
template <int LAYOUT>
__global__ __launch_bounds__(64 * TB_WAVES, 1) void token_bias_kernel(
    const float* __restrict__ z, const float* __restrict__ lnw, const float* __restrict__ lnb,
    const op_t* __restrict__ W, float* __restrict__ out, long rows, int ngroups, int M, int H, float scale, float eps) {
  constexpr int LW = C + 8;
  extern __shared__ __attribute__((aligned(16))) char bl[];
  op_t* sx = reinterpret_cast<op_t*>(bl);
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, m = lane & 31;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  float* stg = reinterpret_cast<float*>(bl + TbLds::ST) + wid * DP_ROWS * TB_SP;
  float* sb = reinterpret_cast<float*>(bl + TbLds::OFF);
  const int nob = M / 32, g4 = lane >> 4, q4 = lane & 15;
  DirectLn<C, 8> ln;
  auto fetch = [&](int g) PF_INLINE {
#pragma unroll
    for (int it = 0; it < 2; ++it)
#pragma unroll
      for (int v = 0; v < 2; ++v) ln.x[it][v] = group_row4(z, g, rows, 8 * wid + 4 * it + g4, 64 * v + 4 * q4);
  };
  if (wid < 8) fetch(blockIdx.x);
  ln.load_gamma(nullptr, lane);
  DirectW<C> w[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int ob = wid + TB_WAVES * k;
    if (ob >= nob) continue;
    w[k].load(W + (long)32 * ob * C, lane);
    w[k].turn(reinterpret_cast<op_t*>(stg), lane);
    const int l = (32 * ob + m) / H;   // this lane's row's layer
    const float b = direct_wbeta<C / 16>(w[k].v, lnb + l * C, h);
    w[k].fold(lnw + l * C, h);
    if (h == 0) sb[32 * ob + m] = b;
  }
  int buf = 0;
  for (int gi = blockIdx.x; gi < ngroups; gi += gridDim.x, buf ^= 1) {
    op_t* sxb = sx + buf * DP_ROWS * LW;
    if (wid < 8) ln.store(sxb, eps, wid, lane);
    __syncthreads();   // sx[buf] is whole; every wave is done with sx[buf ^ 1]
    if (wid < 8 && gi + (int)gridDim.x < ngroups) fetch(gi + gridDim.x);
    const long p0 = (long)DP_ROWS * gi;
    const int left = (int)min((long)DP_ROWS, rows - p0);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int ob = wid + TB_WAVES * k;
      if (ob >= nob) continue;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        f32x16 acc = zero16();
#pragma unroll
        for (int s = 0; s < C / 16; ++s)   // D[output][pair]
          acc = mfma32(w[k].v[s], ld_x8(sxb + (32 * t + m) * LW + 16 * s + 8 * h), acc);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 b4 = *reinterpret_cast<const f32x4*>(sb + 32 * ob + 8 * g + 4 * h);
          f32x4 v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = scale * (acc[4 * g + e] + b4[e]);
          if constexpr (LAYOUT == 0) {
            *reinterpret_cast<f32x4*>(stg + (32 * t + m) * TB_SP + 8 * g + 4 * h) = v;
          } else {
            int zl = lane;
            asm volatile("" : "+v"(zl));   // the address is formed here, not kept across the loop
            const int pr = 32 * t + (zl & 31);
            if (pr < left)
#pragma unroll
              for (int e = 0; e < 4; ++e)
                (out + (long)(32 * ob + 8 * g + e) * rows + p0)[(long)(4 * (zl >> 5)) * rows + pr] = v[e];
          }
        }
      }
      if constexpr (LAYOUT == 0) {   // (a wave's LDS accesses complete in order)
        char* obase = reinterpret_cast<char*>(out + p0 * M + 32 * ob);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int rr = 8 * i + (lane >> 3), c = 4 * (lane & 7);
          if (rr < left)
            *reinterpret_cast<f32x4_any*>(obase + 4u * ((uint32_t)rr * (uint32_t)M + c)) =
                *reinterpret_cast<const f32x4*>(stg + rr * TB_SP + c);
        }
      }
    }
  }
}

// groups of 64 rows and the workgroups that walk them (0: the device cannot be queried)
int group_grid(long rows, int* ngroups) {
  const long g = (rows + DP_ROWS - 1) / DP_ROWS;
  *ngroups = (int)g;
  return (int)min((long)max(device_cus(), 0), g);
}

}  // namespace

// ---------------------------------------------------------------------------------
// C-ABI
// ---------------------------------------------------------------------------------
extern "C" int pf_pair_cond_proj_fwd(const float* z, const float* rel_pos, const float* ln_w, const float* ln_b,
                                     const void* W, float* out, long rows, int c_z, float eps, void* stream) {
  if (!z || !rel_pos || !ln_w || !ln_b || !W || !out) return pf_fail(PF_E_INVALID, "pf_pair_cond_proj_fwd: null pointer");
  if (c_z != C || rows <= 0) return pf_fail(PF_E_INVALID, "pf_pair_cond_proj_fwd: need c_z = 128 and rows > 0 (got %d, %ld)", c_z, rows);
  if (out == z || out == rel_pos) return pf_fail(PF_E_INVALID, "pf_pair_cond_proj_fwd: out must not alias an input");
  if (rows >= (1l << 36)) return pf_fail(PF_E_INVALID, "pf_pair_cond_proj_fwd: shape too large");
  int ngroups = 0;
  const int grid = group_grid(rows, &ngroups);
  if (grid <= 0) return pf_fail(PF_E_LAUNCH, "pf_pair_cond_proj_fwd: cannot query the device");
  if (const int rc = pf_reserve_lds((const void*)cond_proj_kernel, CpLds::BYTES, "cond_proj_kernel")) return rc;
  cond_proj_kernel<<<grid, 64 * CP_WAVES, CpLds::BYTES, (hipStream_t)stream>>>(z, rel_pos, ln_w, ln_b, (const op_t*)W,
                                                                              out, rows, ngroups, eps);
  PF_CHECK_LAUNCH("cond_proj_kernel");
  return PF_OK;
}

extern "C" int pf_token_pair_bias_fwd(const float* z, const float* ln_w, const float* ln_b, const void* W, float* out,
                                      long rows, int c_z, int n_layers, int n_heads, int layout, float scale, float eps,
                                      void* stream) {
  if (!z || !ln_w || !ln_b || !W || !out) return pf_fail(PF_E_INVALID, "pf_token_pair_bias_fwd: null pointer");
  const long M = (long)n_layers * n_heads;
  if (c_z != C || rows <= 0 || n_layers <= 0 || n_heads <= 0 || M % 32 || M > TB_MAX_OUT || (layout != 0 && layout != 1))
    return pf_fail(PF_E_INVALID,
                   "pf_token_pair_bias_fwd: need c_z = 128, n_layers * n_heads a multiple of 32 up to %d, layout 0/1 "
                   "(got c_z=%d L=%d H=%d layout=%d rows=%ld)", TB_MAX_OUT, c_z, n_layers, n_heads, layout, rows);
  if (rows * M >= (1l << 40)) return pf_fail(PF_E_INVALID, "pf_token_pair_bias_fwd: shape too large");
  int ngroups = 0;
  const int grid = group_grid(rows, &ngroups);
  if (grid <= 0) return pf_fail(PF_E_LAUNCH, "pf_token_pair_bias_fwd: cannot query the device");
  auto kern = layout == 0 ? token_bias_kernel<0> : token_bias_kernel<1>;
  if (const int rc = pf_reserve_lds((const void*)kern, TbLds::BYTES, "token_bias_kernel")) return rc;
  kern<<<grid, 64 * TB_WAVES, TbLds::BYTES, (hipStream_t)stream>>>(z, ln_w, ln_b, (const op_t*)W, out, rows, ngroups,
                                                                  (int)M, n_heads, scale, eps);
  PF_CHECK_LAUNCH("token_bias_kernel");
  return PF_OK;
}
