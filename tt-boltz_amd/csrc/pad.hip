// Zero-padded copies at the Python boundary (the pad to a multiple of 64 or 128 tokens,
// tt_bio/tenstorrent.py:2235-2246) for gfx950.
#include "pf_common.h"
#include "pf_internal.h"

namespace {

struct PadShape {
  long sb, s1, sm, s2;            // source strides (elements)
  uint32_t n1, m, n2, n1p, n2p;   // valid and padded lengths
  uint32_t cv;                    // channels in units of VEC
  uint32_t total;                 // units of VEC in dst
};

// dst [B][n1p][M][n2p][C] = src[b, i, m, j, c] for i < N1 and j < N2, else 0; src null: 1.  One pass
// that writes every element once (a fill and a strided copy write the valid part twice: z at
// N = 413 41 us, this 28; at N = 1024, where nothing is padded, 285 us against 178), four units a
// thread with their loads in flight, every store instruction of a wave contiguous.
template <int VEC>
__global__ __launch_bounds__(256) void pad_kernel(const float* __restrict__ src, float* __restrict__ dst, PadShape p) {
  typedef float vec_t __attribute__((ext_vector_type(VEC)));
  constexpr int U = 4;
  const uint32_t row_units = p.n2p * p.cv;
  const uint32_t e0 = blockIdx.x * (256u * U) + threadIdx.x;
  vec_t v[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const uint32_t e = e0 + 256u * u;
    v[u] = (vec_t)(0.f);
    if (e < p.total) {
      const uint32_t row = e / row_units, col = e - row * row_units;
      const uint32_t j = col / p.cv, c = col - j * p.cv;
      const uint32_t t = row / p.m, mm = row - t * p.m;
      const uint32_t b = t / p.n1p, i = t - b * p.n1p;
      if (i < p.n1 && j < p.n2) {
        if (src)
          v[u] = *reinterpret_cast<const vec_t*>(src + b * p.sb + i * p.s1 + mm * p.sm + j * p.s2 + (long)VEC * c);
        else
          v[u] = (vec_t)(1.f);
      }
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const uint32_t e = e0 + 256u * u;
    if (e < p.total) *reinterpret_cast<vec_t*>(dst + (size_t)VEC * e) = v[u];
  }
}

}  // namespace

extern "C" int pf_pad_fwd(const float* src, long sb, long s1, long sm, long s2, float* dst, int B, int N1, int M,
                          int N2, int n1p, int n2p, int C, void* stream) {
  if (!dst) return pf_fail(PF_E_INVALID, "pf_pad_fwd: null pointer");
  if (B <= 0 || N1 <= 0 || M <= 0 || N2 <= 0 || C <= 0 || N1 > n1p || N2 > n2p)
    return pf_fail(PF_E_INVALID, "pf_pad_fwd: bad shape (B=%d N1=%d M=%d N2=%d n1p=%d n2p=%d C=%d)", B, N1, M, N2, n1p,
                   n2p, C);
  const bool vec = C % 4 == 0 && ((uintptr_t)dst & 15) == 0 && ((uintptr_t)src & 15) == 0 &&
                   (!src || ((sb | s1 | sm | s2) & 3) == 0);
  const int cv = vec ? C / 4 : C;
  // (compared by division: the product of five lengths may exceed 64 bits)
  unsigned long long total = 1;
  const int dims[] = {B, n1p, M, n2p, cv};
  for (int d : dims) {
    total *= (unsigned)d;
    if (total >= (1ull << 32) - 1024)
      return pf_fail(PF_E_INVALID, "pf_pad_fwd: more than 2^32 elements (B=%d n1p=%d M=%d n2p=%d C=%d)", B, n1p, M, n2p, C);
  }
  const PadShape p{sb, s1, sm, s2, (uint32_t)N1, (uint32_t)M, (uint32_t)N2, (uint32_t)n1p, (uint32_t)n2p,
                   (uint32_t)cv, (uint32_t)total};
  const unsigned grid = (unsigned)((total + 1023) / 1024);
  if (vec)
    pad_kernel<4><<<grid, 256, 0, (hipStream_t)stream>>>(src, dst, p);
  else
    pad_kernel<1><<<grid, 256, 0, (hipStream_t)stream>>>(src, dst, p);
  PF_CHECK_LAUNCH("pad_kernel");
  return PF_OK;
}
