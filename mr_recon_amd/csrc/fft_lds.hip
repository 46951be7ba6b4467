// Batched complex FFTs along one axis of a row-major grid, staged through LDS: one
// global read and one global write per element per axis (rocFFT's plan for a 160^3
// batch takes four passes per 3D transform). Unnormalised, in place. The inverse
// transform is conj(F(conj(x))), applied on load and store.
//
// Axis access patterns: along the contiguous last axis a block takes NT consecutive
// rows (each row is L contiguous values); along any other axis (stride `inner`) a block
// takes NT consecutive columns, so every row of the load is NT contiguous values.
// Lengths are compile-time (radix plans in fft_lds.h); others go through rocFFT.
#include "capi_util.h"
#include "fft_lds.h"

namespace mra {
namespace fft {

// ROW: transforms along the contiguous last axis (inner == 1), NT consecutive rows per
// block. COL: transforms along an axis of stride `inner` (inner >= NT), NT consecutive
// columns per block.
template <int L, bool ROW>
__global__ __launch_bounds__(Plan<L>::T * (ROW ? Plan<L>::NR : Plan<L>::NC)) void fft_axis_kernel(
    float2* __restrict__ data, long long outer, long long inner, const float2* __restrict__ twg, int inverse) {
  using P = Plan<L>;
  constexpr int NT = ROW ? P::NR : P::NC;
  constexpr bool REV = ROW && RowOrder<L>::REV;
  using TB = Tables<L, REV>;
  __shared__ float2 buf[BufSize<L, NT>::value];
  __shared__ float2 tab[TB::SIZE];
  const int tid = threadIdx.x;
  const int c = ROW ? tid / P::T : tid % NT, j = ROW ? tid % P::T : tid / NT;
  bool valid;
  float2* base;        // rows: this thread's row at j; columns: the block's slab
  unsigned off = 0, row = 8;
  if constexpr (ROW) {
    const long long o = (long long)blockIdx.x * NT + c;
    valid = o < outer;
    base = data + (valid ? o * L : 0) + j;
  } else {
    const long long nblk = (inner + NT - 1) / NT;
    const long long o = blockIdx.x / nblk, i0 = (blockIdx.x - o * nblk) * NT;
    base = data + o * L * inner;
    valid = i0 + c < inner;
    row = (unsigned)inner * 8u;
    off = valid ? j * row + (unsigned)(i0 + c) * 8u : kNone;
  }
  const Slab slab(data + (ROW ? 0 : base - data), ROW ? 0 : L * row);
  const float sgn = inverse ? -1.0f : 1.0f;  // conj on load and store for the inverse
  float2 v[TB::A], x[TB::Z];
  load_first<L>(v, j, [&](int, int d) { return ROW ? base[d] : slab.load(off, d * row); });
#pragma unroll
  for (int q = 0; q < TB::A; ++q) v[q].y *= sgn;
  TB::fill(tab, twg, tid, P::T * NT);
  finish<L, NT, ROW, REV>(v, x, buf, tab, j, c);
  if constexpr (ROW && RowOrder<L>::STAGE) {
    stage_rows<L, NT, REV>(x, buf, j, c);
    float2* blk = data + (long long)blockIdx.x * NT * L;
    for (int e = tid; e < NT * L; e += P::T * NT) {
      const int r = e / L, i = e - r * L;
      if ((long long)blockIdx.x * NT + r < outer) {
        const float2 y = buf[Lay<L, TB::A, NT, true>::at(i, r)];
        blk[e] = make_float2(y.x, sgn * y.y);
      }
    }
  } else {
    emit<L, REV>(x, j, [&](int, int d, float2 y) {
      y.y *= sgn;
      if (!ROW) slab.store(off, d * row, y);
      else if (valid) base[d] = y;
    });
  }
}

template <int L>
int launch_axis(float2* data, long long outer, long long inner, const float2* tw, int inverse, hipStream_t st) {
  using P = Plan<L>;
  if (inner == 1) {
    const long long nb = (outer + P::NR - 1) / P::NR;
    if (nb > 0x7fffffffLL) MRA_FAIL("fft: too many transforms");
    fft_axis_kernel<L, true><<<(unsigned)nb, P::T * P::NR, 0, st>>>(data, outer, inner, tw, inverse);
  } else {
    if (inner < P::NC) MRA_FAIL("fft: inner extent below the column tile");
    if (inner > kMaxInner) MRA_FAIL("fft: inner extent too large");
    const long long nb = outer * ((inner + P::NC - 1) / P::NC);
    if (nb > 0x7fffffffLL) MRA_FAIL("fft: too many transforms");
    fft_axis_kernel<L, false><<<(unsigned)nb, P::T * P::NC, 0, st>>>(data, outer, inner, tw, inverse);
  }
  MRA_CHECK_LAUNCH("fft axis");
  return 0;
}

int dispatch_axis(int L, float2* data, long long outer, long long inner, const float2* tw, int inverse,
                  hipStream_t st) {
  const int rc = with_length(L, [&](auto LL) {
    return launch_axis<decltype(LL)::value>(data, outer, inner, tw, inverse, st);
  });
  if (rc < 0) MRA_FAIL("fft: length without an LDS plan");
  return rc;
}

bool supported(int L) { return plan_supported(L); }

}  // namespace fft
}  // namespace mra

using namespace mra;

extern "C" {

// 1 when every length of n[0..ndim) has an LDS plan and every non-last axis has at
// least 16 columns after it (the column tile), else 0.
int mra_fft_lds_supported(int ndim, const int* n) {
  if (ndim < 1 || ndim > 3) return 0;
  long long inner = 1;
  for (int d = ndim - 1; d >= 0; --d) {
    if (!fft::supported(n[d])) return 0;
    if (d < ndim - 1 && inner < 64) return 0;
    inner *= n[d];
  }
  return 1;
}

// Twiddle table for length L: tw[m] = exp(-2 pi i m / L), host memory, L complex.
int mra_fft_lds_twiddles(int L, float* tw_host) {
  MRA_TRY_BEGIN
  if (L < 1) MRA_FAIL("fft: bad length");
  for (int m = 0; m < L; ++m) {
    const double a = -2.0 * 3.14159265358979323846 * (double)m / (double)L;
    tw_host[2 * m] = (float)cos(a);
    tw_host[2 * m + 1] = (float)sin(a);
  }
  MRA_TRY_END
}

// In-place unnormalised FFT over the trailing ndim axes of `batch` grids of shape n,
// one LDS pass per axis. tw[d] = device twiddle table of length n[d].
int mra_fft_lds(int ndim, const int* n, long long batch, void* data, const void* const* tw, int inverse,
                void* stream) {
  MRA_TRY_BEGIN
  if (!mra_fft_lds_supported(ndim, n)) MRA_FAIL("fft: shape not supported by the LDS transforms");
  if (batch < 1) MRA_FAIL("fft: batch must be positive");
  long long total = batch;
  for (int d = 0; d < ndim; ++d) total *= n[d];
  long long inner = 1;
  for (int d = ndim - 1; d >= 0; --d) {
    const long long outer = total / ((long long)n[d] * inner);
    if (fft::dispatch_axis(n[d], (float2*)data, outer, inner, (const float2*)tw[d], inverse,
                           (hipStream_t)stream))
      return 1;
    inner *= n[d];
  }
  MRA_TRY_END
}

}  // extern "C"
