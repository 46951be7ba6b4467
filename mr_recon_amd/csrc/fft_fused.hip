// FFTs fused with the zero-pad / crop around them, skipping the known zeros.
//
// Forward (image -> oversampled grid spectrum): the padded grid is zero outside the
// image's N points per dim (pixel n sits at grid index (n - c) mod G). The transform
// along the last axis therefore only runs on rows whose leading indices hold pixels,
// reading the image (times SENSE map, apodization and scale) directly instead of a
// padded grid; each further axis transforms columns whose leading indices hold pixels
// and loads only the pixel rows of the transform axis. The final axis writes every
// grid point.
//
// Adjoint (grid spectrum -> image): the mirror image. The first axis transforms every
// column but stores only pixel rows; later axes load all rows of pixel columns and
// store pixel rows; the last axis transforms the pixel rows of all coils of an image
// and reduces them over coils (times conj(map), apodization and scale) straight into
// the image.
//
// Toeplitz normal operator: forward passes, then along axis 0 one kernel transforms,
// multiplies by the PSF spectrum and transforms back (storing pixel rows only), then
// the adjoint passes.
//
// Replaces, fused: the reference's resize + ifftshift + fftn + fftshift + crop chains of
// triton_nufft.forward_FT_only / adjoint_iFT_only (fourier.py:432-468, 505-525) and
// NUFFT.normal_toeplitz (fourier.py:302-352) with SENSE expand / reduce
// (linops.py:1161, 1220, 1265-1306).
#include "capi_util.h"
#include "fft_any.h"
#include "fft_lds.h"

namespace mra {
namespace fused {

using namespace fft;

struct Geo3 {
  int N[3], G[3], c[3];   // image size, grid size, pixel at grid index 0 (leading unused = 1/1/0)
  const float* apod[3];   // per-dim apodization by pixel (nullptr = 1)
  float scale;
};

__device__ __forceinline__ int pix_of(int g, int N, int G, int c) {
  if (g < N - c) return g + c;
  if (g >= G - c) return g - G + c;
  return -1;
}
__device__ __forceinline__ int grid_of(int n, int G, int c) { return n - c < 0 ? n - c + G : n - c; }
__device__ __forceinline__ float apod_at(const Geo3& p, int d, int n) { return p.apod[d] ? p.apod[d][n] : 1.0f; }
__device__ __forceinline__ float2 conjf2(float2 a) { return make_float2(a.x, -a.y); }

// Forward, last axis: NT pixel rows per block (rows enumerate (q, n0, n1)); grid batch q
// uses image img_index[q] (or q / ns) and map q (or q % ns).
template <int L>
__global__ __launch_bounds__(Plan<L>::T * Plan<L>::NR) void pad_row_kernel(
    const float2* __restrict__ x, long long x_stride, const float2* __restrict__ smaps, long long s_stride,
    long long ns, const int* __restrict__ img_index, Geo3 p, long long nrows, float2* __restrict__ grid,
    const float2* __restrict__ twg) {
  using P = Plan<L>;
  constexpr int NT = P::NR;
  constexpr bool REV = RowOrder<L>::REV;
  using TB = Tables<L, REV>;
  __shared__ float2 buf[BufSize<L, NT>::value];
  __shared__ float2 tab[TB::SIZE];
  __shared__ long long rdst[NT];  // grid offset of each row
  const int tid = threadIdx.x;
  const int c = tid / P::T, j = tid % P::T;
  const long long row0 = (long long)blockIdx.x * NT;
  const int N0 = p.N[0], N1 = p.N[1], N2 = p.N[2];
  const bool valid = row0 + c < nrows;
  const float2 *xr = x, *mr = smaps;
  float a01 = 0.f;
  if (valid) {
    const unsigned row = (unsigned)(row0 + c);  // nrows < 2^31
    const unsigned r2 = row / (unsigned)N1, n1 = row - r2 * N1;
    const unsigned q = r2 / (unsigned)N0, n0 = r2 - q * N0;
    const unsigned bq = q / (unsigned)ns;
    const long long bs = img_index ? q : q - bq * (unsigned)ns;
    const long long bx = img_index ? img_index[q] : bq;
    const long long pix = ((long long)n0 * N1 + n1) * N2;
    xr = x + bx * x_stride + pix;
    if (smaps) mr = smaps + bs * s_stride + pix;
    a01 = p.scale * apod_at(p, 0, n0) * apod_at(p, 1, n1);
    if (j == 0)
      rdst[c] = (((long long)q * p.G[0] + grid_of(n0, p.G[0], p.c[0])) * p.G[1] + grid_of(n1, p.G[1], p.c[1])) * L;
  }
  // every load first (a grid point without a pixel reads pixel 0), then the products
  float2 v[TB::A], mv[TB::A], o[TB::Z];
  float av[TB::A];
  const bool act = L / TB::A == P::T || j < L / TB::A;
  auto pix = [&](int q) { return act ? pix_of(j + q * (L / TB::A), N2, L, p.c[2]) : -1; };
#pragma unroll
  for (int q = 0; q < TB::A; ++q) v[q] = xr[max(pix(q), 0)];
  if (smaps) {
#pragma unroll
    for (int q = 0; q < TB::A; ++q) mv[q] = mr[max(pix(q), 0)];
  }
  if (p.apod[2]) {
#pragma unroll
    for (int q = 0; q < TB::A; ++q) av[q] = p.apod[2][max(pix(q), 0)];
  }
  TB::fill(tab, twg, tid, P::T * NT);
#pragma unroll
  for (int q = 0; q < TB::A; ++q) {
    float2 y = v[q];
    if (smaps) y = cmul(y, mv[q]);
    const float a = p.apod[2] ? a01 * av[q] : a01;
    const bool in = pix(q) >= 0;
    v[q] = make_float2(in ? y.x * a : 0.f, in ? y.y * a : 0.f);
  }
  finish<L, NT, true, REV>(v, o, buf, tab, j, c);
  if constexpr (RowOrder<L>::STAGE) {
    stage_rows<L, NT, REV>(o, buf, j, c);
    for (int e = tid; e < NT * L; e += P::T * NT) {
      const int r = e / L, i = e - r * L;
      if (row0 + r < nrows) grid[rdst[r] + i] = buf[Lay<L, TB::A, NT, true>::at(i, r)];
    }
  } else {
    float2* dst = grid + (valid ? rdst[c] : 0);  // written before finish's barrier
    emit<L, REV>(o, j, [&](int i, int, float2 y) {
      if (valid) dst[i] = y;
    });
  }
}

constexpr unsigned kXCDs = 8;

enum ColMode { kFwd = 0, kAdj = 1, kToep = 2 };

// Column pass along axis a in {0, 1} (of the 3-dim view), NT columns per block. Outer
// index: q (axis 0) or (q, n0) over pixel planes (axis 1). kFwd: load pixel rows only,
// forward, store all rows. kAdj: load all rows, inverse, store pixel rows. kToep: load
// pixel rows, forward, multiply by kern (indexed over one grid), inverse, store pixel rows.
template <int L, int MODE>
__global__ __launch_bounds__(Plan<L>::T * Plan<L>::NC) void col_kernel(float2* __restrict__ grid, Geo3 p, int axis,
                                                                      long long inner, unsigned nblk,
                                                                      const float2* __restrict__ twg,
                                                                      const float2* __restrict__ kern) {
  using P = Plan<L>;
  constexpr int NT = P::NC;
  __shared__ float2 buf[BufSize<L, NT>::value];
  __shared__ float2 tab[Tables<L, false>::SIZE];
  const int tid = threadIdx.x;
  const int c = tid % NT, j = tid / NT;
  // kToep: the outer indices (coils) of a column tile run back to back on one XCD, whose L2
  // then serves the tile of kern to all but the first (blocks go to the XCDs in turn)
  unsigned o = blockIdx.x / nblk, t = blockIdx.x - o * nblk;
  if (MODE == kToep) {
    const unsigned no = gridDim.x / nblk, l = blockIdx.x / kXCDs, full = nblk / kXCDs * kXCDs;
    if (blockIdx.x < full * no) {
      o = l % no;
      t = l / no * kXCDs + blockIdx.x % kXCDs;
    } else {
      const unsigned r = blockIdx.x - full * no;
      o = r / (nblk - full);
      t = full + r - o * (nblk - full);
    }
  }
  const long long col0 = (long long)t * NT;
  const bool valid = col0 + c < inner;
  long long base;
  if (axis == 0) {
    base = (long long)o * L * inner;
  } else {  // axis 1: o = q * N0 + n0
    const unsigned q = o / (unsigned)p.N[0];
    const int n0 = (int)(o - q * p.N[0]);
    base = ((long long)q * p.G[0] + grid_of(n0, p.G[0], p.c[0])) * (long long)L * inner;
  }
  const int Na = p.N[axis], ca = p.c[axis];
  const unsigned row = (unsigned)inner * 8u, bytes = L * row;
  const Slab g(grid + base, bytes);
  const unsigned off = valid ? j * row + (unsigned)(col0 + c) * 8u : kNone;
  auto in_pix = [&](int i) { return pix_of(i, Na, L, ca) >= 0; };
  using TB = Tables<L, false>;
  float2 v[TB::A], z[TB::Z];
  load_first<L>(v, j, [&](int i, int d) {
    const float2 x = g.load(MODE == kAdj || in_pix(i) ? off : kNone, d * row);
    return MODE == kAdj ? conjf2(x) : x;
  });
  if constexpr (MODE == kToep) {
    using TR = Tables<L, true>;
    constexpr int NB = L / TR::A;
    __shared__ float2 tabr[P::R1 == TR::A ? 1 : TR::SIZE];  // equal first and last radix: one table does both
    const Slab ks(kern, bytes);
    float2 u[TR::A], y[TR::Z];
    // loaded with the data; with three passes (1024 threads) that would cost the second block of a CU
    auto load_kern = [&] { load_first<L>(u, j, [&](int, int d) { return ks.load(off, d * row); }); };
    if constexpr (!TB::three) load_kern();
    TB::fill(tab, twg, tid, P::T * NT);
    if constexpr (P::R1 != TR::A) TR::fill(tabr, twg, tid, P::T * NT);
    finish<L, NT, false, false>(v, z, buf, tab, j, c);
    if constexpr (TB::three) load_kern();
    if (NB == P::T || j < NB) {
#pragma unroll
      for (int q = 0; q < TR::A; ++q) u[q] = conjf2(cmul(z[q], u[q]));
    }
    __syncthreads();
    finish<L, NT, false, true>(u, y, buf, P::R1 == TR::A ? tab : tabr, j, c);
    emit<L, true>(y, j, [&](int i, int d, float2 w) { g.store(in_pix(i) ? off : kNone, d * row, conjf2(w)); });
  } else {
    TB::fill(tab, twg, tid, P::T * NT);
    finish<L, NT, false, false>(v, z, buf, tab, j, c);
    emit<L, false>(z, j, [&](int i, int d, float2 w) {
      if (MODE == kFwd) g.store(off, d * row, w);
      else g.store(in_pix(i) ? off : kNone, d * row, conjf2(w));
    });
  }
}

// Adjoint, last axis + crop / coil reduce. A block takes NT / 2^LCB image rows (bx, n0, n1)
// and 2^LCB coils of each at a time: the grids [q0, q1) of image bx are inverse-transformed
// and reduced, out[bx][n] (+)= scale * apod(n) * sum_q row_q[g(n)] * (conj) S[q][n]. One coil
// (LCB = 0) is stored from the registers that end the transform. Otherwise the transforms
// go back to LDS, where a row's T 2^LCB threads take its pixels, ng threads to a pixel
// (every ng-th coil each), so that maps are read along the row; the ng partial sums are
// added at the end, in order.
template <int L, int LCB>
__global__ __launch_bounds__(Plan<L>::T * Plan<L>::NA) void crop_row_kernel(
    const float2* __restrict__ grid, Geo3 p, long long nrows, long long ns, const float2* __restrict__ smaps,
    long long s_stride, const int* __restrict__ coil_off, int ng, int conj_maps, int accumulate,
    float2* __restrict__ out, long long x_stride, const float2* __restrict__ twg) {
  using P = Plan<L>;
  constexpr int NT = P::NA, CB = 1 << LCB, RB = NT / CB;
  constexpr bool REV = RowOrder<L>::REV;
  using TB = Tables<L, REV>;
  using LY = Lay<L, TB::A, NT, true>;
  constexpr int GT = P::T * CB;                // threads of an image row
  constexpr int KM = (L + GT - 1) / GT;        // pixels a thread may own
  __shared__ float2 buf[BufSize<L, NT>::value];
  __shared__ float2 tab[TB::SIZE];
  const int tid = threadIdx.x;
  const int c = tid / P::T, j = tid % P::T;
  const int N0 = p.N[0], N1 = p.N[1], N2 = p.N[2];
  const int cr = c >> LCB, cc = c & (CB - 1);
  const long long row = (long long)blockIdx.x * RB + cr;
  const bool live = row < nrows;
  long long q0 = 0, q1 = 0, goff = 0, pix0 = 0, map0 = 0, opix = 0;
  float a01 = 0.f;
  if (live) {
    const unsigned r2 = (unsigned)row / (unsigned)N1, n1 = (unsigned)row - r2 * N1;  // nrows < 2^31
    const unsigned bx = r2 / (unsigned)N0, n0 = r2 - bx * N0;
    q0 = coil_off ? coil_off[bx] : (long long)bx * ns;
    q1 = coil_off ? coil_off[bx + 1] : q0 + ns;
    map0 = coil_off ? 0 : bx * ns;
    goff = ((long long)grid_of(n0, p.G[0], p.c[0]) * p.G[1] + grid_of(n1, p.G[1], p.c[1])) * L;
    pix0 = ((long long)n0 * N1 + n1) * N2;
    opix = bx * x_stride + pix0;
    a01 = p.scale * apod_at(p, 0, n0) * apod_at(p, 1, n1);
  }
  const long long gsz = (long long)p.G[0] * p.G[1] * L;
  // chunks of coils: the most any image of the block has, so that every thread reaches
  // every barrier
  int nch = (int)((ns + CB - 1) / CB);
  if (coil_off) {
    const unsigned per = (unsigned)N0 * N1, last = (unsigned)min(nrows, (long long)(blockIdx.x + 1) * RB) - 1;
    int most = 0;
    for (unsigned b = blockIdx.x * RB / per; b <= last / per; ++b) most = max(most, coil_off[b + 1] - coil_off[b]);
    nch = (most + CB - 1) / CB;
  }
  float2* orow = out + opix;
  auto put = [&](int n2, float2 s) {
    const float a = a01 * apod_at(p, 2, n2);
    float2 y = make_float2(s.x * a, s.y * a);
    if (accumulate) {
      const float2 o = orow[n2];
      y.x += o.x;
      y.y += o.y;
    }
    orow[n2] = y;
  };
  auto term = [&](float2 x, float2 s) {
    const float2 y = conjf2(x);
    if (!smaps) return y;
    return conj_maps ? cmul(y, conjf2(s)) : cmul(y, s);
  };
  float2 v[TB::A], x[TB::Z];
  auto fetch = [&](int k) {
    const long long qc = q0 + (long long)k * CB + cc;
    const bool valid = live && qc < q1;
    const float2* src = grid + (valid ? qc * gsz + goff : 0);  // coils past the last are transformed and not used
    load_first<L>(v, j, [&](int i, int) { return conjf2(src[i]); });
  };
  if (nch > 0) fetch(0);
  TB::fill(tab, twg, tid, P::T * NT);
  if constexpr (LCB == 0) {
    // with no more than one coil the row needs no sum; more (uneven problems) add up in LDS order
    float2 acc[TB::Z];
#pragma unroll
    for (int q = 0; q < TB::Z; ++q) acc[q] = make_float2(0.f, 0.f);
    for (int k = 0; k < nch; ++k) {
      if (k > 0) {
        fetch(k);
        __syncthreads();
      }
      finish<L, NT, true, REV>(v, x, buf, tab, j, c);
      const bool valid = live && q0 + k < q1 && (L / TB::Z == P::T || j < L / TB::Z);
      auto pix = [&](int q) { return pix_of(j + q * (L / TB::Z), N2, L, p.c[2]); };
      float2 s[TB::Z];
      if (smaps) {
        const float2* srow = smaps + (valid ? (q0 + k - map0) * s_stride + pix0 : 0);
#pragma unroll
        for (int q = 0; q < TB::Z; ++q) s[q] = srow[max(pix(q), 0)];
      }
#pragma unroll
      for (int q = 0; q < TB::Z; ++q) {
        const float2 y = term(x[q], s[q]);
        const bool in = valid && pix(q) >= 0;
        acc[q].x = in ? acc[q].x + y.x : acc[q].x;
        acc[q].y = in ? acc[q].y + y.y : acc[q].y;
      }
    }
    if (live && (L / TB::Z == P::T || j < L / TB::Z)) {
#pragma unroll
      for (int q = 0; q < TB::Z; ++q) {
        const int n2 = pix_of(j + q * (L / TB::Z), N2, L, p.c[2]);
        if (n2 >= 0) put(n2, acc[q]);
      }
    }
  } else {
    const int l = cc * P::T + j, pw = GT / ng;
    const int grp = l / pw, n = l - grp * pw;   // grp == ng for the GT % ng threads left over
    float2 acc[KM];
#pragma unroll
    for (int m = 0; m < KM; ++m) acc[m] = make_float2(0.f, 0.f);
    for (int k = 0; k < nch; ++k) {
      if (k > 0) fetch(k);
      finish<L, NT, true, REV>(v, x, buf, tab, j, c);
      stage_rows<L, NT, REV>(x, buf, j, c);
      const long long qk = q0 + (long long)k * CB;
      const int nr = live && grp < ng ? (int)max(0LL, min((long long)CB, q1 - qk)) : 0;
#pragma unroll
      for (int m = 0; m < KM; ++m) {
        const int n2 = n + m * pw;
        if (n2 < N2) {
          const int i = grid_of(n2, L, p.c[2]);
          const float2* s = smaps + (smaps ? (qk - map0) * s_stride + pix0 + n2 : 0);
          for (int b = grp; b < nr; b += 4 * ng) {  // four coils' maps in flight
            float2 sv[4];
            if (smaps) {
#pragma unroll
              for (int u = 0; u < 4; ++u) sv[u] = s[min(b + u * ng, nr - 1) * s_stride];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              const int bu = b + u * ng;
              const float2 y = term(buf[LY::at(i, cr * CB + min(bu, nr - 1))], sv[u]);
              acc[m].x = bu < nr ? acc[m].x + y.x : acc[m].x;
              acc[m].y = bu < nr ? acc[m].y + y.y : acc[m].y;
            }
          }
        }
      }
      __syncthreads();
    }
    if (ng > 1) {  // pw >= N2: one pixel a thread; a row's own part of buf holds its sums
      float2* part = buf + LY::at(0, cr * CB);
      if (grp > 0 && grp < ng && n < N2) part[(grp - 1) * N2 + n] = acc[0];
      __syncthreads();
      if (grp == 0 && n < N2)
        for (int h = 1; h < ng; ++h) {
          const float2 o = part[(h - 1) * N2 + n];
          acc[0].x += o.x;
          acc[0].y += o.y;
        }
    }
    if (live && grp == 0) {
#pragma unroll
      for (int m = 0; m < KM; ++m) {
        const int n2 = n + m * pw;
        if (n2 < N2) put(n2, acc[m]);
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// The same three kernels for run-time lengths (fft_any.h); dynamic LDS: M * (NT + 1) points of
// the transforms, then the M roots. Copies between memory and LDS issue four loads at a time.

template <int TPB, int NT, int KIND>
__global__ __launch_bounds__(TPB) void any_pad_row_kernel(const float2* __restrict__ x, long long x_stride,
                                                          const float2* __restrict__ smaps, long long s_stride,
                                                          long long ns, Geo3 p, AnyPlan ap, long long nrows,
                                                          float2* __restrict__ grid, const float2* __restrict__ tab) {
  using A = Any<TPB, NT>;
  extern __shared__ float2 buf[];
  float2* tw = buf + ap.M * A::NTP;
  __shared__ long long rsrc[NT], rmap[NT], rdst[NT];
  __shared__ float rapo[NT];
  const int tid = threadIdx.x, L = ap.L;
  const long long row0 = (long long)blockIdx.x * NT;
  const int N0 = p.N[0], N1 = p.N[1], N2 = p.N[2];
  if (tid < NT) {
    const unsigned row = (unsigned)min(row0 + tid, nrows - 1);  // nrows < 2^31; rows past the last are not stored
    const unsigned r2 = row / (unsigned)N1, n1 = row - r2 * N1;
    const unsigned q = r2 / (unsigned)N0, n0 = r2 - q * N0;
    const unsigned bq = q / (unsigned)ns;
    const long long pix = ((long long)n0 * N1 + n1) * N2;
    rsrc[tid] = bq * x_stride + pix;
    rmap[tid] = (q - bq * (unsigned)ns) * s_stride + pix;
    rapo[tid] = p.scale * apod_at(p, 0, n0) * apod_at(p, 1, n1);
    rdst[tid] = (((long long)q * p.G[0] + grid_of(n0, p.G[0], p.c[0])) * p.G[1] + grid_of(n1, p.G[1], p.c[1])) * L;
  }
  for (int m = tid; m < ap.M; m += TPB) tw[m] = tab[m];
  __syncthreads();
  const int n = NT * L;
  for (int e0 = tid; e0 < n; e0 += 4 * TPB) {
    float2 v[4], s[4];
    float a[4];
    int c[4], i[4], n2[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int e = min(e0 + u * TPB, n - 1);
      c[u] = (int)__umulhi((unsigned)e, ap.inv_l);
      i[u] = e - c[u] * L;
      n2[u] = pix_of(i[u], N2, L, p.c[2]);
      v[u] = x[rsrc[c[u]] + max(n2[u], 0)];
    }
    if (smaps) {
#pragma unroll
      for (int u = 0; u < 4; ++u) s[u] = smaps[rmap[c[u]] + max(n2[u], 0)];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) a[u] = rapo[c[u]] * apod_at(p, 2, max(n2[u], 0));
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float2 y = smaps ? cmul(v[u], s[u]) : v[u];
      if (e0 + u * TPB < n)
        buf[i[u] * A::NTP + c[u]] = n2[u] >= 0 ? make_float2(y.x * a[u], y.y * a[u]) : make_float2(0.f, 0.f);
    }
  }
  __syncthreads();
  A::template transform<KIND>(buf, tw, tab, ap);
  for (int e = tid; e < n; e += TPB) {
    const int c = (int)__umulhi((unsigned)e, ap.inv_l), i = e - c * L;
    if (row0 + c < nrows) grid[rdst[c] + i] = buf[i * A::NTP + c];
  }
}

template <int TPB, int NT, int KIND, int MODE>
__global__ __launch_bounds__(TPB) void any_col_kernel(float2* __restrict__ grid, Geo3 p, AnyPlan ap, int axis,
                                                      long long inner, unsigned nblk, const float2* __restrict__ tab,
                                                      const float2* __restrict__ kern) {
  using A = Any<TPB, NT>;
  extern __shared__ float2 buf[];
  float2* tw = buf + ap.M * A::NTP;
  const int tid = threadIdx.x, L = ap.L;
  const unsigned o = blockIdx.x / nblk;
  const long long col0 = (long long)(blockIdx.x - o * nblk) * NT;
  long long base;
  if (axis == 0) {
    base = (long long)o * L * inner;
  } else {  // axis 1: o = q * N0 + n0
    const unsigned q = o / (unsigned)p.N[0];
    const int n0 = (int)(o - q * p.N[0]);
    base = ((long long)q * p.G[0] + grid_of(n0, p.G[0], p.c[0])) * (long long)L * inner;
  }
  const int Na = p.N[axis], ca = p.c[axis];
  const unsigned row = (unsigned)inner * 8u;
  const Slab g(grid + base, L * row);
  // a thread's column is the same at every step (TPB % NT == 0)
  const int c = tid % NT;
  const unsigned off = col0 + c < inner ? (unsigned)(col0 + c) * 8u : kNone;
  const int j0 = tid / NT;
  constexpr int JS = TPB / NT;
  for (int j = j0; j < L; j += 4 * JS) {
    float2 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = j + u * JS;
      const bool in = i < L && (MODE == kAdj || pix_of(i, Na, L, ca) >= 0) && off != kNone;
      v[u] = g.load(in ? off + i * row : kNone, 0);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (j + u * JS < L) buf[(j + u * JS) * A::NTP + c] = MODE == kAdj ? conjf2(v[u]) : v[u];
  }
  for (int m = tid; m < ap.M; m += TPB) tw[m] = tab[m];
  __syncthreads();
  A::template transform<KIND>(buf, tw, tab, ap);
  if constexpr (MODE == kToep) {
    const Slab ks(kern, L * row);
    for (int j = j0; j < L; j += 4 * JS) {
      float2 v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int i = j + u * JS;
        v[u] = ks.load(i < L && off != kNone ? off + i * row : kNone, 0);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (j + u * JS < L) {
          float2& y = buf[(j + u * JS) * A::NTP + c];
          y = conjf2(cmul(y, v[u]));
        }
    }
    __syncthreads();
    A::template transform<KIND>(buf, tw, tab, ap);
  }
  for (int j = j0; j < L; j += JS) {
    const float2 y = buf[j * A::NTP + c];
    const bool in = (MODE == kFwd || pix_of(j, Na, L, ca) >= 0) && off != kNone;
    g.store(in ? off + j * row : kNone, 0, MODE == kFwd ? y : conjf2(y));
  }
}

// NT / 2^lcb image rows per block, 2^lcb coils of each at a time; more than one chunk of
// coils only where 2^lcb == NT (one row), whose pixels' sums stay in registers.
template <int TPB, int NT, int KIND>
__global__ __launch_bounds__(TPB) void any_crop_row_kernel(const float2* __restrict__ grid, Geo3 p, AnyPlan ap,
                                                           long long nrows, int ns, const float2* __restrict__ smaps,
                                                           long long s_stride, int lcb, int conj_maps, int accumulate,
                                                           float2* __restrict__ out, long long x_stride,
                                                           const float2* __restrict__ tab) {
  using A = Any<TPB, NT>;
  extern __shared__ float2 buf[];
  float2* tw = buf + ap.M * A::NTP;
  __shared__ long long rgrid[NT], rpix[NT], rout[NT];
  __shared__ float rapo[NT];
  constexpr int KM = (kAnyMax + TPB - 1) / TPB;
  const int tid = threadIdx.x, L = ap.L;
  const int N0 = p.N[0], N1 = p.N[1], N2 = p.N[2];
  const int cb = 1 << lcb, rb = NT >> lcb;
  const long long row0 = (long long)blockIdx.x * rb;
  const long long gsz = (long long)p.G[0] * p.G[1] * L;
  if (tid < rb) {
    const unsigned row = (unsigned)min(row0 + tid, nrows - 1);
    const unsigned r2 = row / (unsigned)N1, n1 = row - r2 * N1;
    const unsigned bx = r2 / (unsigned)N0, n0 = r2 - bx * N0;
    const long long pix = ((long long)n0 * N1 + n1) * N2;
    rgrid[tid] = (long long)bx * ns * gsz + ((long long)grid_of(n0, p.G[0], p.c[0]) * p.G[1] + grid_of(n1, p.G[1], p.c[1])) * L;
    rpix[tid] = pix;
    rout[tid] = bx * x_stride + pix;
    rapo[tid] = p.scale * apod_at(p, 0, n0) * apod_at(p, 1, n1);
  }
  for (int m = tid; m < ap.M; m += TPB) tw[m] = tab[m];
  __syncthreads();
  const int n = NT * L;
  auto put = [&](int r, int n2, float2 s) {
    if (row0 + r >= nrows) return;
    const float a = rapo[r] * apod_at(p, 2, n2);
    float2 y = make_float2(s.x * a, s.y * a);
    float2* o = out + rout[r] + n2;
    if (accumulate) {
      y.x += o->x;
      y.y += o->y;
    }
    *o = y;
  };
  // sum over the chunk's coils [q0, q0 + nr) of pixel n2 of row r
  auto coils = [&](int r, int n2, int q0, int nr) {
    const int at = grid_of(n2, L, p.c[2]) * A::NTP + r * cb;
    const float2* s = smaps ? smaps + q0 * s_stride + rpix[r] + n2 : nullptr;
    float2 acc = make_float2(0.f, 0.f);
    for (int b = 0; b < nr; b += 4) {
      float2 sv[4];
      if (smaps) {
#pragma unroll
        for (int u = 0; u < 4; ++u) sv[u] = s[min(b + u, nr - 1) * s_stride];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        float2 y = conjf2(buf[at + min(b + u, nr - 1)]);
        if (smaps) y = conj_maps ? cmul(y, conjf2(sv[u])) : cmul(y, sv[u]);
        acc.x = b + u < nr ? acc.x + y.x : acc.x;
        acc.y = b + u < nr ? acc.y + y.y : acc.y;
      }
    }
    return acc;
  };
  float2 acc[KM];
#pragma unroll
  for (int m = 0; m < KM; ++m) acc[m] = make_float2(0.f, 0.f);
  for (int q0 = 0; q0 < ns; q0 += cb) {
    const int nr = min(cb, ns - q0);
    for (int e0 = tid; e0 < n; e0 += 4 * TPB) {
      float2 v[4];
      int at[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int e = min(e0 + u * TPB, n - 1);
        const int c = (int)__umulhi((unsigned)e, ap.inv_l), i = e - c * L;
        at[u] = i * A::NTP + c;
        v[u] = grid[rgrid[c >> lcb] + (q0 + min(c & (cb - 1), nr - 1)) * gsz + i];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (e0 + u * TPB < n) buf[at[u]] = conjf2(v[u]);
    }
    __syncthreads();
    A::template transform<KIND>(buf, tw, tab, ap);
    if (cb < NT) {
      const int np = rb * N2;
      for (int e = tid; e < np; e += TPB) {
        const int r = e / N2, n2 = e - r * N2;
        put(r, n2, coils(r, n2, q0, nr));
      }
    } else {
#pragma unroll
      for (int m = 0; m < KM; ++m) {
        const int n2 = tid + m * TPB;
        if (n2 < N2) {
          const float2 y = coils(0, n2, q0, nr);
          acc[m].x += y.x;
          acc[m].y += y.y;
        }
      }
    }
    __syncthreads();
  }
  if (cb == NT) {
#pragma unroll
    for (int m = 0; m < KM; ++m) {
      const int n2 = tid + m * TPB;
      if (n2 < N2) put(0, n2, acc[m]);
    }
  }
}

int fill_geo(Geo3& p, int ndim, const int* N, const int* G, const int* center, const float* apod, float scale) {
  if (ndim < 1 || ndim > 3) MRA_FAIL("fused fft: ndim must be 1..3");
  const int lead = 3 - ndim;
  int off = 0;
  for (int d = 0; d < 3; ++d) {
    if (d < lead) {
      p.N[d] = 1;
      p.G[d] = 1;
      p.c[d] = 0;
      p.apod[d] = nullptr;
    } else {
      const int n = N[d - lead], g = G[d - lead];
      if (n <= 0 || g < n) MRA_FAIL("fused fft: need 0 < N <= G in every dim");
      const int c = center ? center[d - lead] : n / 2;
      if (c < 0 || c > n) MRA_FAIL("fused fft: centre index out of range");
      p.N[d] = n;
      p.G[d] = g;
      p.c[d] = c;
      p.apod[d] = apod ? apod + off : nullptr;
      off += n;
    }
  }
  p.scale = scale;
  return 0;
}

// inner extent of the column pass along axis a (of the 3-dim view)
long long inner_of(const Geo3& p, int a) {
  long long in = 1;
  for (int d = a + 1; d < 3; ++d) in *= p.G[d];
  return in;
}

// Whether axis a runs on its compiled plan: the length has one and the axis is the last or
// has columns for the tile.
bool compiled(const Geo3& p, int a) { return plan_supported(p.G[a]) && (a == 2 || inner_of(p, a) >= 64); }

// Kernels with more than 64 KB of LDS have to say so once.
template <class K>
int allow_lds(K kernel, size_t bytes) {
  if (bytes <= 64 * 1024) return 0;
  if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess) {
    (void)hipGetLastError();
    MRA_FAIL("fused fft: LDS size refused");
  }
  return 0;
}

template <int MODE>
int launch_col_any(int a, float2* grid, const Geo3& p, long long Q, const float2* tab, const float2* kern,
                   hipStream_t st) {
  const AnyPlan* ap = any_plan(p.G[a]);
  if (!ap) MRA_FAIL("fused fft: length outside 2..640");
  const long long inner = inner_of(p, a);
  if (inner > kMaxInner) MRA_FAIL("fused fft: inner extent too large");
  const long long outer = a == 0 ? Q : Q * p.N[0];
  return with_any(*ap, [&](auto TPB, auto NT, auto BL) {
    constexpr int tpb = decltype(TPB)::value, nt = decltype(NT)::value;
    const size_t lds = any_shape(*ap).lds;
    const long long nblk = (inner + nt - 1) / nt;
    if (outer * nblk > 0x7fffffffLL) MRA_FAIL("fused fft: grid too large");
    auto k = any_col_kernel<tpb, nt, decltype(BL)::value, MODE>;
    if (allow_lds(k, lds)) return 1;
    k<<<(unsigned)(outer * nblk), tpb, lds, st>>>(grid, p, *ap, a, inner, (unsigned)nblk, tab, kern);
    return 0;
  });
}

template <int MODE>
int launch_col(int a, float2* grid, const Geo3& p, long long Q, const float2* tw, const float2* kern, hipStream_t st) {
  const long long inner = inner_of(p, a);
  const long long outer = a == 0 ? Q : Q * p.N[0];
  if (!compiled(p, a)) return launch_col_any<MODE>(a, grid, p, Q, tw, kern, st);
  const int rc = with_length(p.G[a], [&](auto LL) {
    constexpr int L = decltype(LL)::value;
    using P = Plan<L>;
    if (inner < P::NC) MRA_FAIL("fused fft: inner extent below the column tile");
    if (inner > kMaxInner) MRA_FAIL("fused fft: inner extent too large");
    const long long nblk = (inner + P::NC - 1) / P::NC;
    if (outer * nblk > 0x7fffffffLL) MRA_FAIL("fused fft: grid too large");
    col_kernel<L, MODE><<<(unsigned)(outer * nblk), P::T * P::NC, 0, st>>>(grid, p, a, inner, (unsigned)nblk, tw, kern);
    return 0;
  });
  if (rc < 0) MRA_FAIL("fused fft: length without an LDS plan");
  return rc;
}

int launch_pad_rows(const float2* x, long long x_stride, const float2* smaps, long long s_stride, long long ns,
                    const int* img_index, const Geo3& p, long long Q, float2* grid, const float2* tw, hipStream_t st) {
  const long long nrows = Q * p.N[0] * p.N[1];
  if (nrows > 0x7fffffffLL) MRA_FAIL("fused fft: grid too large");
  if (!compiled(p, 2)) {
    const AnyPlan* ap = any_plan(p.G[2]);
    if (!ap || img_index) MRA_FAIL("fused fft: length without an LDS plan");
    return with_any(*ap, [&](auto TPB, auto NT, auto BL) {
      constexpr int tpb = decltype(TPB)::value, nt = decltype(NT)::value;
      const size_t lds = any_shape(*ap).lds;
      auto k = any_pad_row_kernel<tpb, nt, decltype(BL)::value>;
      if (allow_lds(k, lds)) return 1;
      k<<<(unsigned)((nrows + nt - 1) / nt), tpb, lds, st>>>(x, x_stride, smaps, s_stride, ns, p, *ap, nrows, grid, tw);
      return 0;
    });
  }
  const int rc = with_length(p.G[2], [&](auto LL) {
    constexpr int L = decltype(LL)::value;
    using P = Plan<L>;
    const long long nb = (nrows + P::NR - 1) / P::NR;
    pad_row_kernel<L><<<(unsigned)nb, P::T * P::NR, 0, st>>>(x, x_stride, smaps, s_stride, ns, img_index, p, nrows,
                                                             grid, tw);
    return 0;
  });
  if (rc < 0) MRA_FAIL("fused fft: length without an LDS plan");
  return rc;
}

int launch_crop_rows(const float2* grid, const Geo3& p, long long nq, long long nx, long long ns,
                     const float2* smaps, long long s_stride, const int* coil_off, int conj_maps, int accumulate,
                     float2* out, long long x_stride, const float2* tw, hipStream_t st) {
  const long long nrows = nx * p.N[0] * p.N[1];
  if (nrows > 0x7fffffffLL) MRA_FAIL("fused fft: image too large");
  if (!compiled(p, 2)) {
    const AnyPlan* ap = any_plan(p.G[2]);
    if (!ap || coil_off) MRA_FAIL("fused fft: length without an LDS plan");
    if (ns > 0x7fffffffLL) MRA_FAIL("fused fft: too many maps");
    return with_any(*ap, [&](auto TPB, auto NT, auto BL) {
      constexpr int tpb = decltype(TPB)::value, nt = decltype(NT)::value;
      int lcb = 0;
      while ((2 << lcb) <= nt && (1 << lcb) < ns) ++lcb;
      const size_t lds = any_shape(*ap).lds;
      const long long rb = nt >> lcb, nb = (nrows + rb - 1) / rb;
      auto k = any_crop_row_kernel<tpb, nt, decltype(BL)::value>;
      if (allow_lds(k, lds)) return 1;
      k<<<(unsigned)nb, tpb, lds, st>>>(grid, p, *ap, nrows, (int)ns, smaps, s_stride, lcb, conj_maps, accumulate, out,
                                        x_stride, tw);
      return 0;
    });
  }
  const int rc = with_length(p.G[2], [&](auto LL) {
    constexpr int L = decltype(LL)::value;
    using P = Plan<L>;
    // coils of a row at a time: the (mean) coil count rounded up to a power of two, as far
    // as the block has rows; the rest of the block takes further image rows
    const long long mean = coil_off ? (nq + nx - 1) / nx : ns;
    auto run = [&](auto LC) {
      constexpr int LCB = decltype(LC)::value;
      if constexpr ((1 << LCB) <= P::NA) {
        constexpr int CB = 1 << LCB, RB = P::NA / CB;
        // threads to a pixel: as many as the row has pixels for (one pixel a thread), else one
        const int ng = max(1, min(CB, P::T * CB / p.N[2]));
        const long long nb = (nrows + RB - 1) / RB;
        crop_row_kernel<L, LCB><<<(unsigned)nb, P::T * P::NA, 0, st>>>(grid, p, nrows, ns, smaps, s_stride, coil_off,
                                                                       ng, conj_maps, accumulate, out, x_stride, tw);
      }
    };
    int lcb = 0;
    while ((2 << lcb) <= P::NA && lcb < 4 && (1 << lcb) < mean) ++lcb;
    switch (lcb) {
      case 0: run(std::integral_constant<int, 0>{}); break;
      case 1: run(std::integral_constant<int, 1>{}); break;
      case 2: run(std::integral_constant<int, 2>{}); break;
      case 3: run(std::integral_constant<int, 3>{}); break;
      default: run(std::integral_constant<int, 4>{}); break;
    }
    return 0;
  });
  if (rc < 0) MRA_FAIL("fused fft: length without an LDS plan");
  return rc;
}

}  // namespace fused
}  // namespace mra

using namespace mra;
using namespace mra::fused;

extern "C" {

// 1 when the fused transforms support grids of shape G (ndim dims): every length has a
// compiled radix plan and every axis but the last has >= 64 points after it.
int mra_fft_fused_supported(int ndim, const int* G) {
  if (ndim < 1 || ndim > 3) return 0;
  long long inner = 1;
  for (int d = ndim - 1; d >= 0; --d) {
    if (!fft::plan_supported(G[d])) return 0;
    if (d < ndim - 1 && inner < 64) return 0;
    inner *= G[d];
  }
  return 1;
}

// 1 when the *_any entry points support grids of shape G: every length in 2..640.
int mra_fft_any_supported(int ndim, const int* G) {
  if (ndim < 1 || ndim > 3) return 0;
  for (int d = 0; d < ndim; ++d)
    if (!fft::any_plan(G[d])) return 0;
  return 1;
}

// How the *_any entry points run length L: shape = {M (the length transformed: L, or the chirp-z
// form's convolution), threads of a block, transforms of a block, kind (0 direct, 1 chirp-z,
// 2 direct with radix 17 or 19), dynamic LDS bytes, passes, radix of each pass}, 16 ints.
int mra_fft_any_shape(int L, int* shape) {
  MRA_TRY_BEGIN
  const fft::AnyPlan* p = fft::any_plan(L);
  if (!p) MRA_FAIL("fft: length outside 2..640");
  const fft::AnyShape s = fft::any_shape(*p);
  const int head[] = {p->M, s.tpb, s.nt, fft::any_kind(*p), (int)s.lds, p->npass};
  for (int i = 0; i < 16; ++i) shape[i] = i < 6 ? head[i] : i - 6 < p->npass ? p->radix[i - 6] : 0;
  MRA_TRY_END
}

// Device table of length L for the *_any entry points: complex values, and their contents
// (host memory). For lengths with a compiled plan the first L values are mra_fft_lds_twiddles'.
long long mra_fft_any_table_len(int L) {
  const fft::AnyPlan* p = fft::any_plan(L);
  return p ? fft::any_table_len(*p) : 0;
}

int mra_fft_any_table(int L, float* host) {
  MRA_TRY_BEGIN
  const fft::AnyPlan* p = fft::any_plan(L);
  if (!p) MRA_FAIL("fft: length outside 2..640");
  try {
    fft::any_table(*p, host);
  } catch (...) {
    MRA_FAIL("fft: out of memory for a table");
  }
  MRA_TRY_END
}

}  // extern "C"

namespace {

// Forward: grid[q] = FFT(pad(x[img(q)] * S[map(q)] * apod * scale)), q < nq, with
// img(q) = img_index[q] or q / ns, map(q) = q or q % ns. tw[d] as for mra_fft_lds.
int pad_forward(int ndim, const int* N, const int* G, const int* center, const void* x, long long x_stride,
                        const void* smaps, long long ns, long long s_stride, const int* img_index, long long nq,
                        const float* apod, float scale, void* grid, const void* const* tw, void* stream) {
  MRA_TRY_BEGIN
  if (nq < 1 || ns < 1) MRA_FAIL("fused fft: batch sizes must be positive");
  Geo3 p{};
  if (fill_geo(p, ndim, N, G, center, apod, scale)) return 1;
  const float2* const* t = (const float2* const*)tw;
  const int lead = 3 - ndim;
  hipStream_t st = (hipStream_t)stream;
  if (launch_pad_rows((const float2*)x, x_stride, (const float2*)smaps, s_stride, ns, img_index, p, nq,
                      (float2*)grid, t[ndim - 1], st))
    return 1;
  for (int a = 1; a >= lead; --a)
    if (launch_col<kFwd>(a, (float2*)grid, p, nq, t[a - lead], nullptr, st)) return 1;
  MRA_CHECK_LAUNCH("fft_pad_forward");
  MRA_TRY_END
}

// Adjoint: out[bx] (+)= scale * apod * sum_{q of bx} crop(iFFT(grid[q])) * (conj) S[q],
// grids of image bx = coil_off[bx] .. coil_off[bx+1]-1 or bx*ns .. bx*ns+ns-1; nq grids
// in all. The grids are overwritten.
int crop_adjoint(int ndim, const int* N, const int* G, const int* center, void* grid, long long nq,
                         long long nx, const void* smaps, long long ns, long long s_stride, const int* coil_off,
                         int conj_maps, const float* apod, float scale, int accumulate, void* out,
                         long long x_stride, const void* const* tw, void* stream) {
  MRA_TRY_BEGIN
  if (nq < 1 || nx < 1 || ns < 1) MRA_FAIL("fused fft: batch sizes must be positive");
  Geo3 p{};
  if (fill_geo(p, ndim, N, G, center, apod, scale)) return 1;
  const float2* const* t = (const float2* const*)tw;
  const int lead = 3 - ndim;
  hipStream_t st = (hipStream_t)stream;
  for (int a = lead; a <= 1; ++a)
    if (launch_col<kAdj>(a, (float2*)grid, p, nq, t[a - lead], nullptr, st)) return 1;
  if (launch_crop_rows((const float2*)grid, p, nq, nx, ns, (const float2*)smaps, s_stride, coil_off, conj_maps, accumulate,
                       (float2*)out, x_stride, t[ndim - 1], st))
    return 1;
  MRA_CHECK_LAUNCH("fft_crop_adjoint");
  MRA_TRY_END
}

// Toeplitz normal operator of one image x and ns maps (2D / 3D):
// out (+)= sum_q conj(S[q]) crop(iFFT(K * FFT(pad(x * S[q])))), K the PSF spectrum in
// the unshifted layout on grid G (normalisation folded in). work holds ns grids.
int toeplitz(int ndim, const int* N, const int* G, const int* center, const void* x, const void* smaps,
                       long long ns, long long s_stride, const void* kern, void* work, int accumulate, void* out,
                       const void* const* tw, void* stream) {
  MRA_TRY_BEGIN
  if (ns < 1) MRA_FAIL("fused fft: batch sizes must be positive");
  Geo3 p{};
  if (fill_geo(p, ndim, N, G, center, nullptr, 1.0f)) return 1;
  const float2* const* t = (const float2* const*)tw;
  const int lead = 3 - ndim;
  hipStream_t st = (hipStream_t)stream;
  float2* g = (float2*)work;
  if (launch_pad_rows((const float2*)x, 0, (const float2*)smaps, s_stride, ns, nullptr, p, ns, g, t[ndim - 1], st))
    return 1;
  // forward along axis 1 (3D), then axis 0 forward * K inverse, then inverse along axis 1 (3D)
  if (ndim == 3 && launch_col<kFwd>(1, g, p, ns, t[1], nullptr, st)) return 1;
  if (launch_col<kToep>(lead, g, p, ns, t[0], (const float2*)kern, st)) return 1;
  if (ndim == 3 && launch_col<kAdj>(1, g, p, ns, t[1], nullptr, st)) return 1;
  if (launch_crop_rows(g, p, ns, 1, ns, (const float2*)smaps, s_stride, nullptr, 1, accumulate, (float2*)out, 0,
                       t[ndim - 1], st))
    return 1;
  MRA_CHECK_LAUNCH("toeplitz_fused");
  MRA_TRY_END
}

}  // namespace

extern "C" {

// The compiled grids only (mra_fft_fused_supported), tw[d] as for mra_fft_lds.
int mra_fft_pad_forward(int ndim, const int* N, const int* G, const int* center, const void* x, long long x_stride,
                        const void* smaps, long long ns, long long s_stride, const int* img_index, long long nq,
                        const float* apod, float scale, void* grid, const void* const* tw, void* stream) {
  if (!mra_fft_fused_supported(ndim, G)) MRA_FAIL("fused fft: grid shape not supported");
  return pad_forward(ndim, N, G, center, x, x_stride, smaps, ns, s_stride, img_index, nq, apod, scale, grid, tw, stream);
}

int mra_fft_crop_adjoint(int ndim, const int* N, const int* G, const int* center, void* grid, long long nq,
                         long long nx, const void* smaps, long long ns, long long s_stride, const int* coil_off,
                         int conj_maps, const float* apod, float scale, int accumulate, void* out,
                         long long x_stride, const void* const* tw, void* stream) {
  if (!mra_fft_fused_supported(ndim, G)) MRA_FAIL("fused fft: grid shape not supported");
  return crop_adjoint(ndim, N, G, center, grid, nq, nx, smaps, ns, s_stride, coil_off, conj_maps, apod, scale,
                      accumulate, out, x_stride, tw, stream);
}

int mra_toeplitz_fused(int ndim, const int* N, const int* G, const int* center, const void* x, const void* smaps,
                       long long ns, long long s_stride, const void* kern, void* work, int accumulate, void* out,
                       const void* const* tw, void* stream) {
  if (ndim < 2) MRA_FAIL("fused Toeplitz: 2D or 3D only");
  if (!mra_fft_fused_supported(ndim, G)) MRA_FAIL("fused fft: grid shape not supported");
  return toeplitz(ndim, N, G, center, x, smaps, ns, s_stride, kern, work, accumulate, out, tw, stream);
}

// Any grid with lengths 2..640 (mra_fft_any_supported), tw[d] = device copy of
// mra_fft_any_table(G[d]). One image batch with the same maps (no per-problem indexing).
int mra_fft_pad_forward_any(int ndim, const int* N, const int* G, const int* center, const void* x, long long x_stride,
                            const void* smaps, long long ns, long long s_stride, long long nq, const float* apod,
                            float scale, void* grid, const void* const* tw, void* stream) {
  if (!mra_fft_any_supported(ndim, G)) MRA_FAIL("fused fft: grid shape not supported");
  return pad_forward(ndim, N, G, center, x, x_stride, smaps, ns, s_stride, nullptr, nq, apod, scale, grid, tw, stream);
}

int mra_fft_crop_adjoint_any(int ndim, const int* N, const int* G, const int* center, void* grid, long long nx,
                             const void* smaps, long long ns, long long s_stride, int conj_maps, const float* apod,
                             float scale, int accumulate, void* out, long long x_stride, const void* const* tw,
                             void* stream) {
  if (!mra_fft_any_supported(ndim, G)) MRA_FAIL("fused fft: grid shape not supported");
  return crop_adjoint(ndim, N, G, center, grid, nx * ns, nx, smaps, ns, s_stride, nullptr, conj_maps, apod, scale,
                      accumulate, out, x_stride, tw, stream);
}

int mra_toeplitz_any(int ndim, const int* N, const int* G, const int* center, const void* x, const void* smaps,
                     long long ns, long long s_stride, const void* kern, void* work, int accumulate, void* out,
                     const void* const* tw, void* stream) {
  if (ndim < 2) MRA_FAIL("fused Toeplitz: 2D or 3D only");
  if (!mra_fft_any_supported(ndim, G)) MRA_FAIL("fused fft: grid shape not supported");
  return toeplitz(ndim, N, G, center, x, smaps, ns, s_stride, kern, work, accumulate, out, tw, stream);
}

}  // extern "C"
