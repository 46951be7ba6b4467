// FFTs of run-time length (2..640) in LDS, fused with the pad / crop like the compiled ones in
// fft_fused.hip: a grid is ceil(oversampling * image) long, so most lengths have no compiled
// plan, and a general library transform takes separate pad, transpose and crop passes (11
// kernels for a 3D grid with a prime edge: 0.82 ms of the 1.9 ms normal operator at 90x104x77,
// 7 coils, width 6; 0.50 ms here. 230x187, 11 coils: 86 and 49 us).
//
// NT transforms of a block sit in LDS as [point][transform]. Lengths whose prime factors are
// at most 19 take Stockham passes of radix 2..19 (fewest passes, then smallest radices), in
// place: a pass reads its inputs into registers, synchronises and writes. Other lengths go
// through Bluestein's chirp-z form (L. Bluestein, "A linear filtering approach to the
// computation of discrete Fourier transform", IEEE Trans. Audio Electroacoust. 18, 1970) as a
// circular convolution of a length M >= 2 L - 1 without larger factors: two transforms of M.
#pragma once
#include <cmath>
#include <mutex>
#include <vector>

#include "capi_util.h"
#include "fft_lds.h"

namespace mra {
namespace fft {

constexpr int kAnyMax = 640;     // longest length (M <= 1280)
constexpr int kMaxPass = 10;

struct AnyPlan {
  int L, M;                      // M == L: direct
  int npass;
  int radix[kMaxPass], ns[kMaxPass];
  unsigned inv_ns[kMaxPass];     // j / ns == umulhi(j, inv_ns) for j < 2^16, ns > 1
  unsigned inv_l;                // e / L likewise
};

// Butterflies of radix R a thread may hold through a pass: 8..16 points (a plan whose passes
// held 16..26 took 256 VGPRs).
constexpr int held(int R) { return R >= 9 ? 1 : R >= 5 ? 2 : 4; }

// Launch shape of a length: 16 transforms (8 above M = 640, for LDS) in the fewest threads that
// hold every pass's butterflies.
struct AnyShape {
  int nt, tpb;
  size_t lds;
};
inline AnyShape any_shape(int M, const int* radix, int npass) {
  for (int nt = M <= 640 ? 16 : 8; nt >= 8; nt -= 8) {
    int need = 0;
    for (int i = 0; i < npass; ++i) {
      const int h = held(radix[i]), b = (M / radix[i] * nt + h - 1) / h;
      need = b > need ? b : need;
    }
    if (need > 1024) continue;
    return AnyShape{nt, nt == 8 || need > 512 ? 1024 : need <= 256 ? 256 : 512, sizeof(float2) * ((size_t)M * (nt + 1) + M)};
  }
  return AnyShape{0, 0, 0};
}
inline AnyShape any_shape(const AnyPlan& p) { return any_shape(p.M, p.radix, p.npass); }

inline unsigned magic(unsigned d) { return (unsigned)(0x100000000ull / d) + 1; }

// Fewest passes, then smallest radix sum, over the radices the kernels have.
inline bool best_radices(int n, const int* set, int nset, std::vector<int>& cur, std::vector<int>& best) {
  if (n == 1) {
    auto sum = [](const std::vector<int>& v) { int s = 0; for (int x : v) s += x; return s; };
    if (best.empty() || cur.size() < best.size() || (cur.size() == best.size() && sum(cur) < sum(best))) best = cur;
    return true;
  }
  bool any = false;
  if (!best.empty() && cur.size() + 1 > best.size()) return false;
  for (int i = 0; i < nset; ++i)
    if (n % set[i] == 0 && (cur.empty() || set[i] <= cur.back())) {
      cur.push_back(set[i]);
      any = best_radices(n / set[i], set, nset, cur, best) || any;
      cur.pop_back();
    }
  return any;
}

inline bool make_any_plan(int L, AnyPlan& p) {
  static const int all[] = {19, 17, 16, 15, 13, 12, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2};
  p = AnyPlan{};
  if (L < 2 || L > kAnyMax) return false;
  p.L = p.M = L;
  std::vector<int> cur, best;
  if (!best_radices(L, all, 16, cur, best)) {
    // convolution length: least (M times passes) among the smooth ones from 2 L - 1 up
    double cost = 1e30;
    for (int M = 2 * L - 1; M <= 2 * kAnyMax && M < 3 * L; ++M) {
      std::vector<int> c2, b2;
      if (!best_radices(M, all + 2, 14, c2, b2) || !any_shape(M, b2.data(), (int)b2.size()).tpb) continue;
      const double k = (double)M * (b2.size() + 1);
      if (k < cost) {
        cost = k;
        best = b2;
        p.M = M;
      }
    }
    if (best.empty()) return false;
  }
  p.npass = (int)best.size();
  int ns = 1;
  for (int i = 0; i < p.npass; ++i) {
    p.radix[i] = best[i];
    p.ns[i] = ns;
    p.inv_ns[i] = magic(ns);
    ns *= best[i];
  }
  p.inv_l = magic(L);
  return true;
}

// Device table of a length: exp(-2 pi i m / M) (M values), then for M > L the chirp
// exp(-pi i n^2 / L) (L values) and the transform of its conjugate over M, divided by M.
inline long long any_table_len(const AnyPlan& p) { return p.M == p.L ? p.M : 2LL * p.M + p.L; }

inline void any_table(const AnyPlan& p, float* t) {
  const double pi = 3.14159265358979323846;
  std::vector<double> wr(p.M), wi(p.M);
  for (int m = 0; m < p.M; ++m) {
    wr[m] = cos(-2.0 * pi * m / p.M);
    wi[m] = sin(-2.0 * pi * m / p.M);
    t[2 * m] = (float)wr[m];
    t[2 * m + 1] = (float)wi[m];
  }
  if (p.M == p.L) return;
  float* chirp = t + 2 * p.M;
  float* conv = chirp + 2 * p.L;
  std::vector<double> br(p.M, 0.0), bi(p.M, 0.0);
  for (int n = 0; n < p.L; ++n) {
    const double a = pi * ((long long)n * n % (2 * p.L)) / p.L;
    chirp[2 * n] = (float)cos(a);
    chirp[2 * n + 1] = (float)-sin(a);
    br[n] = cos(a);
    bi[n] = sin(a);
    if (n > 0) {
      br[p.M - n] = br[n];
      bi[p.M - n] = bi[n];
    }
  }
  for (int k = 0; k < p.M; ++k) {
    double sr = 0.0, si = 0.0;
    for (int n = 0, m = 0; n < p.M; ++n, m = m + k >= p.M ? m + k - p.M : m + k) {
      sr += br[n] * wr[m] - bi[n] * wi[m];
      si += br[n] * wi[m] + bi[n] * wr[m];
    }
    conv[2 * k] = (float)(sr / p.M);
    conv[2 * k + 1] = (float)(si / p.M);
  }
}

inline const AnyPlan* any_plan(int L) {
  static AnyPlan plans[kAnyMax + 1];
  static std::once_flag once;
  try {
    std::call_once(once, [] {
      for (int n = 2; n <= kAnyMax; ++n)
        if (!make_any_plan(n, plans[n]) || !any_shape(plans[n]).tpb) plans[n].L = 0;
    });
  } catch (...) {
    return nullptr;
  }
  return L >= 2 && L <= kAnyMax && plans[L].L ? &plans[L] : nullptr;
}

// What a kernel is compiled for: direct passes up to radix 16, the chirp-z form over them, and
// direct passes with radix 17 or 19 (whose registers halve the blocks of a CU at 1024 threads).
enum AnyKind { kDirect = 0, kChirp = 1, kPrime = 2 };
inline AnyKind any_kind(const AnyPlan& p) {
  if (p.M != p.L) return kChirp;
  for (int i = 0; i < p.npass; ++i)
    if (p.radix[i] > 16) return kPrime;
  return kDirect;
}

template <int TPB, int NT>
struct Any {
  static constexpr int NTP = NT + 1;

  template <int R>
  static __device__ __forceinline__ void pass(float2* buf, const float2* tw, int tid, int M, int ns, unsigned inv) {
    constexpr int MB = held(R);
    const int nb = M / R, total = nb * NT, step = nb / ns;  // M / (ns R)
    float2 v[MB][R];
    int to[MB];
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      const int b = tid + m * TPB;
      if (b < total) {
        const int c = b % NT, j = b / NT;
        const int h = ns > 1 ? (int)__umulhi((unsigned)j, inv) : j, k = j - h * ns;
        to[m] = (h * ns * R + k) * NTP + c;
        const int kt = k * step;
#pragma unroll
        for (int q = 0; q < R; ++q) {
          const float2 x = buf[(j + q * nb) * NTP + c];
          v[m][q] = q == 0 ? x : cmul(x, tw[kt * q]);
        }
        dft<R>(v[m]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < MB; ++m)
      if (tid + m * TPB < total) {
#pragma unroll
        for (int q = 0; q < R; ++q) buf[to[m] + q * ns * NTP] = v[m][q];
      }
    __syncthreads();
  }

  // Forward transform of length M of the NT columns, tw = its M roots in LDS.
  template <bool PRIME>
  static __device__ __forceinline__ void smooth(float2* buf, const float2* tw, const AnyPlan& p) {
    for (int i = 0; i < p.npass; ++i) {
      const int ns = p.ns[i];
      const unsigned inv = p.inv_ns[i];
      // opaque per pass: hoisted out of the loop, every radix's addresses took 210 VGPRs
      int tid = threadIdx.x;
      const int M = p.M;
      asm volatile("" : "+v"(tid));
      switch (p.radix[i]) {
#define MRA_ANY_RADIX(R) \
  case R: pass<R>(buf, tw, tid, M, ns, inv); break;
        MRA_ANY_RADIX(2) MRA_ANY_RADIX(3) MRA_ANY_RADIX(4) MRA_ANY_RADIX(5) MRA_ANY_RADIX(6) MRA_ANY_RADIX(7)
        MRA_ANY_RADIX(8) MRA_ANY_RADIX(9) MRA_ANY_RADIX(10) MRA_ANY_RADIX(11) MRA_ANY_RADIX(12) MRA_ANY_RADIX(13)
        MRA_ANY_RADIX(15) MRA_ANY_RADIX(16)
#undef MRA_ANY_RADIX
        case 17: if constexpr (PRIME) pass<17>(buf, tw, tid, M, ns, inv); break;
        case 19: if constexpr (PRIME) pass<19>(buf, tw, tid, M, ns, inv); break;
      }
    }
  }

  // Forward transform of length L of the NT columns of buf (points 0 .. L - 1), in place.
  // tab: the length's device table. The caller has synchronised after writing buf and tw.
  template <int KIND>
  static __device__ __forceinline__ void transform(float2* buf, const float2* tw, const float2* __restrict__ tab,
                                                   const AnyPlan& p) {
    if constexpr (KIND != kChirp) {
      smooth<KIND == kPrime>(buf, tw, p);
    } else {
      const float2 *chirp = tab + p.M, *conv = chirp + p.L;
      for (int e = threadIdx.x; e < NT * p.M; e += TPB) {
        const int j = e / NT, at = j * NTP + e % NT;
        buf[at] = j < p.L ? cmul(buf[at], chirp[j]) : make_float2(0.f, 0.f);
      }
      __syncthreads();
      smooth<false>(buf, tw, p);
      for (int e = threadIdx.x; e < NT * p.M; e += TPB) {
        const int j = e / NT, at = j * NTP + e % NT;
        const float2 y = cmul(buf[at], conv[j]);
        buf[at] = make_float2(y.x, -y.y);
      }
      __syncthreads();
      smooth<false>(buf, tw, p);
      for (int e = threadIdx.x; e < NT * p.L; e += TPB) {
        const int j = e / NT, at = j * NTP + e % NT;
        const float2 y = buf[at];
        buf[at] = cmul(make_float2(y.x, -y.y), chirp[j]);
      }
      __syncthreads();
    }
  }
};

// f(integral_constant<TPB>, integral_constant<NT>, integral_constant<KIND>) for a plan's shape.
template <class F>
int with_any(const AnyPlan& p, F&& f) {
  using std::integral_constant;
  const AnyShape s = any_shape(p);
  const AnyKind kind = any_kind(p);
  auto go = [&](auto TPB, auto NT) {
    if (kind == kChirp) return f(TPB, NT, integral_constant<int, kChirp>{});
    return kind == kPrime ? f(TPB, NT, integral_constant<int, kPrime>{}) : f(TPB, NT, integral_constant<int, kDirect>{});
  };
  if (s.nt == 8) return go(integral_constant<int, 1024>{}, integral_constant<int, 8>{});
  if (s.tpb == 256) return go(integral_constant<int, 256>{}, integral_constant<int, 16>{});
  if (s.tpb == 512) return go(integral_constant<int, 512>{}, integral_constant<int, 16>{});
  return go(integral_constant<int, 1024>{}, integral_constant<int, 16>{});
}

}  // namespace fft
}  // namespace mra
