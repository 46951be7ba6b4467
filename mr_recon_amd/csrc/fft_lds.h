// Register-and-LDS FFT building blocks shared by the plain per-axis transforms
// (fft_lds.hip) and the fused pad / crop / Toeplitz transforms (fft_fused.hip).
//
// Stockham autosort passes (Govindaraju et al., "High Performance Discrete Fourier
// Transforms on Graphics Processors", SC 2008): for a pass of radix r after
// sub-transform size Ns, butterfly j reads the r values x[j + q L/r], multiplies
// value q by exp(-2 pi i (j mod Ns) q / (Ns r)), takes their r-point DFT and writes
// value q to y[(j / Ns) Ns r + (j mod Ns) + q Ns].
//
// A transform is two passes of radix 8..20 (three of radix 6..10 above 320), T threads per
// transform, one butterfly per thread and pass. The first pass takes its inputs from the
// caller (global memory) into registers and the last hands its outputs over from registers,
// so LDS carries one exchange (two above 320) and one twiddle read per point: 24 bytes a
// point of LDS traffic at L = 160 where passes that start and end in LDS (radix 8, 5, 4)
// took 88, which is what bounded them. The last pass's outputs of a transform are the first
// pass's inputs of one with the radices reversed, so the Toeplitz transform goes from the
// forward to the inverse without leaving the registers.
#pragma once
#include <type_traits>

#include "common.h"

namespace mra {
namespace fft {

// Radices (product == L; R3 = 1: two passes), threads per transform T >= L / min radix, and
// transforms per block: NC along a strided axis (16: loads and stores of 128 contiguous
// bytes; 8 where 16 would need more than 1024 threads), NR along the contiguous axis for
// the forward transform, NA for the adjoint one (whose blocks reduce over coils).
template <int A, int B, int C, int TT, int COL, int ROW, int ADJ> struct Factors {
  static constexpr int R1 = A, R2 = B, R3 = C, T = TT, NC = COL, NR = ROW, NA = ADJ;
};
template <int L> struct Plan;
template <> struct Plan<64> : Factors<8, 8, 1, 8, 16, 32, 32> {};
template <> struct Plan<80> : Factors<8, 10, 1, 10, 16, 16, 16> {};
template <> struct Plan<96> : Factors<8, 12, 1, 12, 16, 16, 16> {};
template <> struct Plan<120> : Factors<10, 12, 1, 12, 16, 16, 16> {};
template <> struct Plan<128> : Factors<8, 16, 1, 16, 16, 16, 16> {};
template <> struct Plan<160> : Factors<16, 10, 1, 16, 16, 16, 16> {};
template <> struct Plan<192> : Factors<16, 12, 1, 16, 16, 16, 16> {};
template <> struct Plan<240> : Factors<16, 15, 1, 16, 16, 16, 16> {};
template <> struct Plan<256> : Factors<16, 16, 1, 16, 16, 16, 16> {};
template <> struct Plan<320> : Factors<16, 20, 1, 20, 16, 16, 16> {};
template <> struct Plan<384> : Factors<8, 8, 6, 64, 16, 4, 16> {};
template <> struct Plan<480> : Factors<8, 10, 6, 80, 8, 4, 8> {};
template <> struct Plan<512> : Factors<8, 8, 8, 64, 16, 4, 16> {};
template <> struct Plan<640> : Factors<8, 8, 10, 80, 8, 4, 8> {};

// A slab of device memory read and written through a buffer descriptor: the address is the
// slab's base (the same in all lanes) + `off` (per lane, bytes) + `d` (the same in all lanes,
// bytes), with no 64-bit arithmetic per lane. Lanes whose off is kNone load zeros and store
// nothing (the hardware's range check), so a predicated run of loads stays straight code with
// all its loads in flight: as branches each load was waited for before the next was issued.
// A slab is under 2 GiB (640^3 points at most), so off + d cannot wrap.
constexpr unsigned kNone = 0x80000000u;
struct Slab {
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ Slab(const float2* base, unsigned bytes)
      : r(__builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)bytes, 0x00020000)) {}
  __device__ __forceinline__ float2 load(unsigned off, unsigned d) const {
    typedef unsigned int u2 __attribute__((ext_vector_type(2)));
    const u2 v = __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, (int)d, 0);
    return make_float2(__uint_as_float(v.x), __uint_as_float(v.y));
  }
  __device__ __forceinline__ void store(unsigned off, unsigned d, float2 x) const {
    typedef unsigned int u2 __attribute__((ext_vector_type(2)));
    u2 v;
    v.x = __float_as_uint(x.x);
    v.y = __float_as_uint(x.y);
    __builtin_amdgcn_raw_buffer_store_b64(v, r, (int)off, (int)d, 0);
  }
};

__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// exp(-2 pi i k / R), k < R, rounded from double at compile time.
template <int R, class F> struct Roots { F re[R] = {}, im[R] = {}; };
template <int R, class F = float>
constexpr Roots<R, F> roots() {
  Roots<R, F> w;
  for (int k = 0; k < R; ++k) {
    // Taylor series about 0 with |x| <= pi (k folded into -R/2 .. R/2)
    const int kk = 2 * k > R ? k - R : k;
    const double x = -2.0 * 3.14159265358979323846 * kk / R;
    double c = 1.0, s = x, tc = 1.0, ts = x;
    for (int i = 1; i < 24; ++i) {
      tc *= -x * x / ((2.0 * i - 1) * (2.0 * i));
      ts *= -x * x / ((2.0 * i) * (2.0 * i + 1));
      c += tc;
      s += ts;
    }
    w.re[k] = (F)c;
    w.im[k] = (F)s;
  }
  return w;
}

// a exp(-2 pi i K / R); multiples of an eighth of a turn without the full product
template <int K, int R>
__device__ __forceinline__ float2 turn(float2 a) {
  constexpr int k = K % R;
  constexpr float h = 0.70710678118654752f;
  if constexpr (k == 0) return a;
  else if constexpr (4 * k == R) return make_float2(a.y, -a.x);
  else if constexpr (2 * k == R) return make_float2(-a.x, -a.y);
  else if constexpr (4 * k == 3 * R) return make_float2(-a.y, a.x);
  else if constexpr (8 * k == R) return make_float2(h * (a.x + a.y), h * (a.y - a.x));
  else if constexpr (8 * k == 3 * R) return make_float2(h * (a.y - a.x), -h * (a.x + a.y));
  else {
    constexpr auto w = roots<R>();
    return cmul(a, make_float2(w.re[k], w.im[k]));
  }
}

// f(integral_constant 0), .., f(integral_constant N - 1)
template <int N, int I = 0, class F>
__device__ __forceinline__ void unroll(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    unroll<N, I + 1>(f);
  }
}

// In-register r-point DFT (forward sign), v[q] -> sum_p v[p] e^{-2 pi i p q / r}.
template <int R>
__device__ __forceinline__ void dft(float2 (&v)[R]) {
  if constexpr (R == 2) {
    const float2 a = v[0], b = v[1];
    v[0] = make_float2(a.x + b.x, a.y + b.y);
    v[1] = make_float2(a.x - b.x, a.y - b.y);
  } else if constexpr (R == 4) {
    const float2 a0 = make_float2(v[0].x + v[2].x, v[0].y + v[2].y);
    const float2 a1 = make_float2(v[0].x - v[2].x, v[0].y - v[2].y);
    const float2 b0 = make_float2(v[1].x + v[3].x, v[1].y + v[3].y);
    const float2 b1 = make_float2(v[1].x - v[3].x, v[1].y - v[3].y);
    // b1 * (-i)
    const float2 b1m = make_float2(b1.y, -b1.x);
    v[0] = make_float2(a0.x + b0.x, a0.y + b0.y);
    v[2] = make_float2(a0.x - b0.x, a0.y - b0.y);
    v[1] = make_float2(a1.x + b1m.x, a1.y + b1m.y);
    v[3] = make_float2(a1.x - b1m.x, a1.y - b1m.y);
  } else if constexpr (R == 8) {
    // radix-2 split: even / odd halves as 4-point DFTs
    float2 e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
    dft<4>(e);
    dft<4>(o);
    unroll<4>([&](auto Q) {
      constexpr int q = decltype(Q)::value;
      const float2 t = turn<q, 8>(o[q]);
      v[q] = make_float2(e[q].x + t.x, e[q].y + t.y);
      v[q + 4] = make_float2(e[q].x - t.x, e[q].y - t.y);
    });
  } else if constexpr (R == 6) {
    // 6 = 2 x 3: two 3-point DFTs of the even / odd samples
    float2 e[3] = {v[0], v[2], v[4]}, o[3] = {v[1], v[3], v[5]};
    dft<3>(e);
    dft<3>(o);
    unroll<3>([&](auto Q) {
      constexpr int q = decltype(Q)::value;
      const float2 t = turn<q, 6>(o[q]);
      v[q] = make_float2(e[q].x + t.x, e[q].y + t.y);
      v[q + 3] = make_float2(e[q].x - t.x, e[q].y - t.y);
    });
  } else if constexpr (R == 3) {
    constexpr float s = 0.86602540378443865f;
    const float2 a = v[0], b = v[1], cc = v[2];
    const float2 t = make_float2(b.x + cc.x, b.y + cc.y);
    const float2 d = make_float2(b.x - cc.x, b.y - cc.y);
    v[0] = make_float2(a.x + t.x, a.y + t.y);
    const float2 m = make_float2(a.x - 0.5f * t.x, a.y - 0.5f * t.y);
    // -i s d
    v[1] = make_float2(m.x + s * d.y, m.y - s * d.x);
    v[2] = make_float2(m.x - s * d.y, m.y + s * d.x);
  } else if constexpr (R == 5) {
    constexpr float c1 = 0.30901699437494742f, c2 = -0.80901699437494742f;
    constexpr float s1 = 0.95105651629515357f, s2 = 0.58778525229247313f;
    const float2 a = v[0];
    const float2 t1 = make_float2(v[1].x + v[4].x, v[1].y + v[4].y);
    const float2 t2 = make_float2(v[2].x + v[3].x, v[2].y + v[3].y);
    const float2 d1 = make_float2(v[1].x - v[4].x, v[1].y - v[4].y);
    const float2 d2 = make_float2(v[2].x - v[3].x, v[2].y - v[3].y);
    v[0] = make_float2(a.x + t1.x + t2.x, a.y + t1.y + t2.y);
    const float2 m1 = make_float2(a.x + c1 * t1.x + c2 * t2.x, a.y + c1 * t1.y + c2 * t2.y);
    const float2 m2 = make_float2(a.x + c2 * t1.x + c1 * t2.x, a.y + c2 * t1.y + c1 * t2.y);
    // n1 = s1 d1 + s2 d2 ; n2 = s2 d1 - s1 d2 ; outputs m -/+ i n
    const float2 n1 = make_float2(s1 * d1.x + s2 * d2.x, s1 * d1.y + s2 * d2.y);
    const float2 n2 = make_float2(s2 * d1.x - s1 * d2.x, s2 * d1.y - s1 * d2.y);
    v[1] = make_float2(m1.x + n1.y, m1.y - n1.x);
    v[4] = make_float2(m1.x - n1.y, m1.y + n1.x);
    v[2] = make_float2(m2.x + n2.y, m2.y - n2.x);
    v[3] = make_float2(m2.x - n2.y, m2.y + n2.x);
  } else if constexpr (R == 7 || R == 11 || R == 13 || R == 17 || R == 19) {
    // odd prime: sums and differences of the pairs (p, R - p); real cosines and sines. From 17
    // the sums of (R - 1) / 2 products run in 64 bits, as fast as in 32 here: in 32 bits they
    // made a transform of 152 x 68 x 176 points 1.4 times as far off as the chirp-z form.
    using F = std::conditional_t<(R >= 17), double, float>;
    constexpr auto w = roots<R, F>();
    constexpr int H = (R - 1) / 2;
    F tx[H], ty[H], dx[H], dy[H];
    const F ax0 = v[0].x, ay0 = v[0].y;
    F sx = ax0, sy = ay0;
#pragma unroll
    for (int p = 0; p < H; ++p) {
      tx[p] = (F)v[p + 1].x + (F)v[R - 1 - p].x;
      ty[p] = (F)v[p + 1].y + (F)v[R - 1 - p].y;
      dx[p] = (F)v[p + 1].x - (F)v[R - 1 - p].x;
      dy[p] = (F)v[p + 1].y - (F)v[R - 1 - p].y;
      sx += tx[p];
      sy += ty[p];
    }
    v[0] = make_float2((float)sx, (float)sy);
#pragma unroll
    for (int q = 1; q <= H; ++q) {
      // two chains each, so that fewer products are rounded into a large sum
      F ax[2] = {0, 0}, ay[2] = {0, 0}, bx[2] = {0, 0}, by[2] = {0, 0};
#pragma unroll
      for (int p = 0; p < H; ++p) {
        const F c = w.re[(p + 1) * q % R], z = w.im[(p + 1) * q % R];  // z = -sin
        ax[p & 1] += c * tx[p];
        ay[p & 1] += c * ty[p];
        bx[p & 1] += z * dx[p];
        by[p & 1] += z * dy[p];
      }
      // a + i b, a - i b
      const F a0 = ax0 + (ax[0] + ax[1]), a1 = ay0 + (ay[0] + ay[1]), b0 = bx[0] + bx[1], b1 = by[0] + by[1];
      v[q] = make_float2((float)(a0 - b1), (float)(a1 + b0));
      v[R - q] = make_float2((float)(a0 + b1), (float)(a1 - b0));
    }
  } else {
    // composite: R = A B, n = B n1 + n2, k = k1 + A k2
    constexpr int A = R == 10 || R == 15 || R == 20 ? 5 : R == 9 ? 3 : 4, B = R / A;
    static_assert(A * B == R, "radix");
    float2 u[B][A];
    unroll<B>([&](auto N2) {
      constexpr int n2 = decltype(N2)::value;
#pragma unroll
      for (int n1 = 0; n1 < A; ++n1) u[n2][n1] = v[B * n1 + n2];
      dft<A>(u[n2]);
      unroll<A>([&](auto K1) {
        constexpr int k1 = decltype(K1)::value;
        u[n2][k1] = turn<n2 * k1, R>(u[n2][k1]);
      });
    });
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
      float2 t[B];
#pragma unroll
      for (int n2 = 0; n2 < B; ++n2) t[n2] = u[n2][k1];
      dft<B>(t);
#pragma unroll
      for (int k2 = 0; k2 < B; ++k2) v[k1 + A * k2] = t[k2];
    }
  }
}

// LDS of one transform batch: NT transforms, [row][transform] (columns) or [transform][row],
// a row skewed by its index over the first radix, so that the first pass's writes (stride
// R1) spread over the banks.
template <int L, int R1, int NT, bool ROW>
struct Lay {
  static constexpr int LP = L + L / R1;
  static __device__ __forceinline__ int put(int r, int c) { return ROW ? c * LP + r : r * NT + c; }
  static __device__ __forceinline__ int at(int i, int c) { return put(i + i / R1, c); }
  // at(i + d, c) for a compile-time multiple d of R1: at(i, c) + step(d)
  static constexpr int step(int d) { return (d + d / R1) * (ROW ? 1 : NT); }
};
template <int L, int NT> struct BufSize {  // complex values of LDS, either pass order
  using P = Plan<L>;
  static constexpr int RL = P::R3 > 1 ? P::R3 : P::R2;
  static constexpr int RM = P::R1 < RL ? P::R1 : RL;
  static constexpr int value = (L + L / RM) * NT;
};

// Twiddle tables in LDS, in the order the passes read them ([q][k], k consecutive over
// lanes): t3[q * NS + k] for the last pass (NS = L / its radix), and for three passes
// t2[q * R1 + k] for the middle one. REV: the radices reversed.
template <int L, bool REV>
struct Tables {
  using P = Plan<L>;
  static constexpr bool three = P::R3 > 1;
  static constexpr int RL = three ? P::R3 : P::R2;
  static constexpr int A = REV ? RL : P::R1, M = three ? P::R2 : 1, Z = REV ? P::R1 : RL;
  static constexpr int N2 = three ? A * M : 0, SIZE = L + N2;
  static __device__ __forceinline__ void fill(float2* t, const float2* __restrict__ tw, int tid, int nthr) {
    constexpr int NS = L / Z;
    for (int e = tid; e < L; e += nthr) t[e] = tw[(e / NS) * (e % NS)];
    if constexpr (three)
      for (int e = tid; e < N2; e += nthr) t[L + e] = tw[(e / A) * (e % A) * (L / N2)];
  }
};

// The passes after the first: v holds thread j's first-pass inputs (zeros for j >= L / A);
// x receives outputs i = j + q L / Z of the transform for j < L / Z. The caller has
// synchronised since buf was last read; the tables may still be being written.
template <int L, int NT, bool ROW, bool REV, int RF, int RZ>
__device__ __forceinline__ void finish(float2 (&v)[RF], float2 (&x)[RZ], float2* buf, const float2* tab, int j, int c) {
  using TB = Tables<L, REV>;
  constexpr int A = TB::A, M = TB::M, Z = TB::Z;
  static_assert(RF == A && RZ == Z, "first and last radix");
  using LY = Lay<L, A, NT, ROW>;
  constexpr int T = Plan<L>::T;
  dft<A>(v);
  if (L / A == T || j < L / A) {
#pragma unroll
    for (int q = 0; q < A; ++q) buf[LY::put(j * (A + 1), c) + q * (ROW ? 1 : NT)] = v[q];  // at(j A + q)
  }
  __syncthreads();
  if constexpr (TB::three) {
    constexpr int NB = L / M;
    static_assert(NB % A == 0, "strides of the skewed layout");
    const int k = j % A;
    float2 u[M];
    if (NB == T || j < NB) {
#pragma unroll
      for (int q = 0; q < M; ++q) {
        const float2 y = buf[LY::at(j, c) + LY::step(q * NB)];
        u[q] = q == 0 ? y : cmul(y, tab[L + q * A + k]);
      }
      dft<M>(u);
    }
    __syncthreads();
    if (NB == T || j < NB) {
      const int base = (j / A) * (A * M) + k;
#pragma unroll
      for (int q = 0; q < M; ++q) buf[LY::at(base, c) + LY::step(q * A)] = u[q];
    }
    __syncthreads();
  }
  constexpr int NS = L / Z;
  if (NS == T || j < NS) {
    const int r = TB::three ? j + j / A : j;  // two passes: j < NS = A
#pragma unroll
    for (int q = 0; q < Z; ++q) {
      const float2 y = buf[LY::put(r, c) + LY::step(q * NS)];
      x[q] = q == 0 ? y : cmul(y, tab[q * NS + j]);
    }
    dft<Z>(x);
  }
}

// out(i, i - j, value) for this thread's outputs of finish.
template <int L, bool REV, int RZ, class Out>
__device__ __forceinline__ void emit(const float2 (&x)[RZ], int j, Out&& out) {
  constexpr int NS = L / RZ;
  if (NS == Plan<L>::T || j < NS) {
#pragma unroll
    for (int q = 0; q < RZ; ++q) out(j + q * NS, q * NS, x[q]);
  }
}

// The outputs of finish back into buf, each transform in order (row layout).
template <int L, int NT, bool REV, int RZ>
__device__ __forceinline__ void stage_rows(const float2 (&x)[RZ], float2* buf, int j, int c) {
  using LY = Lay<L, Tables<L, REV>::A, NT, true>;
  constexpr int NS = L / RZ;
  __syncthreads();
  if (NS == Plan<L>::T || j < NS) {
    const int r = Tables<L, REV>::three ? j + j / Tables<L, REV>::A : j;
#pragma unroll
    for (int q = 0; q < RZ; ++q) buf[LY::put(r, c) + LY::step(q * NS)] = x[q];
  }
  __syncthreads();
}

// Rows (transforms along the contiguous axis): the first pass reads L / A consecutive points
// at once; the radices are reversed where that makes it whole 128-byte segments (10 lanes of
// 8 bytes instead of 16 cost crop_row at L = 160 525 us of its 316 before, at 128^3 x 32).
template <int L>
struct RowOrder {
  using P = Plan<L>;
  static constexpr bool REV = P::R3 == 1 && (L / P::R1) % 16 != 0 && (L / P::R2) % 16 == 0;
  using TB = Tables<L, REV>;
  static constexpr bool STAGE = (L / TB::Z) % 16 != 0;  // outputs through LDS, for the same reason
};

// Thread j's first-pass inputs: in(i, i - j) for i = j + q L / A (i - j is the same in all threads).
template <int L, int RF, class In>
__device__ __forceinline__ void load_first(float2 (&v)[RF], int j, In&& in) {
  constexpr int NB = L / RF;
  if (NB == Plan<L>::T || j < NB) {
#pragma unroll
    for (int q = 0; q < RF; ++q) v[q] = in(j + q * NB, q * NB);
  } else {
#pragma unroll
    for (int q = 0; q < RF; ++q) v[q] = make_float2(0.f, 0.f);
  }
}

// A column block's slab is L <= 640 rows of `inner` values, under 2 GiB (inner is at most
// 640^2 for the supported grids).
constexpr long long kMaxInner = ((1LL << 31) - 1) / (8 * 640);

// Whether a length has a compiled radix plan.
__host__ __device__ inline bool plan_supported(int L) {
  switch (L) {
    case 64: case 80: case 96: case 120: case 128: case 160: case 192: case 240: case 256: case 320:
    case 384: case 480: case 512: case 640: return true;
    default: return false;
  }
}

// Calls f(integral_constant<L>) for a supported runtime length; returns f's status or
// fails for other lengths.
template <class F>
int with_length(int L, F&& f) {
  switch (L) {
#define MRA_FFT_LEN(LL) \
  case LL: return f(std::integral_constant<int, LL>{});
    MRA_FFT_LEN(64) MRA_FFT_LEN(80) MRA_FFT_LEN(96) MRA_FFT_LEN(120) MRA_FFT_LEN(128) MRA_FFT_LEN(160)
    MRA_FFT_LEN(192) MRA_FFT_LEN(240) MRA_FFT_LEN(256) MRA_FFT_LEN(320) MRA_FFT_LEN(384) MRA_FFT_LEN(480)
    MRA_FFT_LEN(512) MRA_FFT_LEN(640)
#undef MRA_FFT_LEN
    default: return -1;
  }
}

}  // namespace fft
}  // namespace mra


