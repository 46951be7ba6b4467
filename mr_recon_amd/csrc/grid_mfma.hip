// Gridding phase 1 on the matrix cores (v_mfma_f32_16x16x4f32), accumulated in registers.
//
// A work item is a tile's slice of sorted samples; its result is the tile's subgrid (SUB^D
// points, SUB = T + P - 1) of every coil, stored dense to the item's scratch slot. The KB
// weight of a sample is separable, so the samples that share a corner row (2D) or a cell of
// corners (3D) add up as a matrix product with K = samples:
//
//   2D:  R[(z, coil, re/im), x]      += sum_s (w0_s[z - l0] y_s[coil]) * w1_s[x - l1]
//   3D:  R[(z, coil, re/im), (p1, x)] += sum_s (w0_s[z - l0] y_s[coil]) * (w1_s[p1 - l1] w2_s[x - l2])
//
// One wave owns a few coils of an item and keeps the whole moving part of the subgrid in its
// accumulators: the 16 rows of a matrix block are R slots of a ring along dim 0 (slot of
// subgrid plane z = z mod R, R >= the patch's planes) times 16 / (2R) coils times re/im, the
// 16 columns a window of subgrid columns. The plan orders an item's samples by dim 0 first, so
// a plane is final once a sample with a higher corner plane arrives: its slot is stored and
// cleared. No partial sum goes through LDS and nothing is read back. LDS only turns the samples
// (one lane each, gathered a chunk ahead) into matrix operands.
//
// Rows / columns / blocks:
//   2D  corners are taken 8 at a time (window w: corner columns 8w .. 8w+7, which reach
//       columns 8w .. 8w + 7 + P - 1, at most 16): one block per window.
//   3D  P <= 5: cells of 2 rows x 4 columns of corners (contiguous in the plan's order) reach
//       (P + 1) x (P + 3) points; a block is 2 rows x 8 columns, (P + 2) / 2 blocks per cell.
//       P >= 6: row pairs (2 x 8 corners); a block is one row x 16 columns, P + 1 blocks.
//   R = 4 where the samples reach at most 4 planes, else 8. With P = 5 that holds for every
//   sample but those whose t - w/2 falls on a grid integer (w = 4: the k-space centre of radial
//   trajectories, and one in some 60 000 by rounding). An item with one of them takes R = 8: in 2D
//   with twice the blocks for the same coils, in 3D, where those would cost a third of the waves,
//   for half the coils at a time. A 2D launch lasts as long as such items: at half the coils they
//   took twice the chain (40 us in the 131 k x 16 case below, 878 us against 835 for 2 M radial
//   samples x 32).
//
// Values that would not stay inside the patch: a block also multiplies a sample's zero weights
// outside its patch, and 0 * inf = nan. Samples with a k-space value (times dcf) or weights that
// are not finite or could overflow in a product are therefore left out of the matrix products
// and added to their patch one by one at the end (grid_odd_samples).
//
// What bounds it: latency in 2D (a wave's chain of chunks: 20 rows to store and ~16 groups per
// chunk; 131 k samples x 16 coils, P 5: matrix cores 12 % busy, LDS 10 %, and 44 % of the CU cycles
// without a wave, since the launch ends on its longest items), in 3D the chains of its two waves
// per SIMD (5.12 M x 32: matrix cores 41 % busy, LDS 15 %, 7.9 GB moved in 2.4 ms; skipping all
// but one of a group's products takes 11 % off, skipping the gathers 20 %). Phase 1 before (2D:
// per-lane LDS read-modify-writes; 3D: products per cell added to an LDS plane ring) and now, MI355X:
//   3D 5.12 M samples x 32 coils, P 5   4.88 -> 2.30 ms     0.76 M x 7, P 7   1.00 -> 0.33 ms
//   3D 1.5 M samples x 1, P 5            155 -> 110 us      2D 131 k x 16, P 5  80 -> 30 us
//   2D 131 k samples x 16, P 7            94 -> 34 us       2D 4096 x 1, P 7    83 -> 15 us
#include <type_traits>

#include "grid_mfma.h"

namespace mra {

typedef float v4f __attribute__((ext_vector_type(4)));

namespace {

constexpr int kCh = 64;        // samples per LDS stage (one per lane)
constexpr int kRows = kCh + 4; // stage records: a group's operand loads run up to 3 past its samples
constexpr float kHuge = 1e37f; // products of staged operands stay below this

// Orders LDS accesses of one wave for the compiler; the hardware runs them in order.
__device__ __forceinline__ void wave_fence() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

__device__ __forceinline__ float max_abs(float m, float a, float b) {  // NaN wins
  return __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, fabsf(a)), fabsf(b));
}

// Lane i of each 16 gets lane (i + 8) % 16.
__device__ __forceinline__ float swap_halves(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xf, 0xf, true));
}
// Lane i of each 16 gets lane i - 4 (lanes 0..3: 0).
__device__ __forceinline__ float shift4(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x114, 0xf, 0xf, true));
}

// Calls f(integral_constant<int, E>) with E = row mod 4. The tests are kept apart (each on a copy
// the compiler knows nothing about): as one switch, the merge of its cases would hold the
// accumulators twice.
template <class F>
__device__ __forceinline__ void with_element(int row, F&& f) {
  auto test = [&](auto E) {
    int e = row & 3;
    asm("" : "+s"(e));
    if (e == E.value) f(E);
  };
  test(std::integral_constant<int, 0>{});
  test(std::integral_constant<int, 1>{});
  test(std::integral_constant<int, 2>{});
  test(std::integral_constant<int, 3>{});
}

// Takes element E out of a result block and clears it on the lanes of the retired slot. The value
// goes to a register of its own before the element is overwritten: read in place, it would keep
// the old block alive beside the new one.
template <int E>
__device__ __forceinline__ float take(v4f& a, bool act) {
  float v = a[E];
  asm("" : "+v"(v));
  a[E] = act ? 0.f : v;
  return v;
}

// Stores of an item's subgrids: byte offset lane_off + off from the item's slot. The hardware
// drops a store whose lane_off is past the nc subgrids of the slot; `off` is no part of that
// check, so it only moves inside one subgrid, and lane_off carries the coil (past the range for
// coils past the last) or kNoLane (lanes without a value).
struct SlotStore {
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ __forceinline__ SlotStore(float2* dst, int nbytes)
      : rsrc(__builtin_amdgcn_make_buffer_rsrc(dst, 0, nbytes, 0x00020000)) {}
  __device__ __forceinline__ void put(float v, int lane_off, int off) const {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), rsrc, lane_off, off, 0);
  }
};
// Clears planes lo .. hi-1 (PP points each) of the nc coils' subgrids (SUBN points, coil after coil).
__device__ __forceinline__ void clear_planes(float2* dst, int lo, int hi, int nc, int PP, int SUBN, int lane) {
  const int n = (hi - lo) * PP;
  for (int c = 0; c < nc; ++c) {
    float2* d = dst + (long long)c * SUBN + lo * PP;
    for (int e = lane; e < n; e += 64) d[e] = make_float2(0.f, 0.f);
  }
}
constexpr int kNoLane = 0x40000000;  // lane offset past any slot

// NB consecutive floats of LDS (16-byte aligned for NB = 4).
template <int NB>
__device__ __forceinline__ void load_vec(float (&y)[NB], const float* p) {
  if constexpr (NB % 4 == 0) {
#pragma unroll
    for (int n = 0; n < NB; n += 4) {
      const v4f v = *(const v4f*)(p + n);
#pragma unroll
      for (int e = 0; e < 4; ++e) y[n + e] = v[e];
    }
  } else {
#pragma unroll
    for (int n = 0; n < NB; ++n) y[n] = p[n];
  }
}

// One lane's sample: plan data, the k-space values of NC coils and the factor on them. Values are
// kept as loaded: arithmetic on them here would wait for the loads.
template <int D, int P, int NC>
struct Sample {
  int base;
  float w[D * P];
  float2 y[NC];
  float dc;
  __device__ __forceinline__ void scale(float s) {
    s *= dc;
#pragma unroll
    for (int c = 0; c < NC; ++c) y[c] = make_float2(y[c].x * s, y[c].y * s);
  }
};

// Loads sorted sample gs (sample slot o). Lanes past the item's end are given its last sample and
// coils past the last are given the last coil's values, so that no load is conditional: neither
// reaches a stored result.
template <int D, int P, int NC>
__device__ __forceinline__ void load_sample(Sample<D, P, NC>& r, long long gs, int o, const float2* __restrict__ ksp,
                                            const float* __restrict__ dcf, const float* __restrict__ wsort,
                                            const int* __restrict__ lbase, const Geom& g, int c0, int nc) {
  r.base = lbase[gs];
  const float* wp = wsort + gs * (D * P);
#pragma unroll
  for (int e = 0; e < D * P; ++e) r.w[e] = wp[e];
  r.dc = dcf ? dcf[g.dcf_plan_order ? gs : g.samp_off + o] : 1.0f;
#pragma unroll
  for (int c = 0; c < NC; ++c) r.y[c] = ksp[g.ksp_off + (long long)(c0 + min(c, nc - 1)) * g.ksp_stride + o];
}

// Whether a sample stays out of the matrix products (see the file comment).
template <int D, int P, int NC>
__device__ __forceinline__ bool odd_sample(const Sample<D, P, NC>& r) {
  float ym = 0.f, m0 = 0.f, m1 = 0.f, m2 = 1.f;
#pragma unroll
  for (int c = 0; c < NC; ++c) ym = max_abs(ym, r.y[c].x, r.y[c].y);
#pragma unroll
  for (int j = 0; j < P; ++j) {
    m0 = __builtin_elementwise_maximum(m0, fabsf(r.w[j]));
    m1 = __builtin_elementwise_maximum(m1, fabsf(r.w[P + j]));
    if constexpr (D == 3) m2 = __builtin_elementwise_maximum(m2, fabsf(r.w[2 * P + j]));
  }
  return !(ym * m0 < kHuge) || !(m1 * m2 < kHuge);
}

// The item's left-out samples, one after the other: a lane per patch point adds to the stored
// subgrid. Rare, so serial and fenced.
template <int D, int P, int T, int NC>
__device__ __noinline__ void grid_odd_samples(const float2* __restrict__ ksp, const float* __restrict__ dcf,
                                              const float* __restrict__ wsort, const int* __restrict__ lbase,
                                              const int* __restrict__ perm, const Geom* __restrict__ geoms,
                                              const Item* __restrict__ items, int iidx, int c0, int nc, float2* dst) {
  constexpr int SUB = T + P - 1, SUBN = ipow(SUB, D), NPT = ipow(P, D);
  const Item it = items[iidx];
  const Geom g = geoms[it.x];
  const int lane = threadIdx.x;
  const long long gs0 = g.samp_off + it.z;
  int edge = 0;
  for (int s = lane; s < it.w; s += 64) edge |= wsort[(gs0 + s) * (D * P) + P - 1] != 0.0f;
  const int PE = (P >= 3 && !__any(edge)) ? P - 1 : P;  // planes the item's samples reach
  for (int s0 = 0; s0 < it.w; s0 += 64) {
    const long long gs = gs0 + min(s0 + lane, it.w - 1);
    Sample<D, P, NC> r;
    load_sample<D, P, NC>(r, gs, sample_slot(perm, g, gs), ksp, dcf, wsort, lbase, g, c0, nc);
    r.scale(g.out_scale);
    unsigned long long todo = __ballot(s0 + lane < it.w && odd_sample<D, P, NC>(r));
    while (todo) {
      const int l = (int)__builtin_ctzll(todo);
      todo &= todo - 1;
      const long long gl = gs0 + s0 + l;
      const int ol = sample_slot(perm, g, gl), base = lbase[gl];
      const float* w = wsort + gl * (D * P);
      const float sc = dcf ? dcf[g.dcf_plan_order ? gl : g.samp_off + ol] * g.out_scale : g.out_scale;
      for (int c = 0; c < nc; ++c) {
        float2 y = ksp[g.ksp_off + (long long)(c0 + c) * g.ksp_stride + ol];
        y.x *= sc;
        y.y *= sc;
        __threadfence();
        for (int p = lane; p < NPT; p += 64) {
          const int p0 = p / (NPT / P), rest = p - p0 * (NPT / P);
          if (p0 >= PE) continue;
          int off;
          float wr;
          if constexpr (D == 3) {
            off = (p0 * SUB + rest / P) * SUB + rest % P;
            wr = w[P + rest / P] * w[2 * P + rest % P];
          } else {
            off = p0 * SUB + rest;
            wr = w[P + rest];
          }
          volatile float* q = (volatile float*)(dst + (long long)c * SUBN + base + off);
          q[0] = q[0] + w[p0] * (wr * y.x);
          q[1] = q[1] + w[p0] * (wr * y.y);
        }
        __threadfence();
      }
    }
  }
}

// Does a sample of the item reach the last patch plane (last dim-0 weight not 0)? Wave-uniform.
// Loads go out eight at a time: one by one they would be a chain of memory latencies.
template <int D, int P>
__device__ __forceinline__ bool reaches_last_plane(const float* __restrict__ wsort, const Geom& g, const Item& it) {
  const float* w = wsort + (g.samp_off + it.z) * (D * P) + P - 1;
  bool any = false;
  for (int s0 = 0; s0 < it.w; s0 += 512) {
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = w[(long long)min(s0 + 64 * j + (int)threadIdx.x, it.w - 1) * (D * P)];
#pragma unroll
    for (int j = 0; j < 8; ++j) any = any || v[j] != 0.0f;
  }
  return __any(any);
}

// The stage's samples cut into groups of up to 4 with one key: every fourth sample from the start
// of its run of equal keys. Lane g's word is group g (kEnd past the last): key << 16 | byte offset
// of its first sample's record (a multiple of 16) | its samples.
constexpr int kEnd = 0x7fff0000;
struct Groups {
  int n;     // groups of the stage
  int word;
  __device__ __forceinline__ Groups(int key, int ns, int lane, int rec_bytes, int* list) {
    const int kprev = __shfl_up(key, 1);
    const unsigned long long runs = __ballot(lane < ns && (lane == 0 || key != kprev));
    const unsigned long long upto = lane == 63 ? ~0ull : (2ull << lane) - 1;
    const int pos = (lane - (63 - __builtin_clzll((runs & upto) | 1ull))) & 3;
    const bool start = lane < ns && pos == 0;
    const unsigned long long gm = __ballot(start);
    n = __popcll(gm);
    if (start) {
      const unsigned long long later = gm & ~upto;
      const int end = later ? (int)__builtin_ctzll(later) : ns;
      list[__popcll(gm & upto) - 1] = key << 16 | lane * rec_bytes | (end - lane);
    }
    wave_fence();
    word = lane < n ? list[lane] : kEnd;
  }
  __device__ __forceinline__ int at(int g) const { return g < n ? __builtin_amdgcn_readlane(word, g) : kEnd; }
};

// Ring of a wave: R slots (4 where the samples reach at most 4 planes, else 8) times the (coil,
// re/im) components of 16 / R rows, NB matrix blocks. Component 2c + re/im of block nb is coil
// c NB + nb.
template <int P, int NB, int R>
struct Ring {
  static_assert((R == 4 && P <= 5) || R == 8, "ring");
  static constexpr int NC = NB * 8 / R;        // coils of a wave
  static constexpr int YC = 16 / R;            // components staged
  static __device__ __forceinline__ int slot(int row16) { return row16 & (R - 1); }
  static __device__ __forceinline__ int comp(int row16) { return row16 / R; }
  // result layout: lane group q holds rows 4q .. 4q+3, so element e is slot e (4 slots) or
  // 4 (q mod 2) + e (8 slots) of component:
  static __device__ __forceinline__ int comp_of_group(int q) { return R == 4 ? q : q >> 1; }
  static __device__ __forceinline__ bool holds(int q, int plane) { return R == 4 || (q & 1) == ((plane >> 2) & 1); }
};
constexpr int ring_slots(int P) { return P <= 5 ? 4 : 8; }  // of items that miss the fifth plane

// ---- 2D -------------------------------------------------------------------------------------

template <int P_, int T_, int NB_, int R>
struct Rows2 : Ring<P_, NB_, R> {
  using Ring<P_, NB_, R>::YC;
  static constexpr int P = P_, T = T_, NB = NB_;
  static constexpr int SUB = T + P - 1, SUBN = SUB * SUB;
  static constexpr int NW = T / 8;             // windows of 8 corners per row
  static constexpr int NK = (SUB + 15) / 16;   // 16-column stores per subgrid row
  // stage record of a sample (floats): 16 dim-1 weights, R dim-0 weights, the k-space values by
  // component; padded so that 16-byte accesses of consecutive lanes spread over all banks
  static constexpr int ZN = R, ZO = 16, YO = ZO + ZN;
  static constexpr int RS = (YO + YC * NB) % 8 == 4 ? YO + YC * NB : (YO + YC * NB + 8) / 8 * 8 - 4;
  static_assert(P <= 8 && 7 + P <= 16 && SUB <= 8 * (NW + 1), "window");
};

// Subgrid row `row` is final: store it (ring slot row mod R, accumulator element E = row mod 4)
// and clear its slot. Columns 8w .. 8w+7 are the first half of window w plus the second half of
// window w - 1.
template <class M, int E>
__device__ __forceinline__ void retire_row(v4f (&acc)[M::NW][M::NB], int row, int lane,
                                           const SlotStore& out) {
  const int x = lane & 15, q = lane >> 4;
  const int comp = M::comp_of_group(q);
  const int loff = ((comp >> 1) * M::NB * M::SUBN + x) * 8 + (comp & 1) * 4;
  const bool act = M::holds(q, row);
  const int l0 = act ? loff : kNoLane;
  const int l1 = M::SUB % 16 == 0 || x < M::SUB % 16 ? l0 : kNoLane;  // the last, partial 16 columns
#pragma unroll
  for (int nb = 0; nb < M::NB; ++nb) {
    float v[M::NW], r[M::NW];
#pragma unroll
    for (int w = 0; w < M::NW; ++w) {
      v[w] = take<E>(acc[w][nb], act);
      r[w] = M::NW > 1 ? swap_halves(v[w]) : 0.f;
    }
#pragma unroll
    for (int k = 0; k < M::NK; ++k) {
      const float a = 2 * k < M::NW ? v[2 * k < M::NW ? 2 * k : 0] : 0.f;
      const float lo = (2 * k >= 1 && 2 * k - 1 < M::NW) ? r[2 * k >= 1 ? (2 * k - 1) % M::NW : 0] : 0.f;
      const float hi = 2 * k + 1 < M::NW ? r[(2 * k + 1) % M::NW] : 0.f;
      out.put(a + (x < 8 ? lo : hi), (k + 1 < M::NK ? l0 : l1) + nb * (M::SUBN * 8), (row * M::SUB + 16 * k) * 8);
    }
  }
}

// One item of a coil chunk.
template <class M>
__device__ __forceinline__ void rows2_item(const float2* __restrict__ ksp, const float* __restrict__ dcf,
                                           const float* __restrict__ wsort, const int* __restrict__ lbase,
                                           const int* __restrict__ perm, const Geom* __restrict__ geoms,
                                           const Item* __restrict__ items, const Geom& g, const Item& it, int iidx,
                                           int c0, int nc, float2* __restrict__ scratch, float* rec,
                                           int* list) {
  constexpr int P = M::P, NB = M::NB, SUB = M::SUB;
  int lane = threadIdx.x;
  asm volatile("" : "+v"(lane));  // keeps lane terms from being carried across the caller's loop
  const int i16 = lane & 15;
  const int kq = (lane >> 4) ^ 2;  // the group's sample in this lane's K slot (their order is free)
  const int zl = M::slot(i16), comp = M::comp(i16);  // this lane's A row
  // byte offsets of this lane's operands from its group's first record
  const int off_w0 = (kq * M::RS + M::ZO) * 4, off_b = (kq * M::RS + i16) * 4;
  const int off_y = (kq * M::RS + M::YO + comp * NB) * 4;
  const int cnt = it.w;
  const long long gs0 = g.samp_off + it.z;
  float2* dst2 = scratch + g.scratch_off + ((long long)(iidx - g.item_base) * g.nbatch + c0) * M::SUBN;
  const SlotStore out(dst2, nc * (M::SUBN * 8));

  Sample<2, P, M::NC> sr;
  const long long gs_end = gs0 + cnt - 1;
  int onext = sample_slot(perm, g, min(gs0 + lane, gs_end));
  auto gather = [&](int s0) {
    load_sample<2, P, M::NC>(sr, min(gs0 + s0 + lane, gs_end), onext, ksp, dcf, wsort, lbase, g, c0, nc);
    onext = sample_slot(perm, g, min(gs0 + s0 + kCh + lane, gs_end));
  };
  gather(0);

  // records past the stage are read as operands (with zero weight): keep them finite
  for (int e = lane; e < (kRows - kCh) * M::RS; e += 64) rec[kCh * M::RS + e] = 0.f;

  v4f acc[M::NW][NB];
#pragma unroll
  for (int w = 0; w < M::NW; ++w)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[w][nb] = v4f{0.f, 0.f, 0.f, 0.f};

  // Rows the item's samples cannot reach are zero; the ring holds row .. row + R - 1
  const int first = lbase[gs0] / SUB, last = min(lbase[gs_end] / SUB + P, SUB);
  clear_planes(dst2, 0, first, nc, M::SUB, M::SUBN, lane);
  clear_planes(dst2, last, SUB, nc, M::SUB, M::SUBN, lane);
  int row = first;  // lowest row not yet stored
  auto retire_to = [&](int to) {
    for (; row < to; ++row) with_element(row, [&](auto E) { retire_row<M, E.value>(acc, row, lane, out); });
  };

  bool any_odd = false;
  for (int s0 = 0; s0 < cnt; s0 += kCh) {
    const int n = min(kCh, cnt - s0);
    sr.scale(g.out_scale);
    const bool odd = odd_sample<2, P, M::NC>(sr);
    any_odd = any_odd || __any(odd);
    const int l0 = sr.base / SUB, l1 = sr.base - l0 * SUB;
    const int key = (l0 << 2) | (l1 >> 3);
    wave_fence();
    const Groups gr(key, n, lane, M::RS * 4, list);
    {
      float* z = rec + lane * M::RS + M::ZO;
#pragma unroll
      for (int j = 0; j < M::ZN; j += 4) {
        v4f v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = j + e < P ? (odd ? 0.f : sr.w[j + e < P ? j + e : 0]) : 0.f;
        *(v4f*)(z + j) = v;
      }
      float* b = rec + lane * M::RS;
#pragma unroll
      for (int j = 0; j < 16; j += 4) *(v4f*)(b + j) = v4f{0.f, 0.f, 0.f, 0.f};
      wave_fence();
#pragma unroll
      for (int j = 0; j < P; ++j) b[(l1 & 7) + j] = odd ? 0.f : sr.w[P + j];
      float* y = rec + lane * M::RS + M::YO;
#pragma unroll
      for (int c = 0; c < M::YC; ++c)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const float2 v = sr.y[(c >> 1) * NB + nb];
          y[c * NB + nb] = odd ? 0.f : ((c & 1) ? v.y : v.x);
        }
    }
    wave_fence();
    if (s0 + kCh < cnt) gather(s0 + kCh);  // lands while this chunk is accumulated

    struct Ops {
      float w0, b, y[NB];
    } o;
    int g = 0, d = gr.at(0);  // the group whose operands are in `o`
    auto load_w0 = [&]() {  // this lane's ring slot holds patch plane zl - row (mod slots)
      o.w0 = *(const float*)((const char*)rec + (d & 0xfff0) + off_w0 + M::slot(zl - row) * 4);
    };
    auto load = [&]() {
      const char* p = (const char*)rec + (d & 0xfff0);
      load_w0();
      o.b = *(const float*)(p + off_b);
      load_vec<NB>(o.y, (const float*)(p + off_y));
    };
    load();
    while (d != kEnd) {
      if ((d >> 18) > row) {  // the loaded operands' ring position moves with the row
        retire_to(d >> 18);
        load_w0();
      }
      const int kr = (d >> 16) & ~3;
      // the row's windows in the plan's order; each loop owns its blocks' registers
      auto groups = [&](auto W) {
        while ((d >> 16) == kr + W.value) {
          const float w0 = kq < (d & 7) ? o.w0 : 0.f, bv = o.b;
          float a[NB];
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) a[nb] = w0 * o.y[nb];
          d = gr.at(++g);
          load();  // the next group's operands arrive behind this group's products
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int nb = 0; nb < NB; ++nb)
            acc[W.value][nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[nb], bv, acc[W.value][nb], 0, 0, 0);
        }
      };
      groups(std::integral_constant<int, 0>{});
      if constexpr (M::NW > 1) groups(std::integral_constant<int, 1>{});
      if constexpr (M::NW > 2) groups(std::integral_constant<int, 2>{});
      if constexpr (M::NW > 3) groups(std::integral_constant<int, 3>{});
    }
  }
  retire_to(last);
  if (any_odd) grid_odd_samples<2, P, M::T, M::NC>(ksp, dcf, wsort, lbase, perm, geoms, items, iidx, c0, nc, dst2);
}

// One wave per (item, coil chunk).
template <int P, int T, int NB>
__global__ __launch_bounds__(64) void grid_rows2d_kernel(const float2* __restrict__ ksp,
                                                         const float* __restrict__ dcf,
                                                         const float* __restrict__ wsort,
                                                         const int* __restrict__ lbase,
                                                         const int* __restrict__ perm,
                                                         const Geom* __restrict__ geoms,
                                                         const Item* __restrict__ items, int nitems, int nchunks,
                                                         float2* __restrict__ scratch) {
  constexpr int R = ring_slots(P);
  using M = Rows2<P, T, NB, R>;
  using W = Rows2<P, T, NB * (8 / R), 8>;  // the same coils with 8 slots
  __shared__ __attribute__((aligned(16))) float rec[kRows * (P == 5 && W::RS > M::RS ? W::RS : M::RS)];
  __shared__ int list[kCh];
  int iidx, cc;
  item_of_block(blockIdx.x, nchunks, iidx, cc);
  if (iidx >= nitems) return;
  const Item it = items[iidx];
  if (it.w <= 0 || it.y < 0) return;  // non-finite coordinates contribute nothing
  const Geom g = geoms[it.x];
  const int c0 = cc * M::NC;
  if (c0 >= g.nbatch) return;
  const int nc = min(M::NC, g.nbatch - c0);
  if constexpr (P == 5) {
    if (reaches_last_plane<2, P>(wsort, g, it)) {
      rows2_item<W>(ksp, dcf, wsort, lbase, perm, geoms, items, g, it, iidx, c0, nc, scratch, rec, list);
      return;
    }
  }
  rows2_item<M>(ksp, dcf, wsort, lbase, perm, geoms, items, g, it, iidx, c0, nc, scratch, rec, list);
}

// ---- 3D -------------------------------------------------------------------------------------

template <int P_, int NB_, int R>
struct Cells3 : Ring<P_, NB_, R> {
  using Ring<P_, NB_, R>::YC;
  static constexpr int P = P_, NB = NB_;
  static constexpr int T = 8, SUB = T + P - 1, PP = SUB * SUB, SUBN = SUB * PP;
  static constexpr bool NARROW = P <= 5;              // blocks of 2 rows x 8 columns, else 1 x 16
  static constexpr int RP = NARROW ? 2 : 1;           // rows per block
  static constexpr int CW = NARROW ? 8 : 16;          // columns per block
  static constexpr int NH = NARROW ? 2 : 1;           // column windows (offset 4 apart)
  static constexpr int NBB = NARROW ? (P + 2) / 2 : P + 1;    // blocks a cell / row pair reaches
  static constexpr int NBLK = 6 / RP + NBB;           // blocks per plane and window
  // stage record of a sample (floats): 8 dim-1 weights, CW dim-2 weights, R dim-0 weights, the
  // k-space values by component; padded so that 16-byte accesses of consecutive lanes spread over
  // all banks
  static constexpr int XO = 8, ZN = R, ZO = XO + CW, YO = ZO + ZN;
  static constexpr int RS = (YO + YC * NB) % 8 == 4 ? YO + YC * NB : (YO + YC * NB + 8) / 8 * 8 - 4;
  static_assert(NBLK * RP >= SUB && (NARROW ? 3 : 7) + P <= CW && NBB <= 8, "blocks");
};

// Plane `pl` is final: store its slot (element E = pl mod 4) and clear it.
template <class M, int E>
__device__ __forceinline__ void retire_plane(v4f (&acc)[M::NH][M::NBLK][M::NB], int pl, int lane,
                                             const SlotStore& out) {
  asm volatile("" : "+v"(lane));  // lane terms are formed here, not held in registers between calls
  const int i16 = lane & 15, q = lane >> 4;
  const int comp = M::comp_of_group(q);
  const int r = M::NARROW ? i16 >> 3 : 0, x = M::NARROW ? i16 & 7 : i16;
  const int loff = ((comp >> 1) * M::NB * M::SUBN + r * M::SUB + x) * 8 + (comp & 1) * 4;
  const bool act = M::holds(q, pl);
  const bool lastrow = (M::NBLK - 1) * M::RP + r < M::SUB;  // rows of the last block
  const int l0 = act && x < M::SUB ? loff : kNoLane;
  const int l0e = lastrow ? l0 : kNoLane;
  const int l1 = act && x >= 4 && x + 4 < M::SUB ? loff + 32 : kNoLane;  // narrow: columns 8.. from window 1
  const int l1e = lastrow ? l1 : kNoLane;
#pragma unroll
  for (int nb = 0; nb < M::NB; ++nb)
#pragma unroll
    for (int b = 0; b < M::NBLK; ++b) {
      const int at = (pl * M::PP + b * M::RP * M::SUB) * 8, coil = nb * (M::SUBN * 8);
      const bool end = b + 1 == M::NBLK;
      if constexpr (M::NARROW) {
        // columns 0..3 window 0, 4..7 both, 8..11 window 1
        const float v0 = take<E>(acc[0][b][nb], act), v1 = take<E>(acc[1][b][nb], act);
        const float s1 = shift4(v1);
        out.put(x >= 4 ? v0 + s1 : v0, (end ? l0e : l0) + coil, at);
        out.put(v1, (end ? l1e : l1) + coil, at);
      } else {
        const float v = take<E>(acc[0][b][nb], act);
        out.put(v, (end ? l0e : l0) + coil, at);
      }
    }
}

// One item of a coil chunk.
template <class M>
__device__ __forceinline__ void cells3_item(const float2* __restrict__ ksp, const float* __restrict__ dcf,
                                            const float* __restrict__ wsort, const int* __restrict__ lbase,
                                            const int* __restrict__ perm, const Geom* __restrict__ geoms,
                                            const Item* __restrict__ items, const Geom& g, const Item& it, int iidx,
                                            int c0, int nc, float2* __restrict__ scratch, float* rec,
                                            int* list) {
  constexpr int P = M::P, NB = M::NB, SUB = M::SUB;
  int lane = threadIdx.x;
  asm volatile("" : "+v"(lane));  // keeps lane terms from being carried across the caller's loop
  const int i16 = lane & 15;
  const int kq = (lane >> 4) ^ 2;  // the group's sample in this lane's K slot (their order is free)
  const int zl = M::slot(i16), comp = M::comp(i16);  // this lane's A row
  const int br = M::NARROW ? i16 >> 3 : 0, bx = M::NARROW ? i16 & 7 : i16;  // B column: row, column in the block
  // byte offsets of this lane's operands from its group's first record
  const int off_w1 = (kq * M::RS + br * 4) * 4, off_w2 = (kq * M::RS + M::XO + bx) * 4;
  const int off_w0 = (kq * M::RS + M::ZO) * 4, off_y = (kq * M::RS + M::YO + comp * NB) * 4;
  const int cnt = it.w;
  const long long gs0 = g.samp_off + it.z;
  float2* dst2 = scratch + g.scratch_off + ((long long)(iidx - g.item_base) * g.nbatch + c0) * M::SUBN;
  const SlotStore out(dst2, nc * (M::SUBN * 8));

  Sample<3, P, M::NC> sr;
  const long long gs_end = gs0 + cnt - 1;
  int onext = sample_slot(perm, g, min(gs0 + lane, gs_end));
  auto gather = [&](int s0) {
    load_sample<3, P, M::NC>(sr, min(gs0 + s0 + lane, gs_end), onext, ksp, dcf, wsort, lbase, g, c0, nc);
    onext = sample_slot(perm, g, min(gs0 + s0 + kCh + lane, gs_end));
  };
  gather(0);

  // records past the stage are read as operands (with zero weight): keep them finite
  for (int e = lane; e < (kRows - kCh) * M::RS; e += 64) rec[kCh * M::RS + e] = 0.f;

  v4f acc[M::NH][M::NBLK][NB];
#pragma unroll
  for (int h = 0; h < M::NH; ++h)
#pragma unroll
    for (int b = 0; b < M::NBLK; ++b)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) acc[h][b][nb] = v4f{0.f, 0.f, 0.f, 0.f};

  // Planes the item's samples cannot reach are zero; the ring holds row .. row + R - 1
  const int first = lbase[gs0] / M::PP, last = min(lbase[gs_end] / M::PP + P, SUB);
  clear_planes(dst2, 0, first, nc, M::PP, M::SUBN, lane);
  clear_planes(dst2, last, SUB, nc, M::PP, M::SUBN, lane);
  int row = first;  // lowest plane not yet stored
  auto retire_to = [&](int to) {
    for (; row < to; ++row) with_element(row, [&](auto E) { retire_plane<M, E.value>(acc, row, lane, out); });
  };

  bool any_odd = false;
  for (int s0 = 0; s0 < cnt; s0 += kCh) {
    const int n = min(kCh, cnt - s0);
    sr.scale(g.out_scale);
    const bool odd = odd_sample<3, P, M::NC>(sr);
    any_odd = any_odd || __any(odd);
    const int l2 = sr.base % SUB, l01 = sr.base / SUB;
    const int l1 = l01 % SUB, l0 = l01 / SUB;
    const int key = (l0 << 3) | ((l1 >> 1) << 1) | (M::NARROW ? l2 >> 2 : 0);
    wave_fence();
    const Groups gr(key, n, lane, M::RS * 4, list);
    {
      float* z = rec + lane * M::RS + M::ZO;
#pragma unroll
      for (int j = 0; j < M::ZN; j += 4) {
        v4f v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = j + e < P ? (odd ? 0.f : sr.w[j + e < P ? j + e : 0]) : 0.f;
        *(v4f*)(z + j) = v;
      }
      // dim-1 weights of block row br, block b: region row 2b + br (narrow: [br][b]) or b
      float* u = rec + lane * M::RS;
      const bool o1 = l1 & 1;
      float wx[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float a = j < P ? sr.w[P + (j < P ? j : 0)] : 0.f;
        const float b = (j >= 1 && j - 1 < P) ? sr.w[P + (j >= 1 && j - 1 < P ? j - 1 : 0)] : 0.f;
        wx[j] = odd ? 0.f : (o1 ? b : a);
      }
      if constexpr (M::NARROW) {
        *(v4f*)u = v4f{wx[0], wx[2], wx[4], wx[6]};
        *(v4f*)(u + 4) = v4f{wx[1], wx[3], wx[5], wx[7]};
      } else {
        *(v4f*)u = v4f{wx[0], wx[1], wx[2], wx[3]};
        *(v4f*)(u + 4) = v4f{wx[4], wx[5], wx[6], wx[7]};
      }
      float* v = u + M::XO;
      const int o2 = M::NARROW ? l2 & 3 : l2;
#pragma unroll
      for (int j = 0; j < M::CW; j += 4) *(v4f*)(v + j) = v4f{0.f, 0.f, 0.f, 0.f};
      wave_fence();
#pragma unroll
      for (int j = 0; j < P; ++j) v[o2 + j] = odd ? 0.f : sr.w[2 * P + j];
      float* y = rec + lane * M::RS + M::YO;
#pragma unroll
      for (int c = 0; c < M::YC; ++c)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const float2 yv = sr.y[(c >> 1) * NB + nb];
          y[c * NB + nb] = odd ? 0.f : ((c & 1) ? yv.y : yv.x);
        }
    }
    wave_fence();
    if (s0 + kCh < cnt) gather(s0 + kCh);  // lands while this chunk is accumulated

    struct Ops {
      float w0, w2, w1[M::NARROW ? 4 : 8], y[NB];
    } o;
    int g = 0, d = gr.at(0);  // the group whose operands are in `o`
    auto load_w0 = [&]() {  // this lane's ring slot holds patch plane zl - row (mod slots)
      o.w0 = *(const float*)((const char*)rec + (d & 0xfff0) + off_w0 + M::slot(zl - row) * 4);
    };
    auto load = [&]() {
      const char* p = (const char*)rec + (d & 0xfff0);
      load_w0();
      load_vec<M::NARROW ? 4 : 8>(o.w1, (const float*)(p + off_w1));
      o.w2 = *(const float*)(p + off_w2);
      load_vec<NB>(o.y, (const float*)(p + off_y));
    };
    load();
    while (d != kEnd) {
      if ((d >> 19) > row) {  // the loaded operands' ring position moves with the plane
        retire_to(d >> 19);
        load_w0();
      }
      const int kr = (d >> 16) & ~7;
      // the plane's cells in the plan's order; each loop owns its blocks' registers
      auto groups = [&](auto J, auto H) {
        constexpr int j0 = J.value * 2 / M::RP, h = H.value, jh = J.value * 2 + h;
        while ((d >> 16) == kr + jh) {
          const float w0 = kq < (d & 7) ? o.w0 : 0.f;
          float a[NB], bv[M::NBB];
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) a[nb] = w0 * o.y[nb];
#pragma unroll
          for (int b = 0; b < M::NBB; ++b) bv[b] = o.w1[b] * o.w2;
          d = gr.at(++g);
          load();  // the next group's operands arrive behind this group's products
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int b = 0; b < M::NBB; ++b)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
              acc[h][j0 + b][nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[nb], bv[b], acc[h][j0 + b][nb], 0, 0, 0);
        }
      };
      auto row_pair = [&](auto J) {
        groups(J, std::integral_constant<int, 0>{});
        if constexpr (M::NARROW) groups(J, std::integral_constant<int, 1>{});
      };
      row_pair(std::integral_constant<int, 0>{});
      row_pair(std::integral_constant<int, 1>{});
      row_pair(std::integral_constant<int, 2>{});
      row_pair(std::integral_constant<int, 3>{});
    }
  }
  retire_to(last);
  if (any_odd) grid_odd_samples<3, P, M::T, M::NC>(ksp, dcf, wsort, lbase, perm, geoms, items, iidx, c0, nc, dst2);
}

template <int P, int NB>
__global__ __launch_bounds__(64) void grid_cells3d_kernel(const float2* __restrict__ ksp,
                                                          const float* __restrict__ dcf,
                                                          const float* __restrict__ wsort,
                                                          const int* __restrict__ lbase,
                                                          const int* __restrict__ perm,
                                                          const Geom* __restrict__ geoms,
                                                          const Item* __restrict__ items, int nitems, int nchunks,
                                                          float2* __restrict__ scratch) {
  constexpr int R = ring_slots(P);
  using M = Cells3<P, NB, R>;
  using W = Cells3<P, NB, 8>;
  __shared__ __attribute__((aligned(16))) float rec[kRows * (P == 5 && W::RS > M::RS ? W::RS : M::RS)];
  __shared__ int list[kCh];
  int iidx, cc;
  item_of_block(blockIdx.x, nchunks, iidx, cc);
  if (iidx >= nitems) return;
  const Item it = items[iidx];
  if (it.w <= 0 || it.y < 0) return;  // non-finite coordinates contribute nothing
  const Geom g = geoms[it.x];
  const int c0 = cc * M::NC;
  if (c0 >= g.nbatch) return;
  const int nc = min(M::NC, g.nbatch - c0);
  if constexpr (P == 5) {
    if (reaches_last_plane<3, P>(wsort, g, it)) {  // half the coils at a time
      for (int c = 0; c < nc; c += W::NC)
        cells3_item<W>(ksp, dcf, wsort, lbase, perm, geoms, items, g, it, iidx, c0 + c, min(W::NC, nc - c), scratch,
                       rec, list);
      return;
    }
  }
  cells3_item<M>(ksp, dcf, wsort, lbase, perm, geoms, items, g, it, iidx, c0, nc, scratch, rec, list);
}

// ---- launch ---------------------------------------------------------------------------------

template <int P, int T, int NB>
void launch_rows2(const GridMfmaArgs& a) {
  constexpr int NC = NB * 8 / ring_slots(P);
  const int nch = (a.nbatch + NC - 1) / NC;
  grid_rows2d_kernel<P, T, NB><<<item_grid(a.nitems, nch), 64, 0, a.stream>>>(
      a.ksp, a.dcf, a.wsort, a.lbase, a.perm, a.geoms, a.items, a.nitems, nch, a.scratch);
}

template <int P, int NB>
void launch_cells3(const GridMfmaArgs& a) {
  constexpr int NC = NB * 8 / ring_slots(P);
  const int nch = (a.nbatch + NC - 1) / NC;
  grid_cells3d_kernel<P, NB><<<item_grid(a.nitems, nch), 64, 0, a.stream>>>(
      a.ksp, a.dcf, a.wsort, a.lbase, a.perm, a.geoms, a.items, a.nitems, nch, a.scratch);
}

// Coils per wave. More of them share the staging and the control of a group, fewer leave more and
// shorter waves, which is what these latency-bound launches need. 2D phase 1, us at 2 / 4 / 8 / 16
// coils a wave, P = 5, and 1 / 2 / 4 / 8, P = 7:
//   131 k spiral samples x 16    33 /  30 /  36 /  47      49 /  38 /  34 /  41
//   131 k radial x 32            53 /  48 /  52 /  62      82 /  61 /  59 /  61
//   2 M spiral x 32             498 / 382 / 382 / 406     868 / 590 / 491 / 481
//   2 M radial x 32             777 / 829 / 822 / 870     874 / 780 / 814 / 825
// A single coil (or pair, with 4 slots) takes one block.
template <int P, int T>
void launch_2d(const GridMfmaArgs& a) {
  constexpr int per_block = 8 / ring_slots(P);
  if (a.nbatch <= per_block) launch_rows2<P, T, 1>(a);
  else launch_rows2<P, T, 4 / per_block>(a);
}

template <int P>
void launch_2d_t(int T, const GridMfmaArgs& a) {
  switch (T) {
    case 8: launch_2d<P, 8>(a); break;
    case 32: launch_2d<P, 32>(a); break;
    default: launch_2d<P, 16>(a); break;
  }
}

// As in 2D; the accumulators (24 registers per coil at P = 5, 56 at P = 7) set the waves per SIMD.
// 5.12 M samples x 32 coils at P = 5: 2 / 4 / 6 / 8 coils per wave take 2.82 / 2.58 / 2.73 / 3.08 ms;
// 0.76 M x 7 at P = 7: 1 / 2 / 3 / 4 coils 0.34 / 0.38 / 0.42 / 0.45 ms.
template <int P>
void launch_3d(const GridMfmaArgs& a) {
  if (P >= 6 || a.nbatch <= 8 / ring_slots(P)) launch_cells3<P, 1>(a);
  else launch_cells3<P, (P >= 6 ? 1 : 2)>(a);
}

}  // namespace

void launch_grid_mfma(int ndim, int P, int T, const GridMfmaArgs& a) {
  if (ndim == 2) {
    switch (P) {
      case 2: launch_2d_t<2>(T, a); break;
      case 3: launch_2d_t<3>(T, a); break;
      case 4: launch_2d_t<4>(T, a); break;
      case 5: launch_2d_t<5>(T, a); break;
      case 6: launch_2d_t<6>(T, a); break;
      case 7: launch_2d_t<7>(T, a); break;
      default: launch_2d_t<8>(T, a); break;
    }
  } else {
    switch (P) {
      case 2: launch_3d<2>(a); break;
      case 3: launch_3d<3>(a); break;
      case 4: launch_3d<4>(a); break;
      case 5: launch_3d<5>(a); break;
      case 6: launch_3d<6>(a); break;
      default: launch_3d<7>(a); break;
    }
  }
}

}  // namespace mra
