// Resident PCG: a whole Jacobi/identity PCG solve (pcg.jl:16-60) in one launch
// for meshes that fit the register files of the chip.
//
// Every workgroup owns a tile of TX x RY elements and keeps its share of r, p,
// x, d, G11, G12, G22 and B in registers (x in LDS where they run short) for the
// whole solve: thread (element, a) holds row a of its element, P nodes of each
// array. An iteration reads and writes no field in memory; workgroups exchange
// only the raw element outputs on the tile edges and the partials of the inner
// products, <p, A p> with the edges, <r, z> and norm(r, Inf) after the update.
// The recurrence is pcg.jl's, term by term. (The form with one exchange per
// iteration of Chronopoulos and Gear, s = A z + beta s, was 7.5 instead of 10 us
// at 128x128 elements, N = 7, but its rounding noise made the objective of the
// steady adjoint ten times less smooth in the coefficient, 3e-14 against 2e-15.)
//
// Exchange between workgroups (which may sit on different XCDs, so on
// different L2 caches): data travels in 64-bit words that also hold a tag of the
// iteration, written and polled with relaxed agent-scope atomics (for readers on the
// writer's XCD alone, written with stores that reach its L2: put). A word is either
// the awaited one or an older one, so no fence and no flag is needed. A workgroup
// writes its words of one exchange again only after the other exchange in between,
// for which every other workgroup must have finished reading, so one buffer for
// each of the two is enough. One value all-to-all:
// 1.7 us over 128 workgroups, 2.3 us over 256; two values 2.1 and 2.8 us (one
// 64-byte line per workgroup, one wave polling four lines a lane; lines shared by
// several writers, trees of two levels and a private copy per reader were
// slower: 3.0, 2.4 to 2.9 and 4.7 us for one value over 256).
//
// Why: two launches per iteration cost 16 to 30 us below 1.1M nodes (18.8 us at
// 64x64 elements, N = 7; 29.9 us at 128x128), most of it launch, load and store
// latency; here the fields never leave the registers.
//
// All workgroups have to be resident at once. The launch has at most one
// workgroup per CU, and a workgroup starts only after a rendezvous: if some
// workgroup does not arrive within kResWait (other work holds its CU), the
// first to run out of patience decides the launch off, every workgroup
// leaves without having changed anything, and the host runs the solve with one
// launch per step. Every later wait is bounded by kResPolls.
#pragma once
#include "sem_device.h"
#include "_gen/gll_dtables.h"

namespace sem {
namespace res {

using u64 = unsigned long long;

constexpr int kResWait = 1 << 15;    // rendezvous polls (about 20 ms)
constexpr int kResPolls = 1 << 24;   // polls of one word (several seconds)
constexpr int kSlotWords = 8;        // one 64-byte line per workgroup
constexpr int kMaxWg = 256;          // slots
constexpr int kGroups = 8;           // XCDs; workgroups go round them in turn
constexpr int kGroupWg = kMaxWg / kGroups;
// words of the exchanged lines: one per workgroup and one per group, twice
constexpr int kSlotArea = 2 * (kMaxWg + kGroups) * kSlotWords;
// Waves per workgroup: two per SIMD (256 registers each) while a thread's
// eight arrays leave room for the temporaries, else one per SIMD (512).
template <typename T, int P>
constexpr int kWaves = sizeof(T) * P <= 80 ? 8 : 4;
// x, which an iteration only adds to, in LDS where it would not leave the
// temporaries enough registers
template <typename T, int P>
constexpr bool kXLds = kWaves<T, P> == 8 && sizeof(T) * P >= 72;
// the exchange's arguments are read where they are used, not kept in registers (FP64,
// P = 8, 64x64 elements: 7.2 -> 7.0 us an iteration; at P = 5 0.1 slower)
template <typename T, int P>
constexpr bool kFresh = sizeof(T) * P >= 64;
template <int P>
constexpr int kEpw = 64 / P;         // elements per wave: none straddles two

template <typename T>
struct ResP {
  const T* __restrict__ b;   // right-hand side of a fresh solve (NULL: r, x hold the state)
  T* __restrict__ x;
  T* __restrict__ r;         // written when the solve will be continued
  T* __restrict__ p;
  const T* __restrict__ d;
  const T* __restrict__ G11;
  const T* __restrict__ G12;
  const T* __restrict__ G22;
  const T* __restrict__ B;
  const T* __restrict__ nu_f;
  const T* __restrict__ k_f;
  T nu, k;
  int has_mass;
  int Ex, Ey, TX, RY, ntx, nty, per_x, per_y, bc;
  u64* ymail;                // [nty][2][L] words (planes: low, high half)
  u64* xmail;                // [ntx][2][NC]
  u64* slots;                // [2][kMaxWg][kSlotWords]: <p, A p>; <r, z> and norm(r, Inf);
                             // then [2][kGroups][kSlotWords]: the groups' sums
  int nwg, near;             // workgroups that take part; the plan's form of exchange
  unsigned tag0;             // tags of this launch start above tag0
  ResCtl *ctl, *ctl_next;    // this launch's words; the next one's, which it clears (or NULL)
  PcgState* state;
  PcgHost* host;             // the state for the host, in its memory (or NULL: it copies)
  double tol;
  int maxiter, k_start, max_its, keep;
};

// A store that every reader of the device sees goes out of the XCD to memory. One
// for readers on the same XCD need only reach its L2, which all its CUs share and
// where their agent-scope loads (past their L1) find it. No scope of the language says
// that (workgroup scope gives this instruction, but promises other workgroups nothing), so
// it is written as the instruction.
__device__ __forceinline__ void put(u64* p, u64 v, bool near) {
  if (near) asm volatile("global_store_dwordx2 %0, %1, off sc0" : : "v"(p), "v"(v));
  else __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 get(const u64* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The value, opaque to the optimiser from here on: what is computed from it
// inside the iteration is computed there, and does not occupy registers for
// the whole solve as a loop invariant.
template <typename I>
__device__ __forceinline__ I fresh_v(I v) {
  asm volatile("" : "+v"(v));
  return v;
}
template <typename I>
__device__ __forceinline__ I fresh_s(I v) {
  asm volatile("" : "+s"(v));
  return v;
}
// element t of an array, by a 32-bit byte offset (the plan checks the size)
template <typename T>
__device__ __forceinline__ T& at(T* q, int t) {
  return *(T*)((char*)q + (unsigned)t * (unsigned)sizeof(T));
}
template <typename T>
__device__ __forceinline__ const T& at(const T* q, int t) {
  return *(const T*)((const char*)q + (unsigned)t * (unsigned)sizeof(T));
}
template <typename T>
using ConstPtr = const T __attribute__((address_space(4)))*;   // scalar loads

// The GLL derivative matrix is centro-antisymmetric, D(P-1-i, P-1-j) = -D(i, j),
// so its products split into halves (even-odd decomposition; Solomonoff 1992):
// with A_b = sum_k E(b,k) (u_k + u_k'), C_b = sum_k O(b,k) (u_k - u_k') and
// k' = P-1-k, (D u)_b = A_b + C_b and (D u)_b' = C_b - A_b, and the transpose
// takes the same tables. 2 (P/2)^2 multiply-adds instead of P^2, and at P = 8
// 32 coefficients instead of 64, which scalar registers can hold per product.
// H pairs; an odd P has a middle node m = H: column m of E, row m of O.
// Layout: E rows b < H of HE entries, then O rows b < HE of H entries.
template <typename T, int P>
struct EoTable {
  static constexpr int H = P / 2, HE = (P + 1) / 2, N = 2 * H * HE;
  T v[N];
};
template <typename T, int P>
constexpr EoTable<T, P> eo_table() {
  using E = EoTable<T, P>;
  EoTable<T, P> t{};
  for (int b = 0; b < E::HE; ++b)
    for (int k = 0; k < E::HE; ++k) {
      const double d = gll_d<P>(b + P * k), e = gll_d<P>(b + P * (P - 1 - k));
      const bool mid = b == P - 1 - b || k == P - 1 - k;
      if (b < E::H) t.v[b * E::HE + k] = T(mid ? d : 0.5 * (d + e));
      if (k < E::H) t.v[E::H * E::HE + b * E::H + k] = T(mid ? d : 0.5 * (d - e));
    }
  return t;
}

template <typename T, int P>
__device__ const EoTable<T, P> kEo = eo_table<T, P>();
// both halves of the table fit the scalar registers together
template <typename T, int P>
constexpr bool kEoWhole = EoTable<T, P>::N * sizeof(T) <= 256;
// The table's rows (E's, then O's) in order, as pointers for scalar loads. Where the
// table does not fit the scalar registers, a chunk of rows can load only once the
// one before it is begun (its pointer depends on the last value before that), so
// that two chunks at most are live; left to the compiler the loads come first and
// more of them are spilled to vector lanes and back. (FP64 still spills 22 scalars at P = 8, 84
// at P = 10, 282 at P = 12 and 430 at P = 15, FP32 27 to 137; at P = 12 the kernel holds 820
// reads of a lane and 290 writes, part of what an iteration costs.) Us per iteration, halves of the table loaded
// as the compiler likes / chunks of 128 bytes: FP64, 56x56 elements, P = 10 8.7 / 8.3,
// P = 12 11.1 / 10.4, P = 14 13.3 / 12.7; FP32 P = 14 10.3 / 9.0, P = 15 12.0 / 10.4. FP32
// at P = 16: 9.8 / 10.2, and 9.5 for the table in one piece.
template <typename T, int P>
struct EoRows {
  static constexpr int H = P / 2, HE = (P + 1) / 2;
  static constexpr int C = kEoWhole<T, P> || (sizeof(T) == 4 && P == 16)
                               ? 2 * HE : 128 / (int)(sizeof(T) * HE);
  static constexpr int off(int r) { return r < H ? r * HE : H * HE + (r - H) * H; }
  ConstPtr<T> cur, nxt;
  __device__ __forceinline__ EoRows(ConstPtr<T> E) : cur(E), nxt(E) {}
  __device__ __forceinline__ ConstPtr<T> at(int r, const T& done) {
    if (r % C == 0) {
      cur = nxt;
      if (C < 2 * HE) {
        u64 o = (u64)cur + sizeof(T) * (off(r + C) - off(r));
        if (r > 0) asm volatile("" : "+s"(o) : "v"(done));
        else asm volatile("" : "+s"(o));
        nxt = (ConstPtr<T>)o;
      }
    }
    return cur + (off(r) - off(r - r % C));
  }
};

// out1 = D u1 and out2 = D u2: two products share the coefficients' loads
template <typename T, int P>
__device__ __forceinline__ void eo_fwd2(const T (&u1)[P], T (&o1)[P], const T (&u2)[P], T (&o2)[P],
                                        ConstPtr<T> E) {
  constexpr int H = P / 2, HE = (P + 1) / 2;
  EoRows<T, P> rows(E);
  T s1[HE], f1[H], s2[HE], f2[H];
#pragma unroll
  for (int k = 0; k < H; ++k) {
    s1[k] = u1[k] + u1[P - 1 - k];
    f1[k] = u1[k] - u1[P - 1 - k];
    s2[k] = u2[k] + u2[P - 1 - k];
    f2[k] = u2[k] - u2[P - 1 - k];
  }
  if constexpr (P % 2) {
    s1[H] = u1[H];
    s2[H] = u2[H];
  }
  T A1[H], A2[H];
#pragma unroll
  for (int b = 0; b < H; ++b) {
    ConstPtr<T> R = rows.at(b, A2[b > 0 ? b - 1 : 0]);
    A1[b] = R[0] * s1[0];
    A2[b] = R[0] * s2[0];
#pragma unroll
    for (int k = 1; k < HE; ++k) {
      A1[b] += R[k] * s1[k];
      A2[b] += R[k] * s2[k];
    }
  }
  T last = A2[H - 1];
#pragma unroll
  for (int b = 0; b < HE; ++b) {
    ConstPtr<T> R = rows.at(H + b, last);
    T c1 = R[0] * f1[0], c2 = R[0] * f2[0];
#pragma unroll
    for (int k = 1; k < H; ++k) {
      c1 += R[k] * f1[k];
      c2 += R[k] * f2[k];
    }
    last = c2;
    if (b < H) {
      o1[b] = c1 + A1[b];
      o1[P - 1 - b] = c1 - A1[b];
      o2[b] = c2 + A2[b];
      o2[P - 1 - b] = c2 - A2[b];
    } else {
      o1[b] = c1;
      o2[b] = c2;
    }
  }
}

// o1 = D' u1, o2 = D' u2
template <typename T, int P>
__device__ __forceinline__ void eo_tr2(const T (&u1)[P], T (&o1)[P], const T (&u2)[P], T (&o2)[P],
                                       ConstPtr<T> E) {
  constexpr int H = P / 2, HE = (P + 1) / 2;
  EoRows<T, P> rows(E);
  T s1[HE], f1[H], s2[HE], f2[H];
#pragma unroll
  for (int k = 0; k < H; ++k) {
    s1[k] = u1[k] + u1[P - 1 - k];
    f1[k] = u1[k] - u1[P - 1 - k];
    s2[k] = u2[k] + u2[P - 1 - k];
    f2[k] = u2[k] - u2[P - 1 - k];
  }
  if constexpr (P % 2) {
    s1[H] = u1[H];
    s2[H] = u2[H];
  }
  T A1[HE], A2[HE];
#pragma unroll
  for (int k = 0; k < H; ++k) {
    ConstPtr<T> R = rows.at(k, A2[HE - 1]);
#pragma unroll
    for (int b = 0; b < HE; ++b) {
      A1[b] = k == 0 ? R[b] * f1[0] : A1[b] + R[b] * f1[k];
      A2[b] = k == 0 ? R[b] * f2[0] : A2[b] + R[b] * f2[k];
    }
  }
  T C1[H], C2[H];
#pragma unroll
  for (int k = 0; k < HE; ++k) {
    ConstPtr<T> R = rows.at(H + k, k == 0 ? A2[HE - 1] : C2[H - 1]);
#pragma unroll
    for (int b = 0; b < H; ++b) {
      C1[b] = k == 0 ? R[b] * s1[0] : C1[b] + R[b] * s1[k];
      C2[b] = k == 0 ? R[b] * s2[0] : C2[b] + R[b] * s2[k];
    }
  }
#pragma unroll
  for (int b = 0; b < H; ++b) {
    o1[b] = A1[b] + C1[b];
    o1[P - 1 - b] = A1[b] - C1[b];
    o2[b] = A2[b] + C2[b];
    o2[P - 1 - b] = A2[b] - C2[b];
  }
  if constexpr (P % 2) {
    o1[H] = A1[H];
    o2[H] = A2[H];
  }
}

// lanes of one wave exchange through LDS: its accesses stay in order
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// A field value on the wire: one word (FP32) or two (FP64)
template <typename T>
struct Wire {
  static constexpr int N = sizeof(T) / 4;
  u64 w[N];
  __device__ __forceinline__ void load(const u64* p, long plane) {
#pragma unroll
    for (int q = 0; q < N; ++q) w[q] = get(p + q * plane);
  }
  __device__ __forceinline__ bool ok(unsigned tag) const {
    bool o = true;
#pragma unroll
    for (int q = 0; q < N; ++q) o = o && (unsigned)(w[q] >> 32) == tag;
    return o;
  }
  __device__ __forceinline__ T value() const {
    if constexpr (N == 1) return __uint_as_float((unsigned)w[0]);
    else return __longlong_as_double((long long)((w[0] & 0xffffffffull) | (w[1] << 32)));
  }
};
template <typename T>
__device__ __forceinline__ void post(u64* p, long plane, unsigned tag, T v, bool near) {
  const u64 t = (u64)tag << 32;
  if constexpr (sizeof(T) == 4) {
    put(p, t | __float_as_uint(v), near);
  } else {
    const u64 b = (u64)__double_as_longlong(v);
    put(p, t | (b & 0xffffffffull), near);
    put(p + plane, t | (b >> 32), near);
  }
}

// Sum / maximum over the wave, uniform: within rows of 16 lanes by DPP, the
// four rows through scalar registers (a shuffle butterfly goes through LDS and
// was 0.3 us, four of them on an iteration's critical path). A fixed order.
template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double lane_of(double v, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                          __builtin_amdgcn_readlane(__double2loint(v), l));
}
__device__ __forceinline__ double uniform(double v) {   // a value equal in all lanes
  return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                          __builtin_amdgcn_readfirstlane(__double2loint(v)));
}
constexpr int kXor1 = 0xB1, kXor2 = 0x4E, kHalfMirror = 0x141, kMirror = 0x140;
__device__ __forceinline__ double sum_wave(double v) {
  v += dpp<kXor1>(v);
  v += dpp<kXor2>(v);
  v += dpp<kHalfMirror>(v);
  v += dpp<kMirror>(v);
  return (lane_of(v, 0) + lane_of(v, 16)) + (lane_of(v, 32) + lane_of(v, 48));
}
// the same over the first eight lanes (a workgroup's waves)
__device__ __forceinline__ double sum_first8(double v) {
  v += dpp<kXor1>(v);
  v += dpp<kXor2>(v);
  v += dpp<kHalfMirror>(v);
  return uniform(v);
}
__device__ __forceinline__ double max_first8(double v) {
  v = fmax(v, dpp<kXor1>(v));
  v = fmax(v, dpp<kXor2>(v));
  v = fmax(v, dpp<kHalfMirror>(v));
  return uniform(v);
}
// (drops NaN: the caller restores it from the sum, which is NaN with any r)
__device__ __forceinline__ double max_wave(double v) {
  v = fmax(v, dpp<kXor1>(v));
  v = fmax(v, dpp<kXor2>(v));
  v = fmax(v, dpp<kHalfMirror>(v));
  v = fmax(v, dpp<kMirror>(v));
  return fmax(fmax(lane_of(v, 0), lane_of(v, 16)), fmax(lane_of(v, 32), lane_of(v, 48)));
}

// All-to-all reduction by wave 0: v[0] summed and (NV = 2) v[1] the maximum. The
// doubles travel in NV + 1 words of 48 bits and a 16-bit tag (every workgroup
// clears its lines before the rendezvous, and a launch uses fewer than 2^16 tags).
//
// kFlat: every workgroup reads every line. kNear: the same with all workgroups on
// one XCD (the launch has eight times as many blocks and those of the other XCDs
// leave at once), so that lines and edges stay in its L2. kTwo: workgroups sum
// their XCD's lines, then the XCDs' sums from one line each, written by the group's
// first workgroup. The dispatcher places blocks round the XCDs in turn; each
// workgroup reports where it runs, and if a group is not on one XCD after all, all
// take kFlat. One exchange of one / two values, us, by workgroups: 32 kFlat 1.5 / 1.9,
// kNear 0.8 / 0.9; 128 kFlat 1.8 / 2.3, kTwo 1.9 / 2.2; 256 kFlat 2.4 / 3.3, kTwo 1.9 / 2.3.
enum : int { kFlat, kNear, kTwo, kTwoFlat };   // the last: kTwo's lines read as kFlat's
__device__ __forceinline__ bool stays(int mode) { return mode == kNear || mode == kTwo; }
constexpr u64 kM48 = 0xffffffffffffull;
// the line of workgroup wg. kTwo: a group's lines side by side, none shares a 128-byte
// line of an L2 with another group's. (kFlat in that order: 0.4 us an exchange slower.)
__device__ __forceinline__ int line_of(int wg, int mode) {
  return mode >= kTwo ? (wg & (kGroups - 1)) * kGroupWg + wg / kGroups : wg;
}
template <int NV>
__device__ __forceinline__ void exch_post(u64* line, int lane, unsigned tag, const double* v,
                                          bool near) {
  if (lane <= NV) {
    const u64 b0 = (u64)__double_as_longlong(v[0]), b1 = (u64)__double_as_longlong(v[NV - 1]);
    const u64 w = lane == NV ? (b0 >> 48) | ((b1 >> 48) << 16) : (lane == 0 ? b0 : b1) & kM48;
    put(line + lane, w | ((u64)tag << 48), near);
  }
}
// the reduction of n lines (NB = 1: side by side; else the lines of the first n
// workgroups), every workgroup in the same order; false when a poll gave up
template <int NV, int NB>
__device__ __forceinline__ bool exch_read(const u64* lines, int n, int mode, int lane,
                                          unsigned tag, double* v) {
  constexpr int W = NV + 1;
  lane = fresh_v(lane);
  u64 a[NB][W];
  int c = 0;
  bool ok;
  for (;;) {
    ok = true;
#pragma unroll
    for (int j = 0; j < NB; ++j)
      if (64 * j < n) {
        const int i = min(lane + 64 * j, n - 1);
        const u64* s = lines + (NB == 1 ? i : line_of(i, mode)) * kSlotWords;
#pragma unroll
        for (int q = 0; q < W; ++q) a[j][q] = get(s + q);
      }
#pragma unroll
    for (int j = 0; j < NB; ++j)
      if (64 * j < n) {
#pragma unroll
        for (int q = 0; q < W; ++q) ok = ok && (unsigned)(a[j][q] >> 48) == (tag & 0xffffu);
      }
    if (__all(ok) || ++c >= kResPolls) break;
    __builtin_amdgcn_s_sleep(1);
  }
  double s0 = 0.0, m = 0.0;
#pragma unroll
  for (int j = 0; j < NB; ++j)
    if (lane + 64 * j < n) {
      auto val = [&](int q) {
        return __longlong_as_double(
            (long long)((a[j][q] & kM48) | (((a[j][NV] >> (16 * q)) & 0xffffull) << 48)));
      };
      s0 += val(0);
      if constexpr (NV == 2) m = fmax(m, val(1));
    }
  v[0] = sum_wave(s0);
  if constexpr (NV == 2) v[1] = max_wave(m);
  return __all(ok);
}
// slots: the kMaxWg lines of this exchange; sums: its kGroups lines
template <int NV>
__device__ __forceinline__ bool exch_wait(const u64* slots, u64* sums, int nwg, int wg, int mode,
                                          int lane, unsigned tag, double* v) {
  if (mode != kTwo) return exch_read<NV, kMaxWg / 64>(slots, nwg, mode, lane, tag, v);
  const int g = wg & (kGroups - 1);
  bool ok = exch_read<NV, 1>(slots + g * kGroupWg * kSlotWords, (nwg - g + kGroups - 1) / kGroups,
                             mode, lane, tag, v);
  if (wg < kGroups) exch_post<NV>(sums + g * kSlotWords, lane, tag, v, false);
  ok = exch_read<NV, 1>(sums, kGroups, mode, lane, tag, v) && ok;
  return ok;
}

// The rendezvous, in two parts with the loads of the fields between them. Every
// thread of the workgroup calls both. arrive: clears this workgroup's lines and
// reports it. decide: -1 when the launch is called off, else the form of exchange
// (every workgroup's the same).
__device__ inline void arrive(ResCtl* c, u64* slots, unsigned tag0, int nwg, int wg, int near) {
  if (threadIdx.x == 0) {
    u64* const sums = slots + 2 * kMaxWg * kSlotWords;
    const int line = line_of(wg, near), g = near == kTwo ? wg & (kGroups - 1) : 0;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      put(slots + line * kSlotWords + q, (u64)tag0 << 48, false);
      put(slots + (kMaxWg + line) * kSlotWords + q, (u64)tag0 << 48, false);
      if (near == kTwo && wg < kGroups) {
        put(sums + wg * kSlotWords + q, (u64)tag0 << 48, false);
        put(sums + (kGroups + wg) * kSlotWords + q, (u64)tag0 << 48, false);
      }
    }
    if (near != kFlat) {
      unsigned xcc;
      asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
      __hip_atomic_fetch_or(&c->xcds[g], 1u << (xcc & 31), __ATOMIC_RELAXED,
                            __HIP_MEMORY_SCOPE_AGENT);
    }
    // The cleared lines have reached memory before the arrival is counted. (They are
    // agent-scope stores, so their completion is all that is needed; a release would
    // write back the whole L2, 3 us and more after kernels that filled it.)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (__hip_atomic_fetch_add(&c->arrived, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
        nwg - 1)
      atomicCAS(&c->decision, 0, 1);
  }
}
__device__ inline int decide(ResCtl* c, int near, int* go) {
  if (threadIdx.x == 0) {
    int dcs, n = 0;
    while ((dcs = __hip_atomic_load(&c->decision, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == 0)
      if (++n > kResWait) atomicCAS(&c->decision, 0, 2);
    // (what is exchanged is read by agent-scope loads: nothing to invalidate)
    int mode = dcs == 1 ? near : -1;
    if (mode > kFlat) {
      unsigned x[kGroups], two = 0;   // (all loads in flight together)
#pragma unroll
      for (int q = 0; q < kGroups; ++q)
        x[q] = __hip_atomic_load(&c->xcds[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int q = 0; q < kGroups; ++q) two |= x[q] & (x[q] - 1);
      if (two) mode = near == kTwo ? kTwoFlat : kFlat;
    }
    *go = mode;
  }
  __syncthreads();
  return __builtin_amdgcn_readfirstlane(*go);
}
// The solve's state for the host, and the next launch's control words cleared: a
// copy and a fill less per solve (some 15 us with the gaps before and after them).
__device__ inline void report(PcgHost* host, ResCtl* next, const PcgState* st, int tid) {
  if (host && tid == 0) {
    host->state = *st;
    host->ctl.decision = 1;
  }
  if (next && tid < (int)(sizeof(ResCtl) / sizeof(int))) reinterpret_cast<int*>(next)[tid] = 0;
}

// Element edges of a tile in LDS, with one line from each neighbouring tile:
// y-lines 0 (below), 1 + 2 hh and 2 + 2 hh (bottom and top of element row hh), one
// above the last; x-lines the same over the elements. The halo y-lines carry one
// extra row at both ends for the corners. Element [0, P) of the array stays
// zero: threads without a partner read it, so that no load sits under a branch.
template <typename T, int P>
struct Edges {
  static constexpr int NE = kWaves<T, P> * kEpw<P>;
  static constexpr int mx(int a, int b) { return a > b ? a : b; }
  // the sum over both kinds is largest for a 1 x NE or NE x 1 tile
  static constexpr int NY = mx(4 * (NE * P + 2), (2 * NE + 2) * (P + 2));
  static constexpr int NX = mx(4 * (NE * P + 1), (2 * NE + 2) * (P + 1));
  T v[P + NY + NX];
};

// per-thread facts, packed so that tests are recomputed and no lane mask
// stays in scalar registers across the iteration
enum : int {
  kAct = 1, kCol = 2, kXShare = 4, kXSide = 8, kY0Share = 16, kY1Share = 32, kOnI = 64, kOn0 = 128,
  kOn1 = 256, kY0In = 512, kY1In = 1024   // the y-partner lies in this tile
};

// NEAR: the launch may exchange in another form than kFlat (a kernel of its own: the
// tests on the form cost kFlat 0.15 us an iteration)
template <typename T, int P, bool NEAR>
__global__ void __launch_bounds__((kWaves<T, P> * 64))
    __attribute__((amdgpu_waves_per_eu((kWaves<T, P> / 4), (kWaves<T, P> / 4))))
    k_pcg_res(const ResP<T> prm) {
  constexpr int NW = kWaves<T, P>, EPW = kEpw<P>;
  constexpr int RS = 65;
  __shared__ T s0_[NW][P * RS];
  __shared__ Edges<T, P> edge_;
  __shared__ T xl_[kXLds<T, P> ? P * NW * 64 : 1];
  __shared__ double red[2][NW], bc[3];
  __shared__ int go, lost_any;
  // parameters are read from the kernel's arguments where they are used
  using PrmPtr = ConstPtr<ResP<T>>;
  const u64 karg = (u64)__builtin_amdgcn_kernarg_segment_ptr();
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  if (NEAR && prm.near == kNear && blockIdx.x % kGroups) return;
  const int wg = NEAR && prm.near == kNear ? blockIdx.x / kGroups : blockIdx.x;
  T* const edge = edge_.v;

  if (tid == 0) lost_any = 0;
  if (tid < P) edge[tid] = T(0);
  if (prm.nwg > 1)
    arrive(prm.ctl, prm.slots, prm.tag0, prm.nwg, wg, NEAR ? prm.near : (int)kFlat);

  // this thread's element (row hh, column e of the tile) and row a
  const int es = lane / P;
  const int a = lane - es * P;
  const int eo = wv * EPW + es;
  const int tx = wg % prm.ntx, ty = wg / prm.ntx;
  const int hh = eo / prm.TX, e = eo - hh * prm.TX;
  const int ex = tx * prm.TX + e, ey = ty * prm.RY + hh;
  T* const s0 = s0_[wv];
  const int L = P * prm.Ex;
  const int base = ex * P + a + L * (ey * P);   // fewer than 2^31 nodes
  // lengths of the lines (x-lines odd: a wave's lanes read one entry of many
  // lines) and the places of this row's own ones
  const int LY = prm.TX * P + 2, LX = (prm.RY * P) | 1;
  const int ybase = P, xbase = P + Edges<T, P>::NY;
  const int yl = ybase + (1 + 2 * hh) * LY + e * P + a + 1;
  const int xl = xbase + (1 + 2 * e + (a == 0 ? 0 : 1)) * LX + hh * P;
  // the tile's own elements (the last tiles may be narrower)
  const int nex = min(prm.TX, prm.Ex - tx * prm.TX), ney = min(prm.RY, prm.Ey - ty * prm.RY);
  int flags = 0;
  if (es < EPW) flags |= kCol;
  if (es < EPW && e < nex && hh < ney) {
    flags |= kAct;
    const int i = ex * P + a;
    if (a == 0 ? (ex > 0 || prm.per_x) : a == P - 1 ? (ex < prm.Ex - 1 || prm.per_x) : false)
      flags |= kXShare;
    if (a == P - 1) flags |= kXSide;
    flags |= (hh > 0 ? kY0In : 0) | (hh < ney - 1 ? kY1In : 0);
    if (ey > 0 || prm.per_y) flags |= kY0Share;
    if (ey < prm.Ey - 1 || prm.per_y) flags |= kY1Share;
    const bool on = !((prm.bc & SEM_BC_XMIN) && i == 0) && !((prm.bc & SEM_BC_XMAX) && i == L - 1);
    if (on) flags |= kOnI;
    if (on && !((prm.bc & SEM_BC_YMIN) && ey == 0)) flags |= kOn0;
    if (on && !((prm.bc & SEM_BC_YMAX) && ey == prm.Ey - 1)) flags |= kOn1;
  }

  T r[P], p[P], x_[kXLds<T, P> ? 1 : P], d[P], g11[P], g12[P], g22[P], bm[P];
  auto x = [&](int b) -> T& {
    if constexpr (kXLds<T, P>) return xl_[b * (NW * 64) + tid];
    else return x_[b];
  };
  {
    // loads without branches (threads without a row read node 0 and drop it),
    // so that all of them are in flight together
    const bool act = flags & kAct, hasd = prm.d != nullptr, mass = prm.has_mass != 0;
    const int t0 = act ? base : 0, st = act ? L : 0;
    const T* const dp = hasd ? prm.d : prm.G11;
    const T* const bp = mass ? prm.B : prm.G11;
    const T* const rp = prm.b ? prm.b : prm.r;
#pragma unroll
    for (int b = 0; b < P; ++b) {
      const int t = t0 + st * b;
      g11[b] = at(prm.G11, t);
      g12[b] = at(prm.G12, t);
      g22[b] = at(prm.G22, t);
      bm[b] = at(bp, t);
      d[b] = at(dp, t);
      r[b] = at(rp, t);
    }
#pragma unroll
    for (int b = 0; b < P; ++b) {
      if (!act) g11[b] = g12[b] = g22[b] = r[b] = T(0);
      if (!act || !mass) bm[b] = T(0);
      if (!act || !hasd) d[b] = T(1);
      p[b] = T(0);
      x(b) = T(0);
    }
    if (!prm.b && act) {
#pragma unroll
      for (int b = 0; b < P; ++b) x(b) = at(prm.x, t0 + st * b);
    }
    if (prm.k_start > 1 && act) {
#pragma unroll
      for (int b = 0; b < P; ++b) p[b] = at(prm.p, t0 + st * b);
    }
  }

  // (the form of exchange stays in LDS: scalar registers are scarce below)
  if (prm.nwg > 1 && decide(prm.ctl, NEAR ? prm.near : (int)kFlat, &go) < 0) return;

  // <r, z>_mult and norm(r, Inf) of the current r, identical in every workgroup
  auto reduce_r = [&](unsigned tag, double* t, double* res) {
    // (read ahead of their use)
    const PrmPtr c0 = NEAR || kFresh<T, P> ? (PrmPtr)fresh_s(karg) : (PrmPtr)karg;
    const int nwg = c0->nwg, mode_ = NEAR ? go : (int)kFlat;
    u64* const s = c0->slots + kMaxWg * kSlotWords;
    const int f = fresh_v(flags);
    const double mx = f & kXShare ? 0.5 : 1.0;
    const double m0 = f & kY0Share ? 0.5 * mx : mx, m1 = f & kY1Share ? 0.5 * mx : mx;
    double rho = 0.0, m = 0.0;
#pragma unroll
    for (int b = 0; b < P; ++b) {
      const T z = d[b] * r[b];
      rho += (double)r[b] * (double)z * (b == 0 ? m0 : b == P - 1 ? m1 : mx);
      m = fmax(m, fabs((double)r[b]));
    }
    rho = sum_wave(rho);
    m = max_wave(m);
    if (lane == 0) {
      red[0][wv] = rho;
      red[1][wv] = m;
    }
    __syncthreads();
    if (wv == 0) {
      const bool in = lane < (int)(blockDim.x >> 6);
      double v[2] = {sum_first8(in ? red[0][lane & (NW - 1)] : 0.0),
                     max_first8(in ? red[1][lane & (NW - 1)] : 0.0)};
      bool ok = true;
      if (nwg > 1) {
        const int mode = NEAR ? __builtin_amdgcn_readfirstlane(mode_) : mode_;
        exch_post<2>(s + line_of(wg, mode) * kSlotWords, lane, tag, v, stays(mode));
        ok = exch_wait<2>(s, s + (kMaxWg + kGroups) * kSlotWords, nwg, wg, mode, lane, tag, v);
      }
      if (lane == 0) {
        bc[1] = v[0];
        bc[2] = v[0] != v[0] ? v[0] : v[1];   // a NaN in r makes <r, z> NaN
        if (!ok) lost_any = 1;
      }
    }
    __syncthreads();
    *t = uniform(bc[1]);
    *res = uniform(bc[2]);
  };

  unsigned tag = prm.tag0 + 1;
  double t, res, t_prev = 1.0;
  reduce_r(tag, &t, &res);
  const int k_start = prm.k_start, maxiter = prm.maxiter, max_its = prm.max_its;
  const T nu = prm.nu, kc = prm.k;
  int k = k_start;
  double tol = prm.tol;
  if (tol < 0.0) tol = k == 1 ? -tol * res : uniform(prm.state->tol_eff);
  if (k > 1) t_prev = uniform(prm.state->t[(k - 1) & 1]);
  bool done = false;
  for (;;) {
    done = !(res > tol) || k - 1 == maxiter;
    if (done || k - k_start == max_its || __builtin_amdgcn_readfirstlane(lost_any)) break;
    ++tag;
    const T beta = k == 1 ? T(0) : T(uniform(t / t_prev));
    // p = z + beta p; the thread's row us = p Ds'; its column a of the element,
    // in place, ur = Dr p
    T h[P];
    double dot = 0.0;
    {
#pragma unroll
      for (int b = 0; b < P; ++b) {
        p[b] = d[b] * r[b] + beta * p[b];
        s0[b * RS + lane] = p[b];
      }
      wave_fence();
      const u64 tab = (u64)&kEo<T, P>;
      ConstPtr<T> E = (ConstPtr<T>)fresh_s(tab);
      // lanes past the last whole element read column 0 of the first and write nothing
      const int cbase = fresh_v(flags & kCol ? a * RS + es * P : 0);
      {
        T us[P];
        {
          T c[P], o[P];
#pragma unroll
          for (int q = 0; q < P; ++q) c[q] = s0[cbase + q];
          eo_fwd2<T, P>(p, us, c, o, E);
          wave_fence();
          if (64 % P == 0 || (flags & kCol)) {
#pragma unroll
            for (int q = 0; q < P; ++q) s0[cbase + q] = o[q];
          }
        }
        wave_fence();
        T wsv[P];
#pragma unroll
        for (int b = 0; b < P; ++b) {
          const T ur = s0[b * RS + lane];
          wsv[b] = g12[b] * ur + g22[b] * us[b];
          s0[b * RS + lane] = g11[b] * ur + g12[b] * us[b];
        }
        wave_fence();
        if constexpr (!kEoWhole<T, P>) E = (ConstPtr<T>)fresh_s(tab);
        T c[P], o[P];
#pragma unroll
        for (int q = 0; q < P; ++q) c[q] = s0[cbase + q];
        eo_tr2<T, P>(wsv, h, c, o, E);   // ws Ds and Dr' wr
        wave_fence();
        if (64 % P == 0 || (flags & kCol)) {
#pragma unroll
          for (int q = 0; q < P; ++q) s0[cbase + q] = o[q];
        }
      }
      wave_fence();
      // H = nu (Dr' wr + ws Ds) + k B p, and its share of <p, A p>: p is
      // continuous and masked, so sum(p .* H) over the copies needs no
      // assembled value
      const PrmPtr c4 = (PrmPtr)karg;
      if (c4->nu_f == nullptr && c4->k_f == nullptr) {
#pragma unroll
        for (int b = 0; b < P; ++b) {
          const T au = s0[b * RS + lane] + h[b];
          h[b] = nu * au + kc * (bm[b] * p[b]);
          dot += (double)p[b] * (double)h[b];
        }
      } else {
        const int bi = fresh_v(flags & kAct ? base : 0), st = flags & kAct ? L : 0;
        const T* const nf = c4->nu_f ? c4->nu_f : c4->G11;
        const T* const kf = c4->k_f ? c4->k_f : c4->G11;
        const bool hn = c4->nu_f != nullptr, hk = c4->k_f != nullptr;
#pragma unroll
        for (int b = 0; b < P; ++b) {
          const T fn = at(nf, bi + st * b), fk = at(kf, bi + st * b);
          const T au = s0[b * RS + lane] + h[b];
          h[b] = (hn ? fn : nu) * au + (hk ? fk : kc) * (bm[b] * p[b]);
          dot += (double)p[b] * (double)h[b];
        }
      }
    }
    // raw edge values to the tile's lines
    const PrmPtr c2 = (PrmPtr)fresh_s(karg);
    const PrmPtr c1 = NEAR || kFresh<T, P> ? c2 : (PrmPtr)karg;
    u64* const slots = c1->slots;
    const int nwg = c1->nwg, mode_ = NEAR ? go : (int)kFlat;   // (read ahead of their use)
    {
      const int f = fresh_v(flags);
      if (f & kAct) {
        edge[yl] = h[0];
        edge[yl + LY] = h[P - 1];
      }
      if (f & kXShare) {
#pragma unroll
        for (int b = 0; b < P; ++b) edge[xl + b] = h[b];
      }
    }
    dot = sum_wave(dot);
    if (lane == 0) red[0][wv] = dot;
    __syncthreads();
    // wave 0 exchanges the sum, the others the edges (a single wave does both)
    const int mode = NEAR ? __builtin_amdgcn_readfirstlane(mode_) : mode_;
    const bool alone = blockDim.x == 64;
    double pap[1];
    if (wv == 0) {
      pap[0] = sum_first8(lane < (int)(blockDim.x >> 6) ? red[0][lane & (NW - 1)] : 0.0);
      if (nwg > 1)
        exch_post<1>(slots + line_of(wg, mode) * kSlotWords, lane, tag, pap, stays(mode));
    }
    if (wv != 0 || alone) {
      const int TX = c2->TX, RY = c2->RY, ntx = c2->ntx, nty = c2->nty;
      const int Ex = c2->Ex, Ey = c2->Ey, per_x = c2->per_x, per_y = c2->per_y;
      const int mtx = wg % ntx, mty = wg / ntx;
      const int nxt = min(TX, Ex - mtx * TX), nyt = min(RY, Ey - mty * RY);
      const int NC = P * Ey;
      const int yplane = 2 * nty * L, xplane = 2 * ntx * NC;
      const int q0 = alone ? lane : tid - 64, qs = alone ? 64 : (int)blockDim.x - 64;
      // out: bottom and top y-line, left and right x-line
      if (nwg > 1) {
        const bool near = mode == kNear;
        const int wy = nxt * P, wx = nyt * P;
        for (int q = fresh_v(q0); q < 2 * (wy + wx); q += qs) {
          int m = q;
          const bool isy = m < 2 * wy;
          if (!isy) m -= 2 * wy;
          const int w = isy ? wy : wx;
          const int up = m >= w ? 1 : 0;
          m -= up * w;
          if (isy ? nty == 1 : ntx == 1) continue;
          if (isy) post<T>(c2->ymail + ((2 * mty + up) * L + mtx * TX * P + m), yplane, tag,
                           edge[ybase + (up ? 2 * nyt : 1) * LY + m + 1], near);
          else post<T>(c2->xmail + ((2 * mtx + up) * NC + mty * RY * P + m), xplane, tag,
                       edge[xbase + (up ? 2 * nxt : 1) * LX + m], near);
        }
      }
      // in: y-lines below and above with their end rows, then x-lines; round a
      // periodic direction of one tile, the tile's own lines
      const int wy = nxt * P + 2, wx = nyt * P;
      for (int q = fresh_v(q0); q < 2 * (wy + wx); q += qs) {
        int m = q;
        const bool isy = m < 2 * wy;
        if (!isy) m -= 2 * wy;
        const int w = isy ? wy : wx;
        const int up = m >= w ? 1 : 0;   // above / right
        m -= up * w;
        // the line's tile, and this entry's row (y) or column (x) of the mesh
        int sty = mty, stx = mtx, pos;
        bool have;
        if (isy) {
          sty = up ? mty + 1 : mty - 1;
          have = per_y || (sty >= 0 && sty < nty);
          sty = sty < 0 ? nty - 1 : sty >= nty ? 0 : sty;
          pos = mtx * TX * P + m - 1;
          have = have && (per_x || (pos >= 0 && pos < L));
          pos = pos < 0 ? L - 1 : pos >= L ? 0 : pos;
        } else {
          stx = up ? mtx + 1 : mtx - 1;
          have = per_x || (stx >= 0 && stx < ntx);
          stx = stx < 0 ? ntx - 1 : stx >= ntx ? 0 : stx;
          pos = mty * RY * P + m;
        }
        if (!have) continue;
        const int own = pos - mtx * TX * P;   // y-line: its row within this tile
        const bool inside = own >= 0 && own < nxt * P;
        // an end row of a y-line that wraps within this tile: the x-line of the
        // tile beside it has it, at the wrapped column
        const bool end = isy && nty == 1 && !inside;
        const bool ym = isy && nty > 1, xm = (!isy || end) && ntx > 1;
        T v;
        if (ym || xm) {
          const int side = end ? (m == 0 ? 1 : 0) : 1 - up;
          if (end) stx = m == 0 ? (mtx == 0 ? ntx - 1 : mtx - 1) : (mtx + 1 == ntx ? 0 : mtx + 1);
          const u64* src = ym ? c2->ymail + ((2 * sty + side) * L + pos)
                              : c2->xmail + ((2 * stx + side) * NC + (end ? (up ? 0 : NC - 1) : pos));
          const int plane = ym ? yplane : xplane;
          Wire<T> wd;
          int tries = 0;
          do wd.load(src, plane);
          while (!wd.ok(tag) && ++tries < kResPolls);
          if (!wd.ok(tag)) lost_any = 1;
          v = wd.value();
        } else {
          v = isy ? edge[ybase + (up ? 1 : 2 * nyt) * LY + own + 1]
                  : edge[xbase + (up ? 1 : 2 * nxt) * LX + m];
        }
        if (isy) edge[ybase + (up ? 2 * nyt + 1 : 0) * LY + m] = v;
        else edge[xbase + (up ? 2 * nxt + 1 : 0) * LX + m] = v;
      }
    }
    if (wv == 0) {
      bool ok = true;
      if (nwg > 1)
        ok = exch_wait<1>(slots, slots + 2 * kMaxWg * kSlotWords, nwg, wg, mode, lane, tag, pap);
      if (lane == 0) {
        bc[0] = pap[0];
        if (!ok) lost_any = 1;
      }
    }
    __syncthreads();
    // QQ': x-pairs first, then y-pairs, every copy in the order of the
    // launch-per-step path: (own + x-partner) + (y-partner + its x-partner)
    {
      const int f = fresh_v(flags);
      const bool xs = f & kXShare, ys0 = f & kY0Share, ys1 = f & kY1Share;
      const int o = f & kXSide ? 1 : -1, xo = xl + o * LX;
      const T y0 = edge[ys0 ? yl - LY : 0], y1 = edge[ys1 ? yl + 2 * LY : 0];
      const T c0 = edge[xs && ys0 ? (f & kY0In ? xo - 1 : yl - LY + o) : 0];
      const T c1 = edge[xs && ys1 ? (f & kY1In ? xo + P : yl + 2 * LY + o) : 0];
      const int xi = xs ? xo : 0;
#pragma unroll
      for (int b = 0; b < P; ++b) h[b] = h[b] + edge[xi + b];
      h[0] = (h[0] + (y0 + c0)) * (f & kOn0 ? T(1) : T(0));
      h[P - 1] = (h[P - 1] + (y1 + c1)) * (f & kOn1 ? T(1) : T(0));
#pragma unroll
      for (int b = 1; b < P - 1; ++b) h[b] = h[b] * (f & kOnI ? T(1) : T(0));
    }
    const T alpha = T(uniform(t / bc[0]));
#pragma unroll
    for (int b = 0; b < P; ++b) {
      x(b) = x(b) + alpha * p[b];
      r[b] = r[b] - alpha * h[b];
    }
    t_prev = t;
    reduce_r(tag, &t, &res);
    ++k;
  }
  const bool failed = lost_any != 0;
  if (flags & kAct) {
    const bool save = prm.keep || !done;
    const int q0 = fresh_v(base);
#pragma unroll
    for (int b = 0; b < P; ++b) {
      const int q = q0 + L * b;
      at(prm.x, q) = x(b);
      if (save) {
        at(prm.r, q) = r[b];
        at(prm.p, q) = p[b];
      }
    }
  }
  if (wg == 0) {
    PcgState* st = prm.state;
    if (tid == 0) {
      st->iters = k - 1;
      st->converged = done && res <= tol ? 1 : 0;
      st->res = res;
      if (k > k_start) st->t[(k - 1) & 1] = t_prev;
      st->alpha[0] = st->alpha[1] = 0.0;   // x is complete
      st->tol_eff = tol;
      st->done = done && !failed ? 1 : 0;
    }
    report(prm.host, prm.ctl_next, st, tid);
  }
  if (failed && tid == 0) {
    atomicExch(&prm.ctl->failed, 1);
    if (prm.host) prm.host->ctl.failed = 1;
  }
}

}  // namespace res
}  // namespace sem
