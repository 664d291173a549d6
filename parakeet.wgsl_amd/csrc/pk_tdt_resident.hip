// pk_tdt_resident.hip - greedy TDT decoding with the decoder's weights held
// in LDS (reference: src/webgpu/kernels/tdt-decoder.ts, shader :1133-2010;
// the arithmetic is the one described in pk_tdt.hip, chain for chain, so the
// results are bit-identical to it).
//
// What bounds a decode is a serial chain: every token needs two LSTM layers,
// a projector and a head, each a chain of 640 or 1280 dependent fused
// multiply-adds, with an exchange of the new vector between them. A kernel
// that streams the 15 MB of weights (30 MB in f32) through a few compute
// units per window spends nearly all of its time on that stream instead. So
// here the whole chip's LDS holds the weights once: `kMembers` workgroups
// ("members"), one per compute unit, each own the four gate columns of a few
// hidden units in both layers; some of them own projector columns too, others
// head columns. All windows of the launch share them: wave w of every member
// decodes windows [wW, wW + W), and the waves of one member never wait for
// each other.
//
// Exchange. A published value is one 64-bit word with a tag in it, written
// and read with relaxed agent-scope atomics: the tag says which step of the
// window the value belongs to, so a reader polls the words themselves, one
// memory round trip after the writer's store, and no ordering between
// different words is needed anywhere. Every vector has two slots by the
// parity of its step. A slot is written again two steps later. By then the
// writer has seen, for the step between, a word of every member that uses
// the vector, and each of them publishes that word after its last use of the
// older value: every member reads h0 and h1 and publishes the next h0; only
// projector members read the f32 h1 and only head members the projection,
// and the next step's words of both depend on them; and a member that owns
// no head column publishes its own word at every joint step, which the head
// members wait for beside their scores.
//
// Residency. Members poll, so all of them must be resident. Each counts
// itself in and waits until the count is full or a bounded time has passed;
// then it raises the abort flag and everyone leaves, as it does when a later
// poll exceeds its limit. The kernels that follow in the stream decode every
// window of an aborted launch from the start and do nothing otherwise: in f16
// tdt_team_kernel, whose small workgroups fit beside others where these do
// not, and for windows whose team gives up too (every f32 one)
// tdt_decode_kernel, one workgroup per window without any waiting. So a device
// busy with other work costs time, never a result.
//
// Measured on whole decodes of 188 frames, synthetic weights, against the
// kernels of pk_tdt.hip that ran before (the longest window has 63 tokens for
// one window, 139 for more): f16 1 window 9.37 -> 1.58 ms, 4 windows 17.96 ->
// 3.30, 16 windows 17.39 -> 5.13, 40 windows 35.9 -> 16.9; f32 1 window 23.9 ->
// 1.53, 4 windows 48.6 -> 3.30, 16 windows 48.9 -> 13.3, 24 windows 20.9. One
// window's token step (18 us) is 9 us of chains, 6 us of exchanges (1.1-2.2 us
// each, a store and a load of the memory beyond the L2s) and 1 us of cell
// updates. With four windows per wave the chains take 13 us (LDS bandwidth)
// and the exchanges 8.
#include "pk_tdt_math.h"

#pragma clang fp contract(off)

namespace pk {
namespace {

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef _Float16 half8v __attribute__((ext_vector_type(8)));

constexpr uint32_t H = kTdtHidden;
constexpr uint32_t kBlock = 256;  // one wave per SIMD: a wave's registers hold its windows' vectors

// kUnits: hidden units of a member; kGatesPerLane: gate columns of one lane
// of a gate chain; kWindows: windows of a wave. A dependent f16 fma takes 8.6
// cycles, packed or not (measured; f32 4.8), so an f16 lane takes two gates.
// The f32 weights of three units, 123 KB, are what one compute unit's LDS
// holds beside the rest.
template <uint32_t WINDOWS>
struct ShapeF16 {
  typedef ProfileF16 P;
  typedef half2v Acc;
  static constexpr uint32_t kUnits = 4, kGatesPerLane = 2, kWindows = WINDOWS, kHeadColumns = 16,
                            kProjectorColumns = 10;
};
template <uint32_t WINDOWS>
struct ShapeF32 {
  typedef ProfileF32 P;
  typedef float Acc;
  static constexpr uint32_t kUnits = 3, kGatesPerLane = 1, kWindows = WINDOWS, kHeadColumns = 9,
                            kProjectorColumns = 8;
};

template <class S>
struct Geometry {
  typedef typename S::P::X X;
  static constexpr uint32_t kMembers = (H + S::kUnits - 1) / S::kUnits;
  // lanes of one unit: (gate or gate pair) x (even, odd rows)
  static constexpr uint32_t kUnitLanes = 2 * 4 / S::kGatesPerLane;
  static constexpr uint32_t kLanes = S::kUnits * kUnitLanes;  // of one window
  // Head outputs in the order durations, tokens, blank (member 0 of the head
  // owns every duration). Workgroups [0, kHeadMembers) own head columns, the
  // last kProjectorMembers projector columns: with workgroups dealt round
  // robin to the XCDs, the readers of each vector are spread over all eight.
  static constexpr uint32_t kOutputs = kTdtBlank + 1 + 5;
  static constexpr uint32_t kHeadMembers = (kOutputs + S::kHeadColumns - 1) / S::kHeadColumns;
  static constexpr uint32_t kHeadLanes = S::kHeadColumns / S::kGatesPerLane;
  static constexpr uint32_t kProjectorMembers = H / S::kProjectorColumns;
  // LDS in 16-byte units, each four rows of a lane's columns: f16 pairs, f32
  // values, the projector's in f32 in both profiles
  static constexpr uint32_t kLayerUnits = 2 * H / 2 / 4 * kLanes;
  static constexpr uint32_t kHeadUnits = H / 4 * kHeadLanes;
  static constexpr uint32_t kProjectorUnits = H / 4 * S::kProjectorColumns;
  static constexpr uint32_t kWeightUnits =
      2 * kLayerUnits + (kHeadUnits > kProjectorUnits ? kHeadUnits : kProjectorUnits);
  // A window's vector: 640 values by row parity for a gate chain (padded
  // against bank conflicts), or 640 in order.
  static constexpr uint32_t kParityBytes = H / 2 * (uint32_t)sizeof(X) + 16;
  static constexpr uint32_t kSlotBytes = H * 4 + 32;
  static constexpr uint32_t kFixedBytes = kWeightUnits * 16 + 16;
  static_assert(kHeadMembers + kProjectorMembers <= kMembers, "a member has at most one of the two roles");
  static_assert(S::kHeadColumns >= 5 && H % S::kProjectorColumns == 0, "column split");
  static_assert(kHeadLanes <= kLanes && S::kHeadColumns % S::kGatesPerLane == 0 && S::kProjectorColumns <= kLanes && S::kWindows * kLanes <= 64, "lanes");
  static_assert(kMembers + 1 <= kTdtResidentBest, "words of a joint step");
  static_assert(2 * kParityBytes <= kSlotBytes, "a slot holds both parities");
};

__device__ __forceinline__ uint64_t xload64(const uint64_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void publish(uint64_t* p, uint32_t value, uint32_t tag) {
  __hip_atomic_store(p, (uint64_t)tag << 32 | value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Orders a wave's LDS accesses of different lanes (one wave's LDS
// operations complete in order, so only the compiler needs telling).
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ uint32_t lane_of(uint32_t v, uint32_t lane) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)lane);
}

// One 16-byte unit of weights: four rows of a pair of f16 columns or of an f32
// column, and their inputs. A row whose input is -0 is left out when SKIP is
// set (the head's rule for inputs that are zero).
template <bool SKIP>
__device__ __forceinline__ void rows(half2v& acc, const uint4& w, const half4& x) {
  const half8v v = __builtin_bit_cast(half8v, w);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const _Float16 xr = x[r];
    const half2v next = __builtin_elementwise_fma(half2v{xr, xr}, half2v{v[2 * r], v[2 * r + 1]}, acc);
    if constexpr (SKIP)
      acc = __builtin_bit_cast(uint16_t, xr) == 0x8000u ? acc : next;
    else
      acc = next;
  }
}
template <bool SKIP>
__device__ __forceinline__ void rows(float& acc, const uint4& w, const float4v& x) {
  const float4v v = __builtin_bit_cast(float4v, w);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float next = __builtin_fmaf(x[r], v[r], acc);
    if constexpr (SKIP)
      acc = __float_as_uint(x[r]) == 0x80000000u ? acc : next;
    else
      acc = next;
  }
}

template <bool C, class A, class B>
struct Select {
  typedef A Type;
};
template <class A, class B>
struct Select<false, A, B> {
  typedef B Type;
};

// A chain over ROWS rows, a batch's LDS reads issued before the multiplies of
// the batch before it. Written out in full (UNROLL) it takes 8.2 cycles a row
// in f16, the fma's own latency, and 8.0 in f32, whose LDS reads bound it; in
// a loop 9.6 and 8.8. Waves of several windows take the loop: beside their
// vectors the written-out form spills. (A batch of eight f32 units has more
// reads than the LDS wait counter's 15; only the loop hides that.)
template <int ROWS, bool SKIP, bool UNROLL, class Acc>
__device__ __forceinline__ Acc chain(Acc acc, const uint4* w, uint32_t stride, const uint4* x) {
  constexpr bool kF32 = __is_same(Acc, float);
  constexpr int N = kF32 && UNROLL ? 4 : 8;  // units of a batch
  constexpr int BATCHES = ROWS / (4 * N);
  typedef typename Select<kF32, float4v, half4>::Type T;
  uint4 wa[N], wb[N];
  T xa[N], xb[N];
  auto load_x = [&](int batch, int g, T(&xd)[N]) {
    if constexpr (kF32) {
      xd[g] = __builtin_bit_cast(T, x[batch * N + g]);
    } else if (g % 2 == 0) {
      const uint4 v = x[(batch * N + g) / 2];
      xd[g] = __builtin_bit_cast(T, make_uint2(v.x, v.y));
      xd[g + 1] = __builtin_bit_cast(T, make_uint2(v.z, v.w));
    }
  };
  auto load = [&](int batch, uint4(&wd)[N], T(&xd)[N]) {
#pragma unroll
    for (int g = 0; g < N; ++g) {
      wd[g] = w[(uint32_t)(batch * N + g) * stride];
      if constexpr (kF32 && UNROLL) load_x(batch, g, xd);
    }
    if constexpr (!(kF32 && UNROLL)) {
#pragma unroll
      for (int g = 0; g < N; ++g) load_x(batch, g, xd);
    }
  };
  auto use = [&](const uint4(&ws)[N], const T(&xs)[N]) {
#pragma unroll
    for (int g = 0; g < N; ++g) rows<SKIP>(acc, ws[g], xs[g]);
  };
  static_assert(BATCHES % 2 == 0, "batches are taken in pairs");
  auto pair = [&](int b) {
    load(b + 1, wb, xb);
    __builtin_amdgcn_sched_barrier(0);
    use(wa, xa);
    if constexpr (kF32 && UNROLL) __builtin_amdgcn_sched_barrier(0);
    load(min(b + 2, BATCHES - 1), wa, xa);
    __builtin_amdgcn_sched_barrier(0);
    use(wb, xb);
    if constexpr (kF32 && UNROLL) __builtin_amdgcn_sched_barrier(0);
  };
  load(0, wa, xa);
  if constexpr (UNROLL) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < BATCHES; b += 2) pair(b);
  } else {
#pragma unroll 1
    for (int b = 0; b < BATCHES; b += 2) pair(b);
  }
  return acc;
}

// Best scores travel as {order, kNoId - id}: the larger the better, the lower
// id first among equals, 0 for none. -0 counts as +0, a NaN competes as the
// lowest finite value and minus infinity never wins. An f16 score's order has
// 16 bits, so order and id share the word's low half and its tag has the high
// half; an f32 order fills the low half, the high one is tag << 12 | id.
constexpr uint32_t kNoId = 0xfffu;

template <class X>
struct Key;
template <>
struct Key<_Float16> {
  typedef uint32_t T;
  static constexpr uint32_t kTagMask = 0xffffffffu;
  __device__ __forceinline__ static T of(_Float16 v, uint32_t id) {
    const uint32_t u = v == (_Float16)0.0f ? 0u : __builtin_bit_cast(uint16_t, v);
    const uint32_t order = v != v ? 1u : u >> 15 ? 0xffffu - u : u | 0x8000u;
    return u == 0xfc00u ? 0u : order << 12 | (kNoId - id);
  }
  __device__ __forceinline__ static void publish_key(uint64_t* p, T key, uint32_t tag) { publish(p, key, tag); }
  __device__ __forceinline__ static uint32_t tag(uint64_t word) { return (uint32_t)(word >> 32); }
  __device__ __forceinline__ static T key(uint64_t word) { return (uint32_t)word; }
};
template <>
struct Key<float> {
  typedef uint64_t T;
  static constexpr uint32_t kTagMask = 0xfffffu;
  __device__ __forceinline__ static T of(float v, uint32_t id) {
    v = v != v ? -3.402823466e+38f : v;
    const uint32_t u = v == 0.0f ? 0u : __float_as_uint(v);
    const uint32_t order = u ^ ((u >> 31) ? 0xffffffffu : 0x80000000u);
    return u == 0xff800000u ? 0u : (uint64_t)order << 12 | (kNoId - id);
  }
  __device__ __forceinline__ static void publish_key(uint64_t* p, T key, uint32_t tag) {
    publish(p, (uint32_t)(key >> 12), tag << 12 | ((uint32_t)key & kNoId));
  }
  __device__ __forceinline__ static uint32_t tag(uint64_t word) { return (uint32_t)(word >> 44); }
  __device__ __forceinline__ static T key(uint64_t word) {
    return (word & 0xffffffffu) << 12 | ((uint32_t)(word >> 32) & kNoId);
  }
};

__device__ __forceinline__ uint32_t shfl_key(uint32_t v, int lane) { return (uint32_t)__shfl((int)v, lane, 64); }
__device__ __forceinline__ uint64_t shfl_key(uint64_t v, int lane) {
  return (uint64_t)shfl_key((uint32_t)(v >> 32), lane) << 32 | shfl_key((uint32_t)v, lane);
}

// The largest value over groups of 8 (ROW false) or 16 neighbouring lanes.
template <bool ROW>
__device__ __forceinline__ uint32_t lanes_max(uint32_t v) {
  v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xb1, 0xf, 0xf, true));   // lane ^ 1
  v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4e, 0xf, 0xf, true));   // lane ^ 2
  v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x141, 0xf, 0xf, true));  // mirrored in 8
  if (ROW) v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x140, 0xf, 0xf, true));  // in 16
  return v;
}
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
  v = lanes_max<true>(v);
  return max(max(lane_of(v, 0), lane_of(v, 16)), max(lane_of(v, 32), lane_of(v, 48)));
}
__device__ __forceinline__ uint64_t wave_max(uint64_t v) {
  const uint32_t high = (uint32_t)(v >> 12);
  const uint32_t best = wave_max(high);
  return (uint64_t)best << 12 | wave_max(high == best ? (uint32_t)v & kNoId : 0u);
}

// Column of the head's matrix at place i of the members' order: durations
// first, then tokens and blank (past the end: the last one again).
__device__ __forceinline__ uint32_t head_output(uint32_t i) {
  return i < 5u ? kTdtBlank + 1u + i : min(i - 5u, kTdtBlank);
}

// The member's share of the weights, from the package's row-major matrices
// into LDS units: the gates of units [4p, 4p + 4), then the columns of its
// role. Returns whether this thread saw a head weight that is not finite
// (then the head's zero inputs have to be left out one by one).
template <class S>
__device__ bool load_weights(const TdtArgs& a, uint32_t p, int head, int projector, uint8_t* lds) {
  typedef Geometry<S> G;
  typedef typename S::P::W Wt;
  constexpr uint32_t U = S::kUnits, C = S::kGatesPerLane;
  for (uint32_t layer = 0; layer < 2; ++layer) {
    const Wt* src = wptr<typename S::P>(a.lstm[layer]);
    uint8_t* dst = lds + layer * G::kLayerUnits * 16;
#pragma unroll 8
    for (uint32_t i = threadIdx.x; i < 2 * H * 4 * U; i += kBlock) {
      const uint32_t u = i % U, g = (i / U) % 4, k = i / (4 * U);
      const uint32_t ch = p * U + u;
      const Wt v = ch < H ? src[(uint64_t)k * kTdtGates + g * H + ch] : (Wt)0.0f;
      const uint32_t lane = u * G::kUnitLanes + 2 * (g / C) + (k & 1);
      const uint32_t row = k >> 1;
      reinterpret_cast<Wt*>(
          dst + ((row / 4) * G::kLanes + lane) * 16)[(row % 4) * C + g % C] = v;
    }
  }
  uint8_t* dst = lds + 2 * G::kLayerUnits * 16;
  bool special = false;
  if (projector >= 0) {
    constexpr uint32_t N = S::kProjectorColumns;
    const Wt* src = wptr<typename S::P>(a.projector) + (uint32_t)projector * N;
#pragma unroll 8
    for (uint32_t i = threadIdx.x; i < H * N; i += kBlock) {
      const uint32_t c = i % N, k = i / N;
      reinterpret_cast<float*>(dst + ((k / 4) * N + c) * 16)[k % 4] = (float)src[(uint64_t)k * H + c];
    }
  }
  if (head >= 0) {
    constexpr uint32_t N = S::kHeadColumns;
    const Wt* src = wptr<typename S::P>(a.head);
#pragma unroll 8
    for (uint32_t i = threadIdx.x; i < H * N; i += kBlock) {
      const uint32_t c = i % N, k = i / N;
      const Wt v = src[(uint64_t)k * kTdtHead + head_output((uint32_t)head * N + c)];
      special |= !(fabsf((float)v) <= 3.402823466e+38f);
      reinterpret_cast<Wt*>(dst + ((k / 4) * G::kHeadLanes + c / C) * 16)[(k % 4) * C + c % C] = v;
    }
  }
  return special;
}

// Two neighbouring channels of a lane: 128 i + 2 lane and the one after it.
template <class X>
struct Pair {
  X v[2];
};

template <class S>
struct Wave {
  typedef Geometry<S> G;
  typedef typename S::P P;
  typedef typename P::X X;
  typedef typename S::Acc Acc;
  static constexpr int W = (int)S::kWindows;
  static constexpr uint32_t C = S::kGatesPerLane;
  // words of a hidden vector per lane: two f16 channels in one, or one f32
  static constexpr bool kPacked = sizeof(X) == 2;
  static constexpr int kHiddenWords = kPacked ? 5 : 10;
  // where the gate chains' h1 lies: behind the packed h0, or the f32 one
  static constexpr uint32_t kH1 = kPacked ? kTdtResidentH0 + H : kTdtResidentH1F32;

  const TdtArgs& a;
  const TdtResident& r;
  uint8_t* lds;
  uint32_t member;           // workgroup
  int head, projector;       // index among the role's members, -1: not one
  uint32_t lane, slot, sub, part, channel;
  bool lane_used, own;       // the lane belongs to a window slot; and to a unit
  uint32_t first;            // first window of this wave, within the launch
  uint8_t* vectors;          // the wave's W vector slots
  Pair<X> h0[W][5];          // the windows' newest first-layer output, 10 channels per lane
  float projection[W][10];
  float hc[2], cc[2], hp[2], cp[2];  // own unit: candidate and committed h, c of each layer
  float projected;           // own projector column
  Acc bias[2];
  Acc head_bias;
  Pair<X> row[W][5];         // the encoder rows of the next joint
  float projector_bias;
  bool special, failed;

  __device__ __forceinline__ uint64_t* window_words(uint32_t w) const {
    return r.exchange + (uint64_t)(r.base + first + w) * kTdtResidentWords;
  }

  __device__ __forceinline__ uint8_t* parity(uint32_t w, uint32_t odd) const {
    return vectors + w * G::kSlotBytes + odd * G::kParityBytes;
  }

  // A vector as the input of a gate chain: even and odd rows apart.
  __device__ __forceinline__ void stage(int w, const Pair<X> (&v)[5]) const {
#pragma unroll
    for (int i = 0; i < 5; ++i) {
      reinterpret_cast<X*>(parity(w, 0))[64 * i + lane] = v[i].v[0];
      reinterpret_cast<X*>(parity(w, 1))[64 * i + lane] = v[i].v[1];
    }
  }

  __device__ __forceinline__ Acc gate_chain(Acc acc, int layer, int half) const {
    const uint4* w = reinterpret_cast<const uint4*>(lds) + layer * G::kLayerUnits + half * (H / 8) * G::kLanes + sub;
    return chain<H / 2, false, W == 1>(acc, w, G::kLanes, reinterpret_cast<const uint4*>(parity(slot, part & 1u)));
  }

  // This lane's words of a vector at `src`: two neighbouring f32 channels in
  // two words, or both in one.
  template <int N>
  __device__ __forceinline__ void load_words(const uint64_t* src, uint64_t (&word)[N]) const {
#pragma unroll
    for (int i = 0; i < N; ++i)
      word[i] = xload64(N == 5 ? src + 64 * i + lane : src + 128 * (i >> 1) + 2 * lane + (i & 1));
  }
  template <int N>
  __device__ __forceinline__ static bool tagged(const uint64_t (&word)[N], uint32_t tag) {
    bool ready = true;
#pragma unroll
    for (int i = 0; i < N; ++i) ready &= (uint32_t)(word[i] >> 32) == tag;
    return ready;
  }

  // Polls the vectors of the windows in `mask` (a bit per slot) until every
  // word carries its window's tag, loading again only where one does not;
  // false when the launch is aborted. `loaded`: `word` holds a first load.
  template <int N>
  __device__ __forceinline__ bool gather(uint32_t mask, uint32_t offset, const uint32_t (&tag)[W],
                                         uint64_t (&word)[W][N], bool loaded = false) {
    uint32_t polls = 0;
    bool ready[W];
#pragma unroll
    for (int w = 0; w < W; ++w) ready[w] = !(mask >> w & 1u) || (loaded && tagged(word[w], tag[w]));
    for (;;) {
      bool all = true;
#pragma unroll
      for (int w = 0; w < W; ++w) all &= ready[w];
      if (__all(all)) return true;
      if (polls && !wait(polls)) return false;
      ++polls;
#pragma unroll
      for (int w = 0; w < W; ++w)
        if (!ready[w]) load_words(window_words(w) + offset + (tag[w] & 1u) * (64u * N), word[w]);
#pragma unroll
      for (int w = 0; w < W; ++w)
        if (!ready[w]) ready[w] = tagged(word[w], tag[w]);
    }
  }

  // After an unsuccessful poll; false once the launch is aborted.
  __device__ __forceinline__ bool wait(uint32_t polls) {
    if ((polls & 63u) == 0u && xload(r.sync + kTdtSyncStride) != 0u) failed = true;
    if (polls > r.spin_limit) {
      if (lane == 0) xstore(r.sync + kTdtSyncStride, 1u);
      failed = true;
    }
    return !failed;
  }

  // sigmoid_f32 (gates 0, 1, 3) or clamped_tanh (gate 2): the same
  // operations, exp / add / divide shared by both.
  __device__ __forceinline__ static float activate(float v, bool is_tanh) {
    const float clamped = fminf(fmaxf(v, is_tanh ? -10.0f : -20.0f), is_tanh ? 10.0f : 20.0f);
    const float e = exp_f32(is_tanh ? 2.0f * fabsf(clamped) : -clamped);
    const float q = (is_tanh ? 2.0f : 1.0f) / (e + 1.0f);
    const float t = 1.0f - q;
    return is_tanh ? (clamped < 0.0f ? -t : t) : q;
  }

  // Cell update of the lane's unit from its gate sums: candidate h and c.
  // Every lane activates its own gates, then the unit's lanes share them.
  __device__ __forceinline__ void cell(int layer, Acc acc, bool need) {
    float ig, fg, gg, og;
    const int base = (int)(lane - part);
    static_assert(kPacked == (C == 2), "an f16 lane has two gates, an f32 lane one");
    if constexpr (C == 1) {
      const float sum = acc + __shfl_xor(acc, 1, 64);
      const float act = activate(sum, (part >> 1) == 2u);
      ig = __shfl(act, base, 64);
      fg = __shfl(act, base + 2, 64);
      gg = __shfl(act, base + 4, 64);
      og = __shfl(act, base + 6, 64);
    } else {
      const half2v sum = acc + __builtin_bit_cast(half2v, __shfl_xor(__builtin_bit_cast(int, acc), 1, 64));
      const float a0 = activate((float)sum[0], part >= 2u), a1 = activate((float)sum[1], false);
      ig = __shfl(a0, base, 64);
      fg = __shfl(a1, base, 64);
      gg = __shfl(a0, base + 2, 64);
      og = __shfl(a1, base + 2, 64);
    }
    const float c = __builtin_fmaf(fg, cp[layer], ig * gg);
    const float h = og * clamped_tanh(c);
    if (need) {
      cc[layer] = c;
      hc[layer] = h;
    }
  }

  // Publishes the lane's unit's new h as the other members read it.
  __device__ __forceinline__ void publish_hidden(uint64_t* dst, float h, uint32_t tag, bool need) const {
    if constexpr (kPacked) {
      // the even channel's first lane packs its neighbour's value beside its own
      const float other = __shfl(h, (int)(lane + G::kUnitLanes), 64);
      const half2v both{(_Float16)h, (_Float16)other};
      if (need && own && part == 0 && (channel & 1u) == 0u)
        publish(dst + (tag & 1u) * (H / 2) + channel / 2, __builtin_bit_cast(uint32_t, both), tag);
    } else {
      if (need && own && part == 0) publish(dst + (tag & 1u) * H + channel, __float_as_uint(h), tag);
    }
  }

  __device__ __forceinline__ static void unpack(Pair<X> (&h)[5], const uint64_t (&word)[kHiddenWords]) {
#pragma unroll
    for (int i = 0; i < 5; ++i) {
      if constexpr (kPacked)
        h[i] = __builtin_bit_cast(Pair<X>, (uint32_t)word[i]);
      else
        h[i] = Pair<X>{{__uint_as_float((uint32_t)word[2 * i]), __uint_as_float((uint32_t)word[2 * i + 1])}};
    }
  }

  // prepare_predictor (tdt-decoder.ts:1341-1500) of the windows in `mask`:
  // candidates from `token` and the committed state. `need`, `token` and
  // `epoch` are the lane's window's.
  // `between` runs while the new h0 travels.
  template <class Between>
  __device__ __forceinline__ bool predictor(uint32_t mask, bool need, uint32_t token, uint32_t epoch, bool initial,
                                            Between between) {
    uint32_t tag[W], previous[W];
#pragma unroll
    for (int w = 0; w < W; ++w) {
      tag[w] = lane_of(epoch, w * G::kLanes);
      previous[w] = tag[w] - 1u;
    }
    uint64_t* words = window_words(slot);
    const bool even = (part & 1u) == 0u;
    Acc acc = even ? bias[0] : Acc{};
    uint64_t h1_word[W][kHiddenWords];
    if (!initial) {
      Pair<X> e[W][5];
#pragma unroll
      for (int w = 0; w < W; ++w) {
        if (!(mask >> w & 1u)) continue;
        const uint32_t id = min(lane_of(token, w * G::kLanes), kTdtBlank);
        const Pair<X>* row = reinterpret_cast<const Pair<X>*>(wptr<P>(a.embedding) + (uint64_t)id * H);
#pragma unroll
        for (int i = 0; i < 5; ++i) e[w][i] = row[64 * i + lane];
      }
      // the previous second-layer output, used after the next exchange
#pragma unroll
      for (int w = 0; w < W; ++w)
        if (mask >> w & 1u)
          load_words(window_words(w) + kH1 + (previous[w] & 1u) * (64u * kHiddenWords), h1_word[w]);
#pragma unroll
      for (int w = 0; w < W; ++w)
        if (mask >> w & 1u) stage(w, e[w]);
      wave_fence();
      acc = gate_chain(acc, 0, 0);
      wave_fence();
#pragma unroll
      for (int w = 0; w < W; ++w)
        if (mask >> w & 1u) stage(w, h0[w]);
      wave_fence();
      acc = gate_chain(acc, 0, 1);
      wave_fence();
    }
    cell(0, acc, need);
    publish_hidden(words + kTdtResidentH0, hc[0], epoch, need);
    between();
    uint64_t h0_word[W][kHiddenWords];
    if (!gather(mask, kTdtResidentH0, tag, h0_word)) return false;
#pragma unroll
    for (int w = 0; w < W; ++w)
      if (mask >> w & 1u) {
        unpack(h0[w], h0_word[w]);
        stage(w, h0[w]);
      }
    wave_fence();
    acc = gate_chain(even ? bias[1] : Acc{}, 1, 0);
    wave_fence();
    if (!initial) {
      if (!gather(mask, kH1, previous, h1_word, true)) return false;
#pragma unroll
      for (int w = 0; w < W; ++w)
        if (mask >> w & 1u) {
          Pair<X> h1[5];
          unpack(h1, h1_word[w]);
          stage(w, h1);
        }
      wave_fence();
      acc = gate_chain(acc, 1, 1);
      wave_fence();
    }
    cell(1, acc, need);
    if (need && own && part == 0)
      publish(words + kTdtResidentH1F32 + (epoch & 1u) * H + channel, __float_as_uint(hc[1]), epoch);
    if constexpr (kPacked) publish_hidden(words + kH1, hc[1], epoch, need);
    if (projector >= 0) {
      // decoder projector (tdt-decoder.ts:1462-1491), one column per lane
      uint64_t word[W][10];
      if (!gather(mask, kTdtResidentH1F32, tag, word)) return false;
#pragma unroll
      for (int w = 0; w < W; ++w)
        if (mask >> w & 1u) {
          float2* x = reinterpret_cast<float2*>(vectors + w * G::kSlotBytes);
#pragma unroll
          for (int i = 0; i < 5; ++i)
            x[64 * i + lane] =
                make_float2(__uint_as_float((uint32_t)word[w][2 * i]), __uint_as_float((uint32_t)word[w][2 * i + 1]));
        }
      wave_fence();
      const uint32_t column = min(sub, S::kProjectorColumns - 1u);
      const float q = chain<H, false, W == 1>(projector_bias, reinterpret_cast<const uint4*>(lds) + 2 * G::kLayerUnits + column,
                                       S::kProjectorColumns,
                                       reinterpret_cast<const uint4*>(vectors + slot * G::kSlotBytes));
      wave_fence();
      if (need) projected = q;
      if (need && column_owner())
        publish(words + kTdtResidentProjection + (epoch & 1u) * H + (uint32_t)projector * S::kProjectorColumns + sub,
                __float_as_uint(q), epoch);
    }
    if (head >= 0) {
      uint64_t word[W][10];
      if (!gather(mask, kTdtResidentProjection, tag, word)) return false;
#pragma unroll
      for (int w = 0; w < W; ++w)
        if (mask >> w & 1u) {
#pragma unroll
          for (int i = 0; i < 10; ++i) projection[w][i] = __uint_as_float((uint32_t)word[w][i]);
        }
    }
    return true;
  }

  __device__ __forceinline__ bool column_owner() const {
    return projector >= 0 && lane_used && sub < S::kProjectorColumns;
  }

  // Loads the encoder rows of the next joint of the windows in `mask`.
  __device__ __forceinline__ void load_rows(uint32_t mask, uint32_t joint_time) {
    if (head < 0) return;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      if (!(mask >> w & 1u)) continue;
      const Pair<X>* src = reinterpret_cast<const Pair<X>*>(
          wptr<P>(a.encoder) +
          ((uint64_t)(r.base + first + w) * a.frames + lane_of(joint_time, w * G::kLanes)) * H);
#pragma unroll
      for (int i = 0; i < 5; ++i) row[w][i] = src[64 * i + lane];
    }
  }

  // run_joint_pair (tdt-decoder.ts:1605-1662, head :977-1031) of the windows
  // in `mask` over the loaded rows and the argmax (:773-853, :1517-1603): the
  // lane's window's token and duration.
  __device__ __forceinline__ bool joint(uint32_t mask, uint32_t step, bool running, uint32_t joint_time,
                                        uint32_t& token, uint32_t& duration) {
    typedef Key<X> K;
    const uint32_t tag = (step + 1u) & K::kTagMask;
    const uint32_t best = kTdtResidentHead + (tag & 1u) * kTdtResidentBest;
    uint32_t touched[W] = {};
    if (head >= 0) {
#pragma unroll
      for (int w = 0; w < W; ++w) {
        if (!(mask >> w & 1u)) continue;
        Pair<X>* x = reinterpret_cast<Pair<X>*>(vectors + w * G::kSlotBytes);
#pragma unroll
        for (int i = 0; i < 5; ++i) {
          Pair<X> in;
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const float s = (float)row[w][i].v[j] + projection[w][2 * i + j];
            in.v[j] = s > 0.0f ? (X)s : (X)-0.0f;  // -0 marks an input the chain leaves out
          }
          x[64 * i + lane] = in;
        }
      }
      wave_fence();
      const uint32_t column = min(sub, G::kHeadLanes - 1u);
      const uint4* w = reinterpret_cast<const uint4*>(lds) + 2 * G::kLayerUnits + column;
      const uint4* x = reinterpret_cast<const uint4*>(vectors + slot * G::kSlotBytes);
      // With finite weights a left-out row is a multiplication by zero: it
      // can only change the sign of a zero, which no comparison sees.
      const Acc acc = special ? chain<H, true, false>(head_bias, w, G::kHeadLanes, x)
                              : chain<H, false, W == 1>(head_bias, w, G::kHeadLanes, x);
      wave_fence();
      X score[C];
      if constexpr (C == 1) {
        score[0] = acc;
      } else {
        score[0] = acc[0];
        score[1] = acc[1];
      }
      typename K::T key = 0;
#pragma unroll
      for (uint32_t c = 0; c < C; ++c) {
        const uint32_t index = (uint32_t)head * S::kHeadColumns + column * C + c;
        const uint32_t output = head_output(index);
        const typename K::T k = K::of(score[c], output);
        if (sub < G::kHeadLanes && index < G::kOutputs && output <= kTdtBlank) key = max(key, k);
      }
      const int base = (int)(slot * G::kLanes);
      if (head == 0) {
        typename K::T best_duration = 0;
#pragma unroll
        for (uint32_t i = 0; i < 5; ++i)
          best_duration = max(best_duration, shfl_key(K::of(score[i % C], i), base + (int)(i / C)));
        if (running && lane_used && sub == 0) K::publish_key(window_words(slot) + best + G::kHeadMembers, best_duration, tag);
      }
      if constexpr (G::kHeadLanes == 8 && G::kLanes % 8 == 0 && sizeof(key) == 4) {
        key = lanes_max<false>(key);
      } else {
#pragma unroll
        for (uint32_t off = 8; off > 0; off >>= 1) {
          const typename K::T other = shfl_key(key, base + (int)min(sub + off, G::kLanes - 1u));
          if (sub + off < G::kHeadLanes) key = max(key, other);
        }
      }
      if (running && lane_used && sub == 0) K::publish_key(window_words(slot) + best + (uint32_t)head, key, tag);
      // While the words travel: bring the rows that a joint after a blank may
      // want (durations up to 4) into this XCD's L2.
#pragma unroll
      for (int w = 0; w < W; ++w) {
        if (!(mask >> w & 1u)) continue;
        const uint32_t t = lane_of(joint_time, w * G::kLanes) + 1u;
        constexpr uint32_t kLines = H * (uint32_t)sizeof(X) / 128u;
        const uint32_t row_ahead = min(t + lane / 16u, a.frames - 1u);
        const uint8_t* src = reinterpret_cast<const uint8_t*>(
            wptr<P>(a.encoder) + ((uint64_t)(r.base + first + w) * a.frames + row_ahead) * H);
        touched[w] = *reinterpret_cast<const uint32_t*>(src + min(lane % 16u, kLines - 1u) * 128u);
      }
    } else if (running && lane_used && sub == 0) {
      K::publish_key(window_words(slot) + best + 1u + member, 0, tag);
    }
    // Scores, the duration and, for a head member, every other member's word.
    constexpr int N = (G::kMembers + 1 + 63) / 64, kScores = (G::kHeadMembers + 1 + 63) / 64;
    const uint32_t count = head >= 0 ? G::kMembers + 1u : G::kHeadMembers + 1u;
    uint32_t polls = 0;
    uint64_t word[W][kScores];
    bool ready[W];
#pragma unroll
    for (int w = 0; w < W; ++w) ready[w] = !(mask >> w & 1u);
    for (;;) {
      bool all = true;
#pragma unroll
      for (int w = 0; w < W; ++w) all &= ready[w];
      if (__all(all)) break;
      if (polls && !wait(polls)) return false;
      ++polls;
      uint64_t extra[W][N];
#pragma unroll
      for (int w = 0; w < W; ++w) {
        if (ready[w]) continue;
        const uint64_t* src = window_words(w) + best;
#pragma unroll
        for (int i = 0; i < N; ++i) {
          if (i >= kScores && head < 0) continue;
          const uint64_t v = xload64(src + min(64 * i + lane, count - 1u));
          extra[w][i] = v;
        }
      }
#pragma unroll
      for (int w = 0; w < W; ++w) {
        if (ready[w]) continue;
        bool ok = true;
#pragma unroll
        for (int i = 0; i < N; ++i) {
          if (i < kScores) word[w][i] = extra[w][i];
          if (i >= kScores && head < 0) continue;
          ok &= K::tag(extra[w][i]) == tag;
        }
        ready[w] = ok;
      }
    }
#pragma unroll
    for (int w = 0; w < W; ++w) {
      asm volatile("" ::"v"(touched[w]));
      if (!(mask >> w & 1u)) continue;
      typename K::T key = 0;
#pragma unroll
      for (int i = 0; i < kScores; ++i)
        if (64 * i + lane < G::kHeadMembers) key = max(key, K::key(word[w][i]));
      key = wave_max(key);
      const uint32_t d = lane_of((uint32_t)K::key(word[w][G::kHeadMembers / 64]), G::kHeadMembers % 64) & kNoId;
      if (slot == (uint32_t)w) {
        token = key ? kNoId - ((uint32_t)key & kNoId) : 0xffffffffu;
        duration = d ? kNoId - d : 0xffffffffu;
      }
    }
    return true;
  }
};

template <class S>
__global__ __launch_bounds__(kBlock) void tdt_resident_kernel(TdtArgs a, TdtResident r) {
  typedef Geometry<S> G;
  typedef typename S::Acc Acc;
  constexpr int W = (int)S::kWindows;
  extern __shared__ __align__(16) uint8_t lds[];
  uint32_t* flag = reinterpret_cast<uint32_t*>(lds + G::kWeightUnits * 16);
  // Members with neighbouring columns share cache lines of the row-major
  // matrices: give each of the eight XCDs (workgroups go to them round
  // robin) a contiguous range.
  const uint32_t xcd = blockIdx.x % 8u;
  const uint32_t p = xcd * (G::kMembers / 8u) + min(xcd, G::kMembers % 8u) + blockIdx.x / 8u;
  const int head = blockIdx.x < G::kHeadMembers ? (int)blockIdx.x : -1;
  const int projector =
      blockIdx.x >= G::kMembers - G::kProjectorMembers ? (int)(blockIdx.x - (G::kMembers - G::kProjectorMembers)) : -1;
  uint32_t* joined = r.sync;
  uint32_t* abort = r.sync + kTdtSyncStride;
  if (threadIdx.x == 0) {
    __hip_atomic_fetch_add(joined, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *flag = xload(abort);
  }
  __syncthreads();
  if (*flag) return;
  // Bring the embedding into this XCD's L2, a share per member.
  for (uint32_t i = blockIdx.x / 8u * kBlock + threadIdx.x; i < (kTdtBlank + 1) * H * sizeof(typename S::P::W) / 128;
       i += G::kMembers / 8u * kBlock) {
    const uint32_t touched = reinterpret_cast<const uint32_t*>(a.embedding)[i * 32u];
    asm volatile("" ::"v"(touched));
  }
  const bool special = __syncthreads_or(load_weights<S>(a, p, head, projector, lds)) != 0;
  if (threadIdx.x == 0) {
    const uint64_t start = wall_clock64();
    uint32_t failed = 0;
    while (r.join_ticks == 0 || xload(joined) < G::kMembers) {
      failed = xload(abort);
      if (!failed && wall_clock64() - start >= r.join_ticks) {
        xstore(abort, 1u);
        failed = 1;
      }
      if (failed) break;
      __builtin_amdgcn_s_sleep(8);
    }
    *flag = failed;
  }
  __syncthreads();
  if (*flag) return;

  const uint32_t wave = threadIdx.x / 64u;
  if (wave * W >= r.windows) return;
  Wave<S> v{a, r};
  v.lds = lds;
  v.member = blockIdx.x;
  v.head = head;
  v.projector = projector;
  v.lane = threadIdx.x & 63u;
  v.lane_used = v.lane < W * G::kLanes;
  v.slot = min(v.lane / G::kLanes, (uint32_t)W - 1u);
  v.sub = min(v.lane - v.slot * G::kLanes, G::kLanes - 1u);
  v.part = v.sub % G::kUnitLanes;
  v.channel = p * S::kUnits + v.sub / G::kUnitLanes;
  v.first = wave * W;
  v.own = v.lane_used && v.channel < H;
  v.vectors = lds + G::kFixedBytes + wave * W * G::kSlotBytes;
  v.special = special;
  v.failed = false;
  const uint32_t channel = min(v.channel, H - 1u);
#pragma unroll
  for (int l = 0; l < 2; ++l) {
    const float* b = a.lstm_bias[l] + (v.part >> 1) * S::kGatesPerLane * H + channel;
    if constexpr (S::kGatesPerLane == 1)
      v.bias[l] = (Acc)b[0];
    else
      v.bias[l] = Acc{(_Float16)b[0], (_Float16)b[H]};
  }
  const uint32_t column =
      (uint32_t)max(head, 0) * S::kHeadColumns + min(v.sub, G::kHeadLanes - 1u) * S::kGatesPerLane;
  if constexpr (S::kGatesPerLane == 1)
    v.head_bias = (Acc)a.head_bias[head_output(column)];
  else
    v.head_bias = Acc{(_Float16)a.head_bias[head_output(column)], (_Float16)a.head_bias[head_output(column + 1u)]};
  v.projector_bias =
      a.projector_bias[(uint32_t)max(projector, 0) * S::kProjectorColumns + min(v.sub, S::kProjectorColumns - 1u)];
#pragma unroll
  for (int l = 0; l < 2; ++l) v.hc[l] = v.cc[l] = v.hp[l] = v.cp[l] = 0.0f;
  v.projected = 0.0f;

  // Control state of the lane's window; every member's copy evolves alike.
  const bool exists = v.first + v.slot < r.windows;
  const uint32_t b = r.base + min(v.first + v.slot, r.windows - 1u);
  const uint32_t limit = min(a.lengths[b], a.frames);
  const uint32_t encoded = min(limit, a.ends[b]);
  const uint32_t start = a.starts[b];
  uint32_t time = min(start, encoded), count = 0, st = 0, symbols = 0;
  bool flushing = false;
  uint32_t flush_blanks = 0, flush_time = 0;
  const bool flush_requested = a.flush[b] != 0 && start < encoded;
  const bool writer = blockIdx.x == 0 && v.sub == 0 && v.lane_used;

  bool running = exists, need = exists && time < encoded, initial = true;
  uint32_t epoch = 0, token = 0, duration = 0;
  auto slots = [&](bool lane_flag) {
    uint32_t mask = 0;
#pragma unroll
    for (int w = 0; w < W; ++w) mask |= (lane_of(lane_flag ? 1u : 0u, w * G::kLanes) & 1u) << w;
    return mask;
  };
  const uint32_t max_steps = 11 * a.frames + 32;
  uint32_t joint_time = 0, active = 0, step = 0;
  // The last joint's outcome, then the frame of the next one, or the end.
  auto control = [&] {
    if (running && step > 0) {
      const bool emitted = token != kTdtBlank;
      const uint32_t frame = flushing ? min(flush_time, encoded - 1u) : time;
      if (emitted) {
        if (count < a.max_tokens) {
          if (writer) {
            const uint64_t at = (uint64_t)b * a.max_tokens + count;
            a.tokens[at] = token;
            a.token_frames[at] = frame;
            a.token_durations[at] = duration;
          }
          ++count;
        } else {
          st |= 1u;
        }
      }
      if (!flushing) {
        symbols += 1;
        if (duration != 0) {
          time += duration;
          symbols = 0;
        } else if (!emitted || symbols >= 10) {
          time += 1;
          symbols = 0;
        }
      } else {
        flush_blanks = emitted ? 0u : flush_blanks + 1u;
        flush_time = min(flush_time + max(1u, duration), encoded);
        symbols += 1;
      }
    }
    // choose the frame of this step's joint, or stop (:1722-1735, :1812-1880)
    bool go = false;
    if (running && step < max_steps) {
      if (!flushing && time < encoded) {
        go = true;
        joint_time = time;
      } else {
        if (!flushing && flush_requested) {
          flushing = true;
          symbols = 0;
          flush_blanks = 0;
          flush_time = time;
        }
        if (flushing && symbols < 10 && flush_blanks < 5) {
          const uint32_t variation = symbols % 3;
          if (variation == 0)
            time = min(flush_time, limit - 1u);
          else if (variation == 1)
            time = min(encoded - 1u, a.frames - 1u);
          else
            time = min(max(encoded, 2u) - 2u, a.frames - 1u);
          go = true;
          joint_time = time;
        }
      }
    }
    running = go;
    active = slots(running);
    v.load_rows(active, joint_time);
  };
  for (;; ++step) {
    const uint32_t predict = slots(need);
    if (predict) {
      if (need) ++epoch;
      if (!v.predictor(predict, need, token, epoch, initial, control)) return;
    } else {
      control();
    }
    initial = false;
    if (!active) break;
    if (!v.joint(active, step, running, joint_time, token, duration)) return;
    need = running && token != kTdtBlank;
    if (need) {
      // commit_predictor (:1502-1515)
#pragma unroll
      for (int l = 0; l < 2; ++l) {
        v.hp[l] = v.hc[l];
        v.cp[l] = v.cc[l];
      }
    }
  }
  if (!exists) return;
  float* state = a.state + (uint64_t)b * 4 * H;
  float* cand = a.scratch + (uint64_t)b * 5 * H;
  if (v.own && v.part == 0) {
#pragma unroll
    for (uint32_t l = 0; l < 2; ++l) {
      state[2 * l * H + v.channel] = v.hp[l];
      state[(2 * l + 1) * H + v.channel] = v.cp[l];
      if (epoch) {
        cand[2 * l * H + v.channel] = v.hc[l];
        cand[(2 * l + 1) * H + v.channel] = v.cc[l];
      }
    }
  }
  if (epoch && v.column_owner()) cand[4 * H + (uint32_t)projector * S::kProjectorColumns + v.sub] = v.projected;
  if (writer) {
    a.counts[b] = count;
    a.status[b] = st;
  }
}

__global__ void tdt_resident_clear(uint4* words, uint32_t count) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < count; i += gridDim.x * blockDim.x)
    words[i] = make_uint4(0u, 0u, 0u, 0u);
}

typedef void (*ResidentKernel)(TdtArgs, TdtResident);

struct ResidentPlan {
  ResidentKernel kernel;
  uint32_t members, lds_bytes;
};

template <class S>
ResidentPlan plan_of(uint32_t windows) {
  typedef Geometry<S> G;
  const uint32_t slots = (windows + S::kWindows - 1) / S::kWindows * S::kWindows;
  return {tdt_resident_kernel<S>, G::kMembers, G::kFixedBytes + slots * G::kSlotBytes};
}

ResidentPlan resident_plan(bool f32, uint32_t windows) {
  // One window per wave while there is a SIMD for each: its chains are written
  // out and no window waits for another's tokens (four windows of 188 frames:
  // f16 3.30 ms against 4.02 with two per wave, f32 3.30 against 4.42). Beyond
  // that as many as fill a wave's lanes, which read the weights from LDS once
  // for all of them (eight f16 windows: 4.50 ms with four or two per wave).
  if (f32) return windows <= 4 ? plan_of<ShapeF32<1>>(windows) : plan_of<ShapeF32<2>>(windows);
  return windows <= 4 ? plan_of<ShapeF16<1>>(windows) : plan_of<ShapeF16<4>>(windows);
}

}  // namespace

uint32_t tdt_resident_windows(bool f32) { return f32 ? 6u : 16u; }

bool tdt_resident_fits(int device, bool f32) {
  int cus = 0, per_cu = 0;
  const ResidentPlan plan = resident_plan(f32, tdt_resident_windows(f32));
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) return false;
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(plan.kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)plan.lds_bytes) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(plan.kernel), (int)kBlock,
                                                   plan.lds_bytes) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return (uint64_t)cus * per_cu >= plan.members;
}

hipError_t launch_tdt_resident(const TdtArgs& args, const TdtResident& resident, uint32_t batch, bool f32,
                               hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
  if (batch == 0) return hipSuccess;
  const uint32_t launches = (batch + tdt_resident_windows(f32) - 1) / tdt_resident_windows(f32);
  if (launches > kTdtResidentLaunches) return hipErrorInvalidValue;
  const uint32_t per_launch = (batch + launches - 1) / launches;
  const ResidentPlan plan = resident_plan(f32, per_launch);
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(plan.kernel),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)plan.lds_bytes);
  if (e != hipSuccess) return e;
  // the sync words precede the exchanged ones: one range to clear
  const uint32_t units =
      (uint32_t)(resident.exchange + (uint64_t)batch * kTdtResidentWords - reinterpret_cast<uint64_t*>(resident.sync)) / 2;
  hipLaunchKernelGGL(tdt_resident_clear, dim3(min((units + 255) / 256, 1024u)), dim3(256), 0, stream,
                     reinterpret_cast<uint4*>(resident.sync), units);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  TdtResident r = resident;
  for (uint32_t i = 0; i < launches && i * per_launch < batch; ++i) {
    r.sync = resident.sync + 2 * i * kTdtSyncStride;
    r.base = i * per_launch;
    r.windows = min(per_launch, batch - r.base);
    if (start && i == 0)
      hipExtLaunchKernelGGL(plan.kernel, dim3(plan.members), dim3(kBlock), plan.lds_bytes, stream, start, nullptr, 0,
                            args, r);
    else
      hipLaunchKernelGGL(plan.kernel, dim3(plan.members), dim3(kBlock), plan.lds_bytes, stream, args, r);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  // windows of an aborted launch; none otherwise
  TdtArgs again = args;
  again.aborted = resident.sync + kTdtSyncStride;
  again.aborted_windows = per_launch;
  if (resident.team.members) {
    if ((e = launch_tdt_team(again, resident.team, batch, stream, nullptr, nullptr, true)) != hipSuccess) return e;
    again.after_team = 1;
  }
  return launch_tdt_decode(again, batch, f32, stream, nullptr, stop);
}

}  // namespace pk
