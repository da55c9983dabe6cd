// gfx950 kernels for MRG8 generation.
//
// Replaces the CUDA generation kernels rng_outer_32 and rng_inner
// (cuda/mrg8_cuda.cu:201-399).  Design:
//   * A wave owns a contiguous run (tile) of outputs of one stream.  The
//     8-word state is wave-uniform (scalar registers); lane k holds the
//     centred coefficients of row 0 of A^(PL k + i + 1), i < PL, so one
//     iteration yields 64 * PL consecutive outputs with eight signed
//     32x32->64 multiply-adds each (v_mad_i64_i32, the PL dot products
//     interleaved) and a Mersenne fold.
//   * The next state is the last eight outputs, read back with v_readlane;
//     no LDS and no barrier in the loop.
//   * Outputs leave through coalesced non-temporal vector stores (16 bytes
//     per lane, 1 KiB per wave store); a run first writes the outputs before
//     its first 1 KiB boundary one per lane.
//   * A wave reaches its first position with a jump: each non-zero byte d
//     at position k of the 64-bit offset is one product with A^(d 256^k)
//     (at most 8 steps).  Eight lane groups of eight lanes jump eight states
//     at once, lane r of a group holding word r and computing row r, with
//     the rows of the next digits already on their way.
//   * k_fill: one stream, one tile per wave, each wave on its own (no LDS, no
//     barrier).
//   * k_batch: many streams (segments), a persistent grid striding over
//     tiles, tables and counts read from one device block; k_batch_short the
//     same for many short tiles, eight at a time on the matrix cores;
//     k_batch_tiles one tile per wave; k_batch_queue a persistent grid that
//     takes its tiles in address order.
//   * Blocks reach their part of the output through xcd_block: the
//     dispatcher deals blocks to the XCDs in turn, and large grids give each
//     XCD runs of consecutive blocks' output instead.
#include "mrg8_device.hpp"

namespace mrg8 {
namespace {

constexpr double kRnorm = 1.0 / 2147483647.0;  // original/mrg8.cpp:233

typedef double d2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u4_t __attribute__((ext_vector_type(4)));

struct Coef {
  int32_t c[8];
  uint64_t b0;
};

__device__ __forceinline__ Coef load_coef(const CoefRecord* __restrict__ p) {
  const u4_t* q = reinterpret_cast<const u4_t*>(p);
  const u4_t a = q[0], b = q[1];
  // the two words of b0 alone: a load into a register nothing reads lets the
  // compiler reuse that register while the load is in flight, which forces a
  // wait for it there, before loads that could be in flight with it
  const u2_t c = *reinterpret_cast<const u2_t*>(q + 2);
  Coef k;
  k.c[0] = (int32_t)a.x; k.c[1] = (int32_t)a.y; k.c[2] = (int32_t)a.z; k.c[3] = (int32_t)a.w;
  k.c[4] = (int32_t)b.x; k.c[5] = (int32_t)b.y; k.c[6] = (int32_t)b.z; k.c[7] = (int32_t)b.w;
  k.b0 = (uint64_t)c.x | ((uint64_t)c.y << 32);
  return k;
}

// w = 2 * hi + lo as one 32x32->64 multiply-add (2^32 == 2 mod p).
__device__ __forceinline__ uint64_t fold_hi(uint32_t hi, uint32_t lo) {
  uint64_t w, carry;
  asm("v_mad_u64_u32 %0, %1, %2, 2, %3" : "=v"(w), "=s"(carry) : "v"(hi), "v"((uint64_t)lo));
  return w;
}

// Canonical residue r in [0, p) of V = B0 + sum_j c_j e_j, where e_j = s_j - 2^30;
// the reference's word for the dot product is r + 1 (see CoefRecord).
__device__ __forceinline__ uint32_t dot_residue(const Coef& k, const int32_t e[8]) {
  uint64_t v = k.b0;
#pragma unroll
  for (int j = 0; j < 8; ++j) v += (uint64_t)((int64_t)k.c[j] * (int64_t)e[j]);
  const uint64_t w = fold_hi((uint32_t)(v >> 32), (uint32_t)v);        // < 3 * 2^32
  const uint32_t x = ((uint32_t)w & kP) + (uint32_t)(w >> 31);          // < 2^31 + 6
  return min(x, x - kP);  // x - p wraps above x when x < p
}

// PL residues at once, the eight multiply-adds of the PL dot products
// interleaved so that consecutive 64-bit multiply-adds are independent and
// issue back to back.
template <int PL>
__device__ __forceinline__ void dot_residues(const Coef (&k)[PL], const int32_t e[8], uint32_t r[PL]) {
  uint64_t v[PL];
#pragma unroll
  for (int i = 0; i < PL; ++i) v[i] = k[i].b0;
#pragma unroll
  for (int j = 0; j < 8; ++j)
#pragma unroll
    for (int i = 0; i < PL; ++i) v[i] += (uint64_t)((int64_t)k[i].c[j] * (int64_t)e[j]);
#pragma unroll
  for (int i = 0; i < PL; ++i) {
    const uint64_t w = fold_hi((uint32_t)(v[i] >> 32), (uint32_t)v[i]);
    const uint32_t x = ((uint32_t)w & kP) + (uint32_t)(w >> 31);
    r[i] = min(x, x - kP);
  }
}

__device__ __forceinline__ void centre(const uint32_t s[8], int32_t e[8]) {
#pragma unroll
  for (int j = 0; j < 8; ++j) e[j] = (int32_t)(s[j] - kCenter);
}

// ---- jumps: eight lanes per state, lane r holding word r and computing row r

// The value of v in the lanes l ^ 0 .. l ^ 7 of this lane's group of eight.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xf, 0xf, true);
}

__device__ __forceinline__ void gather_xor(uint32_t v, uint32_t w[8]) {
  constexpr int kXor1 = 0xB1, kXor2 = 0x4E, kXor3 = 0x1B;  // quad_perm [1,0,3,2], [2,3,0,1], [3,2,1,0]
  const uint32_t m = dpp<0x141>(v);                        // row_half_mirror: lane ^ 7
  w[0] = v;
  w[1] = dpp<kXor1>(v);
  w[2] = dpp<kXor2>(v);
  w[3] = dpp<kXor3>(v);
  w[4] = dpp<kXor3>(m);
  w[5] = dpp<kXor2>(m);
  w[6] = dpp<kXor1>(m);
  w[7] = m;
}

// This lane's row of a jump matrix (entries in the order of gather_xor).
struct JumpRow {
  int32_t c[8];
};

__device__ __forceinline__ JumpRow load_row(const int32_t* p) {  // p: the matrix + 4 * row
  const u4_t a = *reinterpret_cast<const u4_t*>(p), b = *reinterpret_cast<const u4_t*>(p + 32);
  return JumpRow{{(int32_t)a.x, (int32_t)a.y, (int32_t)a.z, (int32_t)a.w, (int32_t)b.x, (int32_t)b.y, (int32_t)b.z,
                  (int32_t)b.w}};
}

// The next centred word from a row's sum (see jump_matrix_entries).
__device__ __forceinline__ int32_t reduce_centred(uint64_t v) {
  const uint64_t f = fold_hi((uint32_t)(v >> 32), (uint32_t)v);
  return (int32_t)(((uint32_t)f & kP) + (uint32_t)(f >> 31) - kCenter);
}

// One product: this lane's centred word of (matrix) x (state), the state's
// words being the centred e of the group's lanes.
__device__ __forceinline__ int32_t jump_row(const JumpRow& m, int32_t e) {
  uint32_t w[8];
  gather_xor((uint32_t)e, w);
  uint64_t v = kJumpBase;
#pragma unroll
  for (int k = 0; k < 8; ++k) v += (uint64_t)((int64_t)m.c[k] * (int64_t)(int32_t)w[k]);
  return reduce_centred(v);
}

__device__ __forceinline__ int32_t centre_word(uint32_t s) { return (int32_t)(s >= kCenter ? s - kP : s); }
__device__ __forceinline__ uint32_t word_of(int32_t e) { return (uint32_t)(e > 0 ? e : e + (int32_t)kP); }  // in [1, p]

__device__ __forceinline__ uint32_t digit_of(uint32_t half, int k) { return (half >> (8 * (k & 3))) & 0xffu; }

// The product for a state that has a zero word (this lane's word s, its
// group's digit d): bigDotProd is 0 exactly where every product of a row is.
// A state without a zero word never gets one (no row of a power of A is
// zero), so only waves that start with such a state need this.
__device__ __forceinline__ uint32_t jump_zero_words(uint32_t s, uint32_t d, const int32_t* position) {
  const JumpRow m = load_row(position + d * kJumpMatrixInts + 4 * (threadIdx.x & 7));
  uint32_t w[8];
  gather_xor(s, w);
  bool any = false;
#pragma unroll
  for (int q = 0; q < 8; ++q) any = any || (m.c[q] != 0 && w[q] != 0u);
  const uint32_t y = word_of(jump_row(m, centre_word(s)));
  return any ? y : 0u;
}

// Rows of four byte positions of an offset (32 bits of it), and their
// products; positions where no group of the wave has a digit are skipped.
__device__ __forceinline__ void load_rows4(JumpRow m[4], const int32_t* positions, uint32_t half) {
#pragma unroll
  for (int b = 0; b < 4; ++b)
    m[b] = load_row(positions + b * kPositionInts + digit_of(half, b) * kJumpMatrixInts + 4 * (threadIdx.x & 7));
}

__device__ __forceinline__ int32_t apply_rows4(const JumpRow m[4], uint32_t half, int32_t e) {
#pragma unroll
  for (int b = 0; b < 4; ++b)
    if (__ballot(digit_of(half, b) != 0u)) e = jump_row(m[b], e);
  return e;
}

// Jumps eight states at once: this lane's group of eight holds one state (word
// s of it here) and its own 64-bit offset.  The rows of all of an offset's
// digits are independent loads: four of them are in flight, so a jump does not
// wait for memory once per digit.  65536 random 63-bit jumps and 256 words
// each: 25.5 us, 27.4 us with 48-byte records fetched one digit ahead and
// words gathered through LDS swizzles; one tile per wave 73 against 104 us.
__device__ __forceinline__ uint32_t jump_group(uint32_t s, uint64_t off, const int32_t* __restrict__ digits) {
  constexpr int kAhead = 4;
  if (!__ballot(off != 0)) return s;
  const uint32_t lo = (uint32_t)off, hi = (uint32_t)(off >> 32);
  const bool more = __ballot(hi != 0u);
  auto row = [&](int k) {
    return load_row(digits + k * kPositionInts + digit_of(k < 4 ? lo : hi, k) * kJumpMatrixInts + 4 * (threadIdx.x & 7));
  };
  // issued before the state is looked at, which may still be on its way
  JumpRow m[kAhead];
#pragma unroll
  for (int k = 0; k < kAhead; ++k) m[k] = row(k);
  if (__ballot(s == 0u)) {
#pragma unroll 1
    for (int k = 0; k < kJumpPositions; ++k) {
      const uint32_t d = digit_of(k < 4 ? lo : hi, k);
      if (__ballot(d != 0u)) s = jump_zero_words(s, d, digits + k * kPositionInts);
    }
    return s;
  }
  int32_t e = centre_word(s);
#pragma unroll
  for (int k = 0; k < kJumpPositions; ++k) {
    if (k == 4 && !more) break;
    if (__ballot(digit_of(k < 4 ? lo : hi, k) != 0u)) e = jump_row(m[k % kAhead], e);
    if (k + kAhead < 4 || (k + kAhead < kJumpPositions && more)) m[k % kAhead] = row(k + kAhead);
  }
  return word_of(e);
}

// A pointer that the compiler takes as read anew, still to global memory (a
// flat access counts as an LDS access too, and waits for those).
template <typename T>
__device__ __forceinline__ const T* opaque(const T* p) {
  uint64_t address = reinterpret_cast<uint64_t>(p);
  asm("" : "+s"(address));
  return (const T*)(const __attribute__((address_space(1))) T*)address;
}

// jump_group with one uniform offset, for the state in a wave's first lane
// group: digits and row addresses stay scalar (nothing is counted over the
// lanes, no address is added in vector registers).  2^28 doubles 323 -> 320
// us at full clock, 365 -> 351 us in launches 6 to 25 after idle, where the
// power manager holds the clock down by the work of the vector units; 2^22
// 8.0 -> 8.2 us.
__device__ __forceinline__ uint32_t jump_uniform(uint32_t s, uint64_t off, const int32_t* digits) {
  if (off == 0) return s;
  const uint32_t lo = (uint32_t)off;
  uint32_t hi = (uint32_t)(off >> 32);
  const uint32_t row = 4 * (threadIdx.x & 7);
  auto load = [&](int k) {
    return load_row(opaque(digits + k * kPositionInts + digit_of(k < 4 ? lo : hi, k) * kJumpMatrixInts) + row);
  };
  JumpRow m[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) m[k] = load(k);
  if (__ballot(s == 0u)) {
#pragma unroll 1
    for (int k = 0; k < kJumpPositions; ++k) {
      const uint32_t d = digit_of(k < 4 ? lo : hi, k);
      if (d) s = jump_zero_words(s, d, digits + k * kPositionInts);
    }
    return s;
  }
  int32_t e = centre_word(s);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (digit_of(lo, k)) e = jump_row(m[k], e);
    asm("" : "+s"(hi));  // compared anew: one comparison kept for all is kept in vector registers
    if (hi) m[k] = load(k + 4);
  }
  asm("" : "+s"(hi));
  if (hi) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (digit_of(hi, k)) e = jump_row(m[k], e);
  }
  return word_of(e);
}

// A state in uniform registers, its word j in lane j < 8 (jump_group's first
// lane group; the other lanes hold 1, no zero word).  Eight lane writes: a
// select by lane takes 23 operations, and a load by lane waits for memory.
// The wait states are for a DPP read of the result.
__device__ __forceinline__ uint32_t own_word(const uint32_t st[8]) {
  uint32_t w = 1;
  asm("v_writelane_b32 %0, %1, 0\n\tv_writelane_b32 %0, %2, 1\n\tv_writelane_b32 %0, %3, 2\n\t"
      "v_writelane_b32 %0, %4, 3\n\tv_writelane_b32 %0, %5, 4\n\tv_writelane_b32 %0, %6, 5\n\t"
      "v_writelane_b32 %0, %7, 6\n\tv_writelane_b32 %0, %8, 7\n\ts_nop 1"
      : "+v"(w)
      : "s"(st[0]), "s"(st[1]), "s"(st[2]), "s"(st[3]), "s"(st[4]), "s"(st[5]), "s"(st[6]), "s"(st[7]));
  return w;
}

template <int FMT>
struct Out;
template <>
struct Out<0> { typedef double T; };
template <>
struct Out<1> { typedef double T; };
template <>
struct Out<2> { typedef uint32_t T; };

// Output value for residue r, the reference's word being x = r + 1.
template <int FMT>
__device__ __forceinline__ typename Out<FMT>::T convert(uint32_t r) {
  if constexpr (FMT == 0) return __fma_rn((double)r, kRnorm, kRnorm);  // double(x) * (1/p), one rounding: original/mrg8.cpp:236
  else if constexpr (FMT == 1) return (double)r * kRnorm;              // double(x - 1) * (1/p): cuda/mrg8_cuda.cu:363
  else return r + 1u;                                                  // x: original/mrg8.cpp:219
}

// Output value of the all-zero state (whose words stay 0).
template <int FMT>
__device__ __forceinline__ typename Out<FMT>::T convert_zero() {
  if constexpr (FMT == 0) return 0.0;
  else if constexpr (FMT == 1) return (double)0xffffffffu * kRnorm;  // (x - 1) wraps in 32 bits
  else return 0u;
}

// Which outputs of an iteration (64 * PL consecutive outputs) a lane makes.
// Doubles with PL = 4 use two halves: lane k makes outputs 2k, 2k+1 and
// 128+2k, 128+2k+1, so each of the lane's two 16-byte stores belongs to a
// fully contiguous 1 KiB store of the wave.  Otherwise lane k makes outputs
// PL k .. PL k + PL - 1 (one store of 4, 8 or 16 bytes).
template <int FMT, int PL>
struct LaneLayout {
  static constexpr bool kSplit = FMT != 2 && PL == 4;
  static __device__ __forceinline__ uint32_t index(uint32_t lane, int i) {
    if constexpr (kSplit) return 128u * (uint32_t)(i / 2) + 2u * lane + (uint32_t)(i % 2);
    else return PL * lane + (uint32_t)i;
  }
  // the slot (0..PL-1) and lane that make output o of an iteration
  static constexpr int slot_of(int o) { return kSplit ? 2 * (o / 128) + o % 2 : o % PL; }
  static constexpr int lane_of(int o) { return kSplit ? (o % 128) / 2 : o / PL; }
};

// Non-temporal stores of one lane's PL outputs of the iteration at `base`.
template <int FMT, int PL>
__device__ __forceinline__ void store_lane(typename Out<FMT>::T* base, uint32_t lane, const uint32_t r[PL]) {
  if constexpr (FMT == 2 && PL == 4) {
    u4_t v = {r[0] + 1u, r[1] + 1u, r[2] + 1u, r[3] + 1u};
    __builtin_nontemporal_store(v, reinterpret_cast<u4_t*>(base + 4 * lane));
  } else if constexpr (FMT == 2 && PL == 2) {
    u2_t v = {r[0] + 1u, r[1] + 1u};
    __builtin_nontemporal_store(v, reinterpret_cast<u2_t*>(base + 2 * lane));
  } else if constexpr (FMT != 2 && PL == 4) {
    d2_t v0 = {convert<FMT>(r[0]), convert<FMT>(r[1])};
    d2_t v1 = {convert<FMT>(r[2]), convert<FMT>(r[3])};
    __builtin_nontemporal_store(v0, reinterpret_cast<d2_t*>(base + 2 * lane));
    __builtin_nontemporal_store(v1, reinterpret_cast<d2_t*>(base + 128 + 2 * lane));
  } else if constexpr (FMT != 2 && PL == 2) {
    d2_t v = {convert<FMT>(r[0]), convert<FMT>(r[1])};
    __builtin_nontemporal_store(v, reinterpret_cast<d2_t*>(base + 2 * lane));
  } else {
#pragma unroll
    for (int i = 0; i < PL; ++i) __builtin_nontemporal_store(convert<FMT>(r[i]), base + PL * lane + i);
  }
}

// This lane's PL records: row 0 of A^(o + 1) for each output o it makes.
template <int FMT, int PL>
__device__ __forceinline__ void load_lane_coefs(Coef (&k)[PL], const CoefRecord* __restrict__ lane_rec) {
  const uint32_t lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < PL; ++i) k[i] = load_coef(lane_rec + LaneLayout<FMT, PL>::index(lane, i));
}

// Writes the first k (< 64) outputs of a run one per lane and advances the
// wave-uniform state past them.
template <int FMT>
__device__ __forceinline__ void peel_outputs(typename Out<FMT>::T* __restrict__ dst, uint32_t k, uint32_t s[8],
                                             const CoefRecord* __restrict__ lane_rec) {
  const uint32_t lane = threadIdx.x & 63;
  uint32_t any = 0;
#pragma unroll
  for (int j = 0; j < 8; ++j) any |= s[j];
  if (any == 0u) {  // the all-zero state stays zero
    if (lane < k) __builtin_nontemporal_store(convert_zero<FMT>(), dst + lane);
    return;
  }
  const Coef c = load_coef(lane_rec + lane);  // row 0 of A^(lane+1)
  int32_t e[8];
  centre(s, e);
  const uint32_t r = dot_residue(c, e);
  if (lane < k) __builtin_nontemporal_store(convert<FMT>(r), dst + lane);
  // new state: the k new words (newest first) followed by the 8-k oldest kept
  uint32_t ns[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const uint32_t src = (uint32_t)j < k ? k - 1 - (uint32_t)j : 0u;
    const uint32_t fresh = __builtin_amdgcn_readlane(r, src) + 1u;
    uint32_t kept = s[0];
#pragma unroll
    for (int q = 1; q < 8; ++q) kept = (uint32_t)(j - q) == k ? s[q] : kept;  // s[j - k]
    kept = (uint32_t)j == k ? s[0] : kept;
    ns[j] = (uint32_t)j < k ? fresh : kept;
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) s[j] = ns[j];
}

// Byte alignment of the wide-store loop's wave stores: 64 lanes x 16 bytes.
constexpr uintptr_t kStoreAlign = 1024;

// Writes the outputs of a run before its first ALIGN-byte boundary (at most
// 63 per round, one per lane) and advances dst, cnt and the state past them.
// With ALIGN = kStoreAlign every 1 KiB wave store of the loop that follows
// covers whole cache lines: on MI355X a 2^28-double fill whose destination
// was 8 or 16 bytes off such a boundary took 471-473 us with a 16-byte peel,
// 346-350 us with this one (aligned: 342 us).
template <int FMT, uintptr_t ALIGN>
__device__ __forceinline__ void peel_to_boundary(typename Out<FMT>::T*& dst, uint64_t& cnt, uint32_t s[8],
                                                 const CoefRecord* __restrict__ lane_rec) {
  typedef typename Out<FMT>::T T;
  uint64_t b = ((ALIGN - (reinterpret_cast<uintptr_t>(dst) & (ALIGN - 1))) & (ALIGN - 1)) / sizeof(T);
  if (b > cnt) b = cnt;
  while (b) {
    const uint32_t k = b < 63 ? (uint32_t)b : 63u;
    peel_outputs<FMT>(dst, k, s, lane_rec);
    dst += k;
    cnt -= k;
    b -= k;
  }
}

// Generates `cnt` outputs of the stream whose wave-uniform state (at the
// first output) is s, into dst[0..cnt), with this lane's records k (and the
// lane records, for the outputs before the first 1 KiB boundary).  `cnt` and
// s must be wave-uniform; dst need only be element-aligned.
// NARROW (k a variable of the caller) keeps the coefficients 32 bits wide: the
// compiler otherwise widens them ahead of the loop, half of them with a copy
// each.  It frees some 25 registers, which pays where a group's start is waited
// for (address-order grid: batches of less than 2^26 outputs 2 to 5 % faster,
// 17 GB the same) and not where more resident waves loosen the order of the
// stores (2^28 doubles 352 against 320 us, one tile per wave 2 to 3 % slower
// for large batches).
template <int FMT, int PL, uintptr_t ALIGN = kStoreAlign, bool NARROW = false>
__device__ __forceinline__ void generate_run(typename Out<FMT>::T* __restrict__ dst, uint64_t cnt, uint32_t s[8],
                                             const Coef (&k)[PL], const CoefRecord* __restrict__ lane_rec) {
  typedef LaneLayout<FMT, PL> L;
  constexpr int kPer = 64 * PL;
  const uint32_t lane = threadIdx.x & 63;
  uint32_t any = 0;
#pragma unroll
  for (int j = 0; j < 8; ++j) any |= s[j];
  if (any == 0u) {  // degenerate all-zero state
    for (uint64_t i = lane; i < cnt; i += 64) __builtin_nontemporal_store(convert_zero<FMT>(), dst + i);
    return;
  }
  typename Out<FMT>::T* base = dst;
  peel_to_boundary<FMT, ALIGN>(base, cnt, s, lane_rec);
  const uint64_t full = cnt / kPer;
  const uint64_t rem = cnt - full * kPer;
  for (uint64_t it = 0; it < full; ++it) {
    if constexpr (NARROW) {
#pragma unroll
      for (int i = 0; i < PL; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) asm("" : "+v"(const_cast<Coef&>(k[i]).c[j]));
    }
    int32_t e[8];
    centre(s, e);
    uint32_t r[PL];
    dot_residues<PL>(k, e, r);
    store_lane<FMT, PL>(base, lane, r);
    base += kPer;
    // next state: the last eight words, newest first (not needed after the
    // run's last iteration: 8 of 16 readlanes of a 256-output tile at 2 per lane)
    if (it + 1 < full || rem) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        s[j] = __builtin_amdgcn_readlane(r[L::slot_of(kPer - 1 - j)], L::lane_of(kPer - 1 - j)) + 1u;
    }
  }
  if (rem) {
    int32_t e[8];
    centre(s, e);
    uint32_t r[PL];
    dot_residues<PL>(k, e, r);
#pragma unroll
    for (int i = 0; i < PL; ++i) {
      const uint32_t o = L::index(lane, i);
      if (o < rem) __builtin_nontemporal_store(convert<FMT>(r[i]), base + o);
    }
  }
}

// First output of wave w of a fill: wave 0 also takes the head (the outputs
// before the first tile-aligned address), every later wave starts on one.
__device__ __forceinline__ uint64_t fill_first(const FillArgs& a, uint64_t w) { return w ? a.head + w * a.tile : 0; }

// The part of the output that block b of an nb-block grid writes.  The
// dispatcher deals blocks to the XCDs in turn (block b to XCD (b + r) mod x,
// r where its turn stood after earlier launches), so in dispatch order the
// XCDs interleave block by block.  With group g > 1, the blocks of one XCD
// (b mod x alike) instead take runs of g consecutive blocks' output within
// every span of x g blocks, whatever r is.  Blocks past the last whole span
// keep their own part.  Either way every part is written by exactly one
// block.  x and g are powers of two: with divisions this was 60 scalar and 15
// vector operations at the start of every wave, now nine scalar ones.
__device__ __forceinline__ uint64_t xcd_block(uint32_t b, uint32_t nb, uint32_t x, uint32_t g) {
  if (g <= 1) return b;
  const uint32_t lx = __builtin_ctz(x), lg = __builtin_ctz(g), span = lx + lg;
  if (b >= nb >> span << span) return b;
  const uint32_t q = b >> lx;
  return (q >> lg << span) + ((b & (x - 1)) << lg) + (q & (g - 1));
}

// Bound by the store stream for long fills and by the latency of a wave's
// start (rows of its jump, then its lane records) for short ones.  A wave jumps
// its own state, all eight lane groups alike: with the block's states jumped
// by one wave and handed over in LDS behind a barrier, 2^28 doubles took 327
// us against 320 us, 2^26 86 against 82 us (64-thread blocks, 1024 outputs
// per wave).  The lane records are loaded after the jump: loaded before it, or
// between its loads and its products, 2^24 doubles took 25.1 and 24.9 us
// against 24.1 us (2^28: 314 and 316 against 320 us).  Limited to 80
// registers for a sixth wave per SIMD it spills (2^28: 401 us).
// IN_STEP: the waves of a block wait for one another before their outputs (see
// fill_in_step).
template <int FMT, int PL, bool IN_STEP>
__global__ __launch_bounds__(1024) void k_fill(FillArgs a) {
  const uint32_t wib = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform wave index
  const uint32_t nw = blockDim.x >> 6;
  const uint64_t w = xcd_block(blockIdx.x, gridDim.x, a.xcds, a.xcd_group) * nw + wib;
  const uint64_t first = fill_first(a, w);
  if (!IN_STEP && first >= a.n) return;
  const uint64_t cnt = min(a.head + (w + 1) * a.tile, a.n) - first;
  const uint32_t word = jump_uniform(own_word(a.start.state), a.start.offset + first, a.digits);
  if constexpr (IN_STEP) {
    __syncthreads();  // every wave of the block, with outputs or not
    if (first >= a.n) return;
  }
  uint32_t s[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) s[j] = __builtin_amdgcn_readlane(word, j);
  Coef k[PL];
  load_lane_coefs<FMT, PL>(k, a.lane);
  generate_run<FMT, PL>(static_cast<typename Out<FMT>::T*>(a.out) + first, cnt, s, k, a.lane);
}

// One tile of a batch segment at dst (generate_run peels the outputs before
// the first ALIGN-byte boundary; only tile 0 of a segment can have any).  The
// persistent kernel passes ALIGN = 16: with the 1 KiB peel it ran 10 % slower
// on the 4096-stream batch.
template <int FMT, int PL, uintptr_t ALIGN = kStoreAlign, bool NARROW = false>
__device__ __forceinline__ void batch_tile(void* out, uint64_t cnt, uint32_t s[8], const Coef (&k)[PL],
                                           const CoefRecord* __restrict__ lane_rec) {
  if (cnt) generate_run<FMT, PL, ALIGN, NARROW>(static_cast<typename Out<FMT>::T*>(out), cnt, s, k, lane_rec);
}

__device__ __forceinline__ uint64_t readlane_u64(uint64_t v, int lane) {
  const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)v, lane);
  const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(v >> 32), lane);
  return (uint64_t)lo | ((uint64_t)hi << 32);
}

// A device address read from memory as a pointer: known to be global memory,
// so that stores through it are global and not flat, which also count as LDS
// accesses (4096 streams on the address-order grid: 2.601 to 2.591 ms).
__device__ __forceinline__ void* global_pointer(uint64_t address) {
  return (void*)(__attribute__((address_space(1))) void*)address;
}

// The tables of a batch block (see BatchHeader).
struct BatchTables {
  const BatchSegment* segs;
  const uint64_t* tile_begin;
  const uint32_t* tile_seg;
  uint64_t ntiles;
};

__device__ __forceinline__ BatchTables batch_tables(const uint8_t* block) {
  const BatchHeader* hdr = reinterpret_cast<const BatchHeader*>(block);
  BatchTables t;
  t.segs = reinterpret_cast<const BatchSegment*>(block + sizeof(BatchHeader));
  t.tile_begin = reinterpret_cast<const uint64_t*>(block + hdr->tile_begin_off);
  t.tile_seg = reinterpret_cast<const uint32_t*>(block + hdr->tile_seg_off);
  t.ntiles = hdr->ntiles;
  return t;
}

// Destination, output count, stream position and state source of tile t.
struct TileInfo {
  uint64_t dst;
  uint64_t cnt;
  uint64_t offset;
  const uint32_t* state;
  int32_t fmt;
};

__device__ __forceinline__ TileInfo lookup_tile(const BatchTables& tab, const BatchArgs& a, uint64_t t) {
  const uint32_t seg = tab.tile_seg[t];
  const BatchSegment* sp = tab.segs + seg;
  TileInfo ti;
  ti.fmt = sp->format;
  const uint64_t kt = t - tab.tile_begin[seg];  // tile number within the segment
  uint64_t first, end;
  tile_bounds(segment_head(sp->out, ti.fmt, sp->count, a.tile), sp->count, a.tile, kt, &first, &end);
  ti.cnt = end - first;
  ti.dst = reinterpret_cast<uint64_t>(sp->out) + first * (ti.fmt == 2 ? 4u : 8u);
  ti.offset = sp->offset + first;
  const uint32_t sid = sp->stream;
  ti.state = sid == kInlineState ? sp->state : a.states + 8ull * sid;
  return ti;
}

// Persistent batched kernel.  With W waves in the grid, wave w takes tiles
// w, w + W, w + 2W, ...: at any moment the grid writes a window of about W
// consecutive tiles, as a one-tile-per-wave launch would, and equal tiles
// keep the waves in step without any atomic.  A wave looks up its next
// kGroup tiles together (one 8-lane group each: segment, destination, count,
// start state, which the group then jumps) and generates them one after
// another, so a tile starts storing without waiting on memory.
constexpr uint32_t kGroup = 8;

__global__ __launch_bounds__(1024) void k_batch(BatchArgs a) {
  const int lane = threadIdx.x & 63;
  const int grp = lane >> 3;
  const BatchTables tab = batch_tables(a.block);
  const uint64_t ntiles = tab.ntiles;
  const uint64_t nwaves = (uint64_t)gridDim.x * (blockDim.x >> 6);
  const uint64_t wave =
      xcd_block(blockIdx.x, gridDim.x, a.xcds, a.xcd_group) * (blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (wave >= ntiles) return;
  const uint64_t mine_total = (ntiles - wave + nwaves - 1) / nwaves;
  for (uint64_t j0 = 0; j0 < mine_total; j0 += kGroup) {
    const uint32_t ngrp = (uint32_t)min<uint64_t>(kGroup, mine_total - j0);
    const bool mine = (uint32_t)grp < ngrp;
    const TileInfo ti = lookup_tile(tab, a, (j0 + (mine ? grp : 0)) * nwaves + wave);
    const uint32_t s = jump_group(ti.state[lane & 7], mine ? ti.offset : 0, a.digits);
    // loaded after the jumps so that they hold no registers during them
    Coef k[2];
    load_lane_coefs<0, 2>(k, a.lane);  // the PL = 2 layout is the same for every format
    for (uint32_t g = 0; g < ngrp; ++g) {
      uint32_t u[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) u[j] = __builtin_amdgcn_readlane(s, 8 * g + j);
      void* out = global_pointer(readlane_u64(ti.dst, 8 * g));
      const uint64_t ucnt = readlane_u64(ti.cnt, 8 * g);
      switch (__builtin_amdgcn_readlane(ti.fmt, 8 * g)) {
        case 0: batch_tile<0, 2, 16>(out, ucnt, u, k, a.lane); break;
        case 1: batch_tile<1, 2, 16>(out, ucnt, u, k, a.lane); break;
        default: batch_tile<2, 2, 16>(out, ucnt, u, k, a.lane); break;
      }
    }
  }
}

// One tile of a batch with the fill's layout (4 outputs per lane).
template <int FMT, bool NARROW = false>
__device__ __forceinline__ void batch_tile_alone(void* out, uint64_t cnt, uint32_t s[8],
                                                 const CoefRecord* __restrict__ lane_rec) {
  Coef k[4];
  load_lane_coefs<FMT, 4>(k, lane_rec);
  batch_tile<FMT, 4, kStoreAlign, NARROW>(out, cnt, s, k, lane_rec);
}

// Batched kernel with one tile per wave (grid = tiles / waves per block):
// wave 0 of a block looks up and jumps the start states of the block's tiles
// (8-lane groups) and leaves them in LDS; every wave then generates its own
// tile and exits.
__global__ __launch_bounds__(kTileBlockThreads) void k_batch_tiles(BatchArgs a) {
  constexpr int kWaves = kTileBlockThreads / 64;
  __shared__ uint32_t start_state[kWaves][8];
  __shared__ uint64_t start_dst[kWaves], start_cnt[kWaves];
  __shared__ int32_t start_fmt[kWaves];
  const int lane = threadIdx.x & 63;
  const BatchTables tab = batch_tables(a.block);
  const uint32_t wib = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t nw = blockDim.x >> 6;
  // < ntiles: the grid covers the tiles exactly
  const uint64_t tile0 = xcd_block(blockIdx.x, gridDim.x, a.xcds, a.xcd_group) * nw;
  if (wib == 0) {
    const uint32_t target = lane >> 3;
    const bool mine = target < nw && tile0 + target < tab.ntiles;
    const TileInfo ti = lookup_tile(tab, a, mine ? tile0 + target : tile0);
    const uint32_t s = jump_group(ti.state[lane & 7], mine ? ti.offset : 0, a.digits);
    if (mine) start_state[target][lane & 7] = s;
    if (mine && (lane & 7) == 0) {
      start_dst[target] = ti.dst;
      start_cnt[target] = ti.cnt;
      start_fmt[target] = ti.fmt;
    }
  }
  __syncthreads();
  if (tile0 + wib >= tab.ntiles) return;
  uint32_t u[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) u[j] = __builtin_amdgcn_readfirstlane(start_state[wib][j]);
  const uint64_t d = start_dst[wib], c = start_cnt[wib];
  void* out = global_pointer(readlane_u64(d, 0));
  const uint64_t cnt = readlane_u64(c, 0);
  switch (__builtin_amdgcn_readfirstlane(start_fmt[wib])) {
    case 0: batch_tile_alone<0>(out, cnt, u, a.lane); break;
    case 1: batch_tile_alone<1>(out, cnt, u, a.lane); break;
    default: batch_tile_alone<2>(out, cnt, u, a.lane); break;
  }
}

// Persistent batched kernel that takes its work in address order: each block
// works on groups of (waves per block) consecutive tiles as k_batch_tiles
// works on its block's tiles (waves 0-1 look up and jump the group's start
// states and leave them in LDS, every wave generates one tile).  A block's
// first group is its index, every further one the next from a counter in the
// batch block's header, taken while the current group is worked on.  Blocks
// stay resident, but the grid writes its tiles in the order a
// one-tile-per-wave grid is dispatched in.  The counter makes launches of one
// batch block that overlap in time incorrect, which the host prevents.
// The counter's atomics are its cost: some 13 ns each, one after the other.
// With one for every group, waited for before its lookups, and another at
// every block's end, 768 blocks took 20 us for one segment of 2048 doubles
// (now 4.9), 54.8 for 500 of 32768 (31.4) and 139 for 2600 (116).  Striding
// through the groups without a counter: 26.7 and 120 us, and 4013 segments of
// 256 to 2^19 doubles 430 against 375 us.
__global__ __launch_bounds__(1024) void k_batch_queue(BatchArgs a) {
  __shared__ uint32_t start_state[16][8];
  __shared__ uint64_t start_dst[16], start_cnt[16];
  __shared__ int32_t start_fmt[16];
  __shared__ uint32_t group;
  const int lane = threadIdx.x & 63;
  const BatchTables tab = batch_tables(a.block);
  BatchHeader* hdr = reinterpret_cast<BatchHeader*>(const_cast<uint8_t*>(a.block));
  const uint32_t wib = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t nw = blockDim.x >> 6;
  const uint64_t ngroups = (tab.ntiles + nw - 1) / nw;
  for (uint64_t g = blockIdx.x; g < ngroups;) {  // the same value in every wave: the block leaves the loop together
    const uint64_t tile0 = g * nw;
    // read per group: addresses and records held across the loop spill
    const int32_t* digits = opaque(a.digits);
    const CoefRecord* lane_rec = opaque(a.lane);
    const bool takes = ngroups > gridDim.x && threadIdx.x == blockDim.x - 64;
    uint32_t taken = 0;
    if (takes) taken = atomicAdd(&hdr->queue_next, 1u);
    if (wib * 8 < nw) {
      const uint32_t target = wib * 8 + (lane >> 3);
      const bool mine = target < nw && tile0 + target < tab.ntiles;
      const TileInfo ti = lookup_tile(tab, a, mine ? tile0 + target : tile0);
      const uint32_t s = jump_group(ti.state[lane & 7], mine ? ti.offset : 0, digits);
      if (mine) start_state[target][lane & 7] = s;
      if (mine && (lane & 7) == 0) {
        start_dst[target] = ti.dst;
        start_cnt[target] = ti.cnt;
        start_fmt[target] = ti.fmt;
      }
    }
    __syncthreads();
    if (tile0 + wib < tab.ntiles) {
      uint32_t u[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) u[j] = __builtin_amdgcn_readfirstlane(start_state[wib][j]);
      const uint64_t d = start_dst[wib], c = start_cnt[wib];
      void* out = global_pointer(readlane_u64(d, 0));
      const uint64_t cnt = readlane_u64(c, 0);
      switch (__builtin_amdgcn_readfirstlane(start_fmt[wib])) {
        case 0: batch_tile_alone<0, true>(out, cnt, u, lane_rec); break;
        case 1: batch_tile_alone<1, true>(out, cnt, u, lane_rec); break;
        default: batch_tile_alone<2, true>(out, cnt, u, lane_rec); break;
      }
    }
    if (ngroups <= gridDim.x) return;
    if (takes) {
      group = gridDim.x + taken;
      // the grid takes ngroups times: all but the first gridDim.x groups, and
      // once in vain in every block
      if (taken == ngroups - 1) atomicExch(&hdr->queue_next, 0u);
    }
    __syncthreads();  // LDS is rewritten by the next group
    g = group;
  }
}

// ---- bulk advance: many states, offsets of up to kAdvanceWords words --------

__device__ __forceinline__ const int32_t* position_table(const AdvanceArgs& a, int k) {
  return k < kJumpPositions ? a.digits + k * kPositionInts : a.digits_wide + (k - kJumpPositions) * kPositionInts;
}

// The jump of a state that has a zero word (see jump_zero_words).
__device__ __forceinline__ uint32_t advance_zero_words(uint32_t s, const uint32_t* off, const AdvanceArgs& a) {
  for (int k = 0; k < 8 * (int)a.words; ++k) {
    const uint32_t d = digit_of(off[k / 4], k);
    if (__ballot(d != 0u)) s = jump_zero_words(s, d, position_table(a, k));
  }
  return s;
}

// Eight lanes per state, lane r holding word r and computing row r of each
// product; the byte positions of the offset in order, the rows of four
// positions fetched while the four before them are computed (launched back to
// back, 20011 states, 64-bit offsets: 3.8 us, one position ahead 4.3 us; 1000
// states, 256 bits: 5.5 and 8.1 us; alone in a trace 4.4 and 5.8 us).  Positions where
// no state of the wave has a digit are skipped.  A state is read before it is
// written, so `in` and `out` may be the same buffer.
__global__ __launch_bounds__(256) void k_advance(AdvanceArgs a) {
  const int row = threadIdx.x & 7;
  const uint64_t item = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 3;
  const bool live = item < a.n;
  const uint32_t* off = reinterpret_cast<const uint32_t*>(a.offsets) + (live ? item : 0) * 2 * a.words;
  const uint32_t s = live ? a.in[8 * item + row] : 1u;
  uint32_t out;
  if (__ballot(s == 0u)) {
    out = advance_zero_words(s, off, a);
  } else {
    int32_t e = centre_word(s);
    JumpRow m0[4], m1[4];
    uint32_t d0 = off[0], d1 = off[1];
    load_rows4(m0, position_table(a, 0), d0);
    for (uint32_t w = 0; w < a.words; ++w) {
      load_rows4(m1, position_table(a, 8 * w + 4), d1);
      e = apply_rows4(m0, d0, e);
      const uint32_t da = d1;
      if (w + 1 < a.words) {
        d0 = off[2 * w + 2];
        d1 = off[2 * w + 3];
        load_rows4(m0, position_table(a, 8 * w + 8), d0);
      }
      e = apply_rows4(m1, da, e);
    }
    out = word_of(e);
  }
  if (live) a.out[8 * item + row] = out;
}

// The same jumps with each position's 256 matrices (64 KB) staged in LDS by
// the block: 256 x G states, G per group of four lanes, take one position
// together while the next one's matrices are copied to the other buffer
// (global-to-LDS loads, no registers; two arrays, so that reads of one wait
// for no copy into the other).  From memory, each state and digit costs 256
// bytes of L2 and L1 traffic, which bounds k_advance at large n; here that is
// 64 KB per block and position, and the step is bound by its 18 64-bit
// multiply-adds and 16 other VALU operations per two rows.
// Lane r of a group holds words r and r + 4 and computes both rows, so it
// reaches the other six words with six quad permutations for two rows (seven
// for one with eight lanes per state).  Odd groups keep the two words in the
// other order, so that neighbouring groups read different halves of a matrix
// (all four 64-byte quarters in turn would remove the LDS bank conflicts
// left, at four more operations a step: measured the same).
// 2^20 states, 200-bit offsets: see advance_states_per_group.
constexpr int kAdvanceGroups = 256;  // groups of four lanes in a block

struct JumpPair {  // rows of a lane's first and second word: entries for the words held alike, and for the other ones
  u4_t near0, far0, near1, far1;
};

__device__ __forceinline__ void mad4(uint64_t& v, const u4_t& c, const uint32_t w[4]) {
#pragma unroll
  for (int k = 0; k < 4; ++k) v += (uint64_t)((int64_t)(int32_t)c[k] * (int64_t)(int32_t)w[k]);
}

__device__ __forceinline__ void gather_quad(uint32_t v, uint32_t w[4]) {
  w[0] = v;
  w[1] = dpp<0xB1>(v);
  w[2] = dpp<0x4E>(v);
  w[3] = dpp<0x1B>(v);
}

template <int G>
__global__ __launch_bounds__(4 * kAdvanceGroups) void k_advance_lds(AdvanceArgs a) {
  constexpr int kThreads = 4 * kAdvanceGroups, kStates = kAdvanceGroups * G;
  constexpr int kNoLoads = 0x0f70;  // s_waitcnt vmcnt(0)
  __shared__ __attribute__((aligned(1024))) int32_t table0[kPositionInts], table1[kPositionInts];
  __shared__ uint32_t used;
  const uint32_t tid = threadIdx.x, grp = tid >> 2, r = tid & 3, odd = grp & 1;
  const uint32_t word0 = r + 4 * odd, word1 = r + 4 * (odd ^ 1);
  const uint64_t first = (uint64_t)blockIdx.x * kStates;
  const uint32_t count = (uint32_t)min((uint64_t)kStates, a.n - first);
  const uint32_t halves = 2 * a.words;  // an offset as 32-bit halves
  const uint32_t* const in = a.in + 8 * first;
  uint32_t* const out = a.out + 8 * first;
  const uint32_t* const offs = reinterpret_cast<const uint32_t*>(a.offsets) + first * halves;
  auto state = [&](int g) { return min(grp + kAdvanceGroups * g, count - 1); };  // past the end: the last one again
  // copies position k's matrices to LDS, 4 KiB per wave
  auto stage = [&](int k, int32_t* table) {
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int kInts = kPositionInts / (kThreads / 64);
    const int32_t* src = position_table(a, k) + wave * kInts + 4 * (tid & 63);
#pragma unroll
    for (int i = 0; i < kInts / 256; ++i)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + 256 * i),
                                       (__attribute__((address_space(3))) void*)&table[wave * kInts + 256 * i], 16, 0, 0);
  };
  if (tid == 0) used = 0u;
  uint32_t zero = 0;  // bit g: this group's state g has a zero word
  int32_t e0[G], e1[G];
  {
    uint32_t s0[G], s1[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      s0[g] = in[8 * state(g) + word0];
      s1[g] = in[8 * state(g) + word1];
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
      zero |= s0[g] == 0u || s1[g] == 0u ? 1u << g : 0u;
      e0[g] = centre_word(s0[g]);
      e1[g] = centre_word(s1[g]);
    }
    zero |= dpp<0xB1>(zero);
    zero |= dpp<0x4E>(zero);
  }
  // byte positions at which some offset of the block has a digit
  uint32_t mine = 0;
  for (uint32_t i = tid; i < count * halves; i += kThreads) {
    const uint32_t h = offs[i], q = i % halves;
#pragma unroll
    for (int b = 0; b < 4; ++b) mine |= digit_of(h, b) ? 1u << (4 * q + b) : 0u;
  }
#pragma unroll
  for (int d = 1; d < 64; d *= 2) mine |= __shfl_xor(mine, d);
  __syncthreads();
  if ((tid & 63) == 0) atomicOr(&used, mine);
  __syncthreads();
  uint32_t todo = __builtin_amdgcn_readfirstlane(used);
  uint64_t base = kJumpBase;
  asm("" : "+v"(base));  // in vector registers: the first multiply-add's addend
  uint32_t half[G];
  auto fetch_half = [&](int q) {
#pragma unroll
    for (int g = 0; g < G; ++g) half[g] = offs[state(g) * halves + (uint32_t)q];
  };
  // takes position k from `table` while position `next` is copied to `other`
  auto position = [&](int k, int next, const int32_t* table, int32_t* other) {
    if (next >= 0) stage(next, other);
    const uint32_t m0 = 16 * word0, m1 = 16 * word1;
    const uint32_t sel = 0x03020000u + ((4u + (uint32_t)(k & 3)) << 8);  // the digit goes into bits 8..15
    auto rows = [&](uint32_t digits) {
      const uint8_t* t = reinterpret_cast<const uint8_t*>(table);
      const uint8_t* p0 = t + __builtin_amdgcn_perm(digits, m0, sel);
      const uint8_t* p1 = t + __builtin_amdgcn_perm(digits, m1, sel);
      return JumpPair{*reinterpret_cast<const u4_t*>(p0), *reinterpret_cast<const u4_t*>(p0 + 128),
                      *reinterpret_cast<const u4_t*>(p1), *reinterpret_cast<const u4_t*>(p1 + 128)};
    };
    JumpPair cur = rows(half[0]);
#pragma unroll
    for (int g = 0; g < G; ++g) {
      JumpPair ahead{};
      if (g + 1 < G) ahead = rows(half[g + 1]);
      uint32_t w0[4], w1[4];
      gather_quad((uint32_t)e0[g], w0);
      gather_quad((uint32_t)e1[g], w1);
      uint64_t v0 = base, v1 = base;
      mad4(v0, cur.near0, w0);
      mad4(v1, cur.near1, w1);
      mad4(v0, cur.far0, w1);
      mad4(v1, cur.far1, w0);
      e0[g] = reduce_centred(v0);
      e1[g] = reduce_centred(v1);
      cur = ahead;
    }
    if (next >= 0 && next / 4 != k / 4) fetch_half(next / 4);
    __builtin_amdgcn_s_waitcnt(kNoLoads);  // this wave's part of the next matrices is in LDS
    __syncthreads();
  };
  if (todo) {
    int k = __builtin_ctz(todo);
    todo &= todo - 1;
    stage(k, table0);
    fetch_half(k / 4);
    __builtin_amdgcn_s_waitcnt(kNoLoads);
    __syncthreads();
    for (;;) {
      int next = todo ? __builtin_ctz(todo) : -1;
      todo &= todo - 1;
      position(k, next, table0, table1);
      if (next < 0) break;
      k = next;
      next = todo ? __builtin_ctz(todo) : -1;
      todo &= todo - 1;
      position(k, next, table1, table0);
      if (next < 0) break;
      k = next;
    }
  }
#pragma unroll
  for (int g = 0; g < G; ++g)
    if (grp + kAdvanceGroups * g < count && !((zero >> g) & 1u)) {
      out[8 * state(g) + word0] = word_of(e0[g]);
      out[8 * state(g) + word1] = word_of(e1[g]);
    }
  // states with a zero word, eight lanes each: the two groups of four in turn
#pragma unroll 1
  for (int g = 0; g < 2 * G; ++g) {
    const int src = (int)((tid & 0x38u) | (g & 1 ? 4u : 0u)) * 4;  // a lane of the group that owns the state
    const bool theirs = (uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)(zero >> (g / 2))) & 1u;
    const uint32_t at = (grp & ~1u) + (g & 1) + kAdvanceGroups * (g / 2);
    const bool mine_zero = theirs && at < count;
    if (!__ballot(mine_zero)) continue;
    const uint32_t i = mine_zero ? at : 0;
    const uint32_t z = advance_zero_words(mine_zero ? in[8 * i + (tid & 7)] : 1u, offs + i * halves, a);
    if (mine_zero) out[8 * i + (tid & 7)] = z;
  }
}

// Staging copy of a batch block: the host writes the block into coherent
// pinned memory and this kernel moves it to device memory (16 bytes per
// thread, then 4-byte words for the tail).  On MI355X the runtime's
// host-to-device copy of these few kilobytes occasionally blocked the
// calling thread for 6-7 ms, where a kernel launch returns in microseconds.
__global__ __launch_bounds__(256) void k_stage(const u4_t* __restrict__ src, u4_t* __restrict__ dst, uint64_t n16,
                                                uint64_t tail_words) {
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n16) dst[i] = src[i];
  if (i < tail_words)
    reinterpret_cast<uint32_t*>(dst + n16)[i] = reinterpret_cast<const uint32_t*>(src + n16)[i];
}

// ---- matrix-core fill ---------------------------------------------------------
//
// A tile of 16 COL consecutive outputs is cut into 16 columns of COL (64
// or 128); column c starts from its own state (its 8 preceding words)
// and one step makes its next 16 outputs.  Output j of a step (j < 16) is
// dot(R_j, w) for the column's state w (oldest word first), with R_j the
// block rows.  In exact integers mod p:
//   * each state word is centred, e = w - 2^30, and cut into four balanced
//     base-256 digits e = sum_b 2^(8b) d_b (d_b in [-128, 127]);
//   * M_b = 2^(8b) R_j mod p (centred) is cut the same way,
//     M_b = sum_a 2^(8a) m_(b,a), so that
//     dot(R_j, e) == sum_a 2^(8a) sum_(q,b) m_(b,a)[q] d_b[q]  (mod p):
//     four int8 products of K = 8 words x 4 digits = 32, one per class a,
//     v_mfma_i32_16x16x32_i8 with the step's rows as M, the columns as N;
//   * the accumulators start from per-row constants (the C operand) that
//     carry the 2^30 sum R_j, the reference's -1 and the biases, so that
//     t = C_0 + 2^8 C_1 and u = C_2 + 2^8 C_3 are non-negative and below
//     2^29, and x = t + ((u << 16) & p) + (u >> 15) (2^16 u mod p is a 31-bit
//     rotation) is the residue plus at most one p: five 32-bit operations
//     per output (mfma_step_residue).  2^28 words: 171 us, 176 us with eight.
// MFMA layouts (gfx950; the fill's parity tests depend on them): lane
// l = n + 16 g holds the 8 bytes of K-group g for row/column n, and result
// register i of lane l is row 4 g + i of column n.  K-group g, byte i is word W(g) + i / 4, digit
// i % 4, with W = (0, 4, 2, 6); row 4 g + i is step position 2 g + i for
// i < 2 and 8 + W(g) + i - 2 for i >= 2.  So the step's last eight outputs
// (positions 8..15, the column's next state) are registers 2 and 3 of
// exactly the lanes whose K-group needs them: no lane exchange.
// A wave makes a few consecutive tiles (up to 32 KiB of output: the store
// pattern of short-lived waves in address order, which persistent waves
// striding over the tiles, with a product by A^(2048 waves) from one to the
// next, do not match: 192-217 against 170 us for 2^28 words, 371-480 against
// 325 us for doubles).  The 16 column states of the wave's next tile are the current
// ones times A^2048: one more product of the same form, whose rows put the
// new words in registers 0 and 1 of the lanes that need them.  Only a
// wave's first tile computes its column states from the tile state (the
// fan-out records).  Registers stay below 128 and the tile's staging below
// 8.5 KiB, so four waves per SIMD are resident.
// The outputs of a tile are staged in LDS (16 columns x 132 words per wave)
// and leave as the vector kernel's 1 KiB wave stores in address order.

typedef int32_t v4i_t __attribute__((ext_vector_type(4)));


// Balanced base-256 digits of w - 2^30 (w < 2^31), one per byte.
__device__ __forceinline__ uint32_t mfma_digits(uint32_t w) { return (w + 0x40808080u) ^ 0x80808080u; }

__device__ __forceinline__ long mfma_operand(uint32_t w0, uint32_t w1) {
  return (long)((uint64_t)mfma_digits(w0) | ((uint64_t)mfma_digits(w1) << 32));
}

__device__ __forceinline__ uint64_t mad_u64_u32(uint32_t a, uint32_t b, uint64_t c) {
  uint64_t w, carry;
  asm("v_mad_u64_u32 %0, %1, %2, %3, %4" : "=v"(w), "=s"(carry) : "v"(a), "s"(b), "v"(c));
  return w;
}

// Residue in [0, p) of a step output (result register i of the four classes,
// accumulators started from the step constants, class 2 taken twice): with
// u = C_2 + 2^8 C_3, acc[2] + 2^9 acc[3] is 2 u, whose 16-bit halves are
// 2 (u mod 2^15) and u >> 15, so one two-term dot product with (2^15, 1) adds
// 2^16 u mod p, the 31-bit rotation of u, to t.  Five operations an output
// (eight with the rotation from shifts and a mask).
typedef unsigned short us2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t mfma_step_residue(const v4i_t (&acc)[kMfmaClasses], int i) {
  const uint32_t t = (uint32_t)acc[0][i] + ((uint32_t)acc[1][i] << 8);   // [0, 2 beta + 2^16)
  const uint32_t u2 = (uint32_t)acc[2][i] + ((uint32_t)acc[3][i] << 9);  // 2 u, u in [0, 2 beta + 2^15)
  const uint32_t x = __builtin_amdgcn_udot2(__builtin_bit_cast(us2_t, u2), us2_t{1u << 15, 1}, t, false);  // < 2 p
  return min(x, x - kP);
}

// The products of a step: class 2 twice (see mfma_step_residue); C0 holds the
// step constants with class 2's doubled.
__device__ __forceinline__ void mfma_step(v4i_t (&acc)[kMfmaClasses], const long (&A)[kMfmaClasses],
                                          const v4i_t (&C0)[kMfmaClasses], long B) {
#pragma unroll
  for (int q = 0; q < kMfmaClasses; ++q) acc[q] = __builtin_amdgcn_mfma_i32_16x16x32_i8(A[q], B, C0[q], 0, 0, 0);
  acc[2] = __builtin_amdgcn_mfma_i32_16x16x32_i8(A[2], B, acc[2], 0, 0, 0);
}

// Residue in [0, p) of a stride output (accumulators started from 0, k in
// [kMfmaBeta, kMfmaBeta + p)).
__device__ __forceinline__ uint32_t mfma_stride_residue(const v4i_t (&acc)[kMfmaClasses], int i, uint32_t k) {
  const uint32_t t = (uint32_t)acc[0][i] + ((uint32_t)acc[1][i] << 8);              // [-beta, beta]
  const uint32_t u = (uint32_t)acc[2][i] + ((uint32_t)acc[3][i] << 8) + kMfmaBeta;  // [0, 2 beta]
  const uint64_t y = mad_u64_u32(u, 65536u, (uint64_t)(t + k));                    // < 2^45
  const uint32_t x = ((uint32_t)y & kP) + (uint32_t)(y >> 31);                      // < 2^31 + 2^14
  return min(x, x - kP);
}

// Between a wave's writes to LDS and its lanes' reads of one another's words,
// and between those reads and the next writes.  A wave's LDS operations take
// effect in the order of the program; this keeps the compiler to that order
// and is no instruction.
__device__ __forceinline__ void wave_lds_handover() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// The tiles [t0, t0 + nt) of a matrix-core fill with columns of COL outputs,
// made by one wave with the LDS area st (kMfmaColumns * (COL + 4) words: the
// 4-word pad spreads the columns over the LDS banks).
template <int FMT, int COL>
__device__ __forceinline__ void mfma_tiles(const MfmaFillArgs& a, uint64_t t0, uint32_t nt, uint32_t* st) {
  typedef typename Out<FMT>::T T;
  constexpr int kTile = kMfmaColumns * COL;
  constexpr int kStride = COL + 4;  // LDS words per column
  constexpr int kSteps = COL / 16;
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t n = lane & 15, g = lane >> 4;
  const uint32_t wg = (g & 1) * 4 + (g >> 1) * 2;  // W(g): first word of this K-group
  long A[kMfmaClasses];
  v4i_t C0[kMfmaClasses];
#pragma unroll
  for (int q = 0; q < kMfmaClasses; ++q) {
    A[q] = reinterpret_cast<const long*>(a.mfma_a)[q * 64 + lane];
    C0[q] = reinterpret_cast<const v4i_t*>(a.mfma_c)[q * 4 + g];
  }
  C0[2] *= 2;
  long AJ[kMfmaClasses] = {};
  u2_t KJ = {};
  if (nt > 1) {
#pragma unroll
    for (int q = 0; q < kMfmaClasses; ++q) AJ[q] = reinterpret_cast<const long*>(a.mfma_next_a)[q * 64 + lane];
    KJ = reinterpret_cast<const u2_t*>(a.mfma_next_k)[g];
  }
  // the first tile's column states: words W(g), W(g) + 1 (oldest first) of
  // column n are the tile's outputs 128 n - 8 + q, from the tile state
  long B;
  {
    const uint32_t word = jump_uniform(own_word(a.start.state), a.start.offset + a.head + t0 * kTile, a.digits);
    uint32_t s[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) s[j] = __builtin_amdgcn_readlane(word, j);
    Coef k2[2];
    const CoefRecord* fan = a.mfma_fan + (n ? n - 1 : 0) * 8 + wg;  // outputs COL n - 8 + q
    k2[0] = load_coef(fan);
    k2[1] = load_coef(fan + 1);
    int32_t e[8];
    centre(s, e);
    uint32_t r[2];
    dot_residues<2>(k2, e, r);
    // column 0 starts from the tile state itself: word q is s[7 - q]
    uint32_t s0 = s[7], s1 = s[6];
#pragma unroll
    for (int q = 2; q < 8; q += 2) {
      s0 = wg == (uint32_t)q ? s[7 - q] : s0;
      s1 = wg == (uint32_t)q ? s[6 - q] : s1;
    }
    B = mfma_operand(n ? r[0] + 1u : s0, n ? r[1] + 1u : s1);
  }

  // A tile's outputs go through LDS into this lane's slice of its 1 KiB wave
  // stores (pend: 32 residues, chunk ch = this lane's part of store ch), and
  // the stores leave during the next tile's steps, kChunks / kSteps per step,
  // so that every wave keeps writing while it computes.
  constexpr int kChunks = kTile * (int)sizeof(T) / 1024;  // 1 KiB stores per tile
  constexpr int kPer = 1024 / (64 * (int)sizeof(T));      // outputs per lane per store
  static_assert(kChunks % kSteps == 0 && COL % kPer == 0, "tile shape");
  uint32_t pend[kChunks * kPer];
  T* pend_base = nullptr;
  auto store_chunk = [&](int ch) {
    if constexpr (FMT == 2) {
      const u4_t o = {pend[4 * ch] + 1u, pend[4 * ch + 1] + 1u, pend[4 * ch + 2] + 1u, pend[4 * ch + 3] + 1u};
      __builtin_nontemporal_store(o, reinterpret_cast<u4_t*>(pend_base + 256 * ch + 4 * lane));
    } else {
      const d2_t o = {convert<FMT>(pend[2 * ch]), convert<FMT>(pend[2 * ch + 1])};
      __builtin_nontemporal_store(o, reinterpret_cast<d2_t*>(pend_base + 128 * ch + 2 * lane));
    }
  };
  uint32_t* const col = st + n * kStride;
  for (uint32_t t = 0; t < nt; ++t) {
    const long B0 = B;
#pragma unroll
    for (int step = 0; step < kSteps; ++step) {
      v4i_t acc[kMfmaClasses];
      mfma_step(acc, A, C0, B);
      uint32_t r[4];
#pragma unroll
      for (int i = 3; i >= 0; --i) r[i] = mfma_step_residue(acc, i);  // registers 2, 3 first: the next operand
      if (step + 1 < kSteps) B = mfma_operand(r[2] + 1u, r[3] + 1u);
      *reinterpret_cast<u2_t*>(col + 16 * step + 2 * g) = u2_t{r[0], r[1]};
      *reinterpret_cast<u2_t*>(col + 16 * step + 8 + wg) = u2_t{r[2], r[3]};
      if (t) {
#pragma unroll
        for (int k = 0; k < kChunks / kSteps; ++k) store_chunk(step * (kChunks / kSteps) + k);
      }
    }
    // the next tile's column states: A^(16 COL) times this tile's (register
    // i < 2 of this lane: word W(g) + i)
    if (t + 1 < nt) {
      v4i_t acc[kMfmaClasses];
#pragma unroll
      for (int q = 0; q < kMfmaClasses; ++q)
        acc[q] = __builtin_amdgcn_mfma_i32_16x16x32_i8(AJ[q], B0, v4i_t{}, 0, 0, 0);
      B = mfma_operand(mfma_stride_residue(acc, 0, KJ.x) + 1u, mfma_stride_residue(acc, 1, KJ.y) + 1u);
    }
    // this tile's slice of every store: tile outputs ch E + kPer lane .. + kPer - 1
    // (E = 1024 / sizeof(T) per store), within one column
    wave_lds_handover();
#pragma unroll
    for (int ch = 0; ch < kChunks; ++ch) {
      const uint32_t pos = ch * (1024 / (int)sizeof(T)) + kPer * lane;
      const uint32_t* src = st + (pos / COL) * kStride + pos % COL;
      if constexpr (FMT == 2) {
        const u4_t v = *reinterpret_cast<const u4_t*>(src);
        pend[4 * ch] = v.x; pend[4 * ch + 1] = v.y; pend[4 * ch + 2] = v.z; pend[4 * ch + 3] = v.w;
      } else {
        const u2_t v = *reinterpret_cast<const u2_t*>(src);
        pend[2 * ch] = v.x; pend[2 * ch + 1] = v.y;
      }
    }
    wave_lds_handover();
    pend_base = static_cast<T*>(a.out) + a.head + (t0 + t) * kTile;
  }
#pragma unroll
  for (int ch = 0; ch < kChunks; ++ch) store_chunk(ch);
}

// Matrix-core fill: waves [0, a.waves) make tiles, the next a.extra waves
// the short runs before the first tile and after the last with the vector
// kernel's loop.
template <int FMT, int COL, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void k_fill_mfma(MfmaFillArgs a) {
  __shared__ uint32_t stage[WAVES][kMfmaColumns * (COL + 4)];
  const uint32_t wib = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint64_t w = xcd_block(blockIdx.x, gridDim.x, a.xcds, a.xcd_group) * WAVES + wib;
  if (w < a.waves) {
    const uint64_t t0 = w * a.tiles_per_wave;
    mfma_tiles<FMT, COL>(a, t0, (uint32_t)min((uint64_t)a.tiles_per_wave, a.tiles - t0), stage[wib]);
    return;
  }
  const uint64_t e = w - a.waves;
  if (e >= a.extra) return;
  const uint64_t first = a.extra_first[e], cnt = a.extra_count[e];
  const uint32_t word = jump_uniform(own_word(a.start.state), a.start.offset + first, a.digits);
  uint32_t s[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) s[j] = __builtin_amdgcn_readlane(word, j);
  Coef k[4];
  load_lane_coefs<FMT, 4>(k, a.lane);
  generate_run<FMT, 4>(static_cast<typename Out<FMT>::T*>(a.out) + first, cnt, s, k, a.lane);
}

// Persistent batched kernel for short tiles: a wave takes eight tiles at once,
// eight lanes looking up and jumping each, and generates them together with
// the matrix cores in sixteen columns: 256 outputs of every tile a run, the
// two halves from the tile's state and from A^128 times it, 16 outputs of
// every column a step (see the matrix-core fill).  A run goes through LDS and
// leaves tile by tile.  In the vector kernel a short tile is mostly start:
// eight lane broadcasts and two chains of eight multiply-adds, one tile after
// the other, and nothing left to store when the next jumps wait for memory.
// Here the next group is looked up before the current one's steps and jumped
// before its stores (loads wait for all earlier stores), and what is left is
// bound by the issue of the jumps' 64-bit multiply-adds and the residues.
// Not kept: sixteen tiles in columns of their own with four lanes jumping each
// (65536 x 256 words 20.8 us, but 2048 x 256 13.3 and 32768 x 512 30); halves
// of fewer than 128 outputs where a tile needs no more (the rows then wait for
// the lookup: 131072 x 256 words 42.7 against 40.4).
// Which batches take it: see batch_kernel.
constexpr uint32_t kShortGroup = 8;
constexpr int kShortRun = kBatchSkip, kShortStride = kShortRun + 4;  // outputs of a column in a run, its LDS words

// A run of a tile of cnt outputs from its output `done` on, the tile's two
// columns at `col` and 8 columns on: four outputs a lane.
struct RunWords {
  uint32_t w[4];
};

template <int FMT>
__device__ __forceinline__ uint32_t run_output(int i) {  // first output of this lane's pair i (of 2)
  return FMT == 2 ? 4 * threadIdx.x + 2 * i : kShortRun * i + 2 * threadIdx.x;
}

template <int FMT>
__device__ __forceinline__ RunWords read_run(const uint32_t* col) {
  if constexpr (FMT == 2) {  // four consecutive outputs
    const u4_t v = *reinterpret_cast<const u4_t*>(col + (threadIdx.x >> 5) * (8 * kShortStride) + 4 * (threadIdx.x & 31));
    return RunWords{{v.x, v.y, v.z, v.w}};
  } else {  // two of each half, so that each store of the wave is contiguous
    const u2_t a = *reinterpret_cast<const u2_t*>(col + 2 * threadIdx.x);
    const u2_t b = *reinterpret_cast<const u2_t*>(col + 8 * kShortStride + 2 * threadIdx.x);
    return RunWords{{a.x, a.y, b.x, b.y}};
  }
}

template <int FMT>
__device__ __forceinline__ void store_run(void* out, uint64_t done, uint64_t cnt, const RunWords& r, bool zero) {
  typedef typename Out<FMT>::T T;
  typedef T pair_t __attribute__((ext_vector_type(2), aligned(sizeof(T))));
  typedef T quad_t __attribute__((ext_vector_type(4), aligned(sizeof(T))));
  T v[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = zero ? convert_zero<FMT>() : convert<FMT>(r.w[i]);
  T* const p = static_cast<T*>(out) + done;
  const uint64_t left = cnt - done;
  if (FMT == 2 && run_output<FMT>(1) + 1 < left) {
    __builtin_nontemporal_store(quad_t{v[0], v[1], v[2], v[3]}, reinterpret_cast<quad_t*>(p + run_output<FMT>(0)));
    return;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const uint32_t o = run_output<FMT>(i);
    if (o + 1 < left) __builtin_nontemporal_store(pair_t{v[2 * i], v[2 * i + 1]}, reinterpret_cast<pair_t*>(p + o));
    else if (o < left) __builtin_nontemporal_store(v[2 * i], p + o);
  }
}

// A run of every tile of a group: tiles of one format, none with the all-zero
// state, the LDS reads first.
template <int FMT>
__device__ __forceinline__ void store_runs(const TileInfo& ti, uint32_t ngrp, uint64_t done, const uint32_t* stage) {
  RunWords v[kShortGroup];
#pragma unroll
  for (int t = 0; t < (int)kShortGroup; ++t) v[t] = read_run<FMT>(stage + t * kShortStride);
#pragma unroll
  for (int t = 0; t < (int)kShortGroup; ++t) {
    const uint64_t cnt = (uint32_t)t < ngrp ? readlane_u64(ti.cnt, 8 * t) : 0;
    if (done < cnt) store_run<FMT>(global_pointer(readlane_u64(ti.dst, 8 * t)), done, cnt, v[t], false);
  }
}

__global__ __launch_bounds__(64) void k_batch_short(BatchArgs a) {
  __shared__ __attribute__((aligned(16))) uint32_t stage[kMfmaColumns * kShortStride];
  const uint32_t lane = threadIdx.x, n = lane & 15, g = lane >> 4;
  const uint32_t wg = (g & 1) * 4 + (g >> 1) * 2;  // W(g), as in mfma_tiles
  const uint32_t grp = lane >> 3;
  const BatchTables tab = batch_tables(a.block);
  const uint64_t ntiles = tab.ntiles;
  // Full rounds of one group a wave, then one of as many waves as there are
  // full groups left, but enough of them to reach every SIMD (65536 x 16 words
  // 16.2 us; with equal rounds of fewer waves, uneven over the SIMDs, 17.7).
  const uint32_t waves = gridDim.x, wave = blockIdx.x;
  const uint64_t round = (uint64_t)kShortGroup * waves, rounds = ntiles / round;
  const uint32_t last = (uint32_t)(ntiles - rounds * round);  // its tiles
  const uint32_t last_waves = max((last + kShortGroup - 1) / kShortGroup, min(a.min_waves, min(last, waves)));
  auto group_size = [&](uint64_t r) {
    if (r < rounds) return kShortGroup;
    return r == rounds && wave < last_waves ? (last - wave + last_waves - 1) / last_waves : 0u;
  };
  auto lookup = [&](uint64_t r) {
    const uint32_t in_group = grp < group_size(r) ? grp : 0;
    return lookup_tile(tab, a, r * round + (uint64_t)in_group * (r < rounds ? waves : last_waves) + wave);
  };
  if (group_size(0) == 0) return;
  long A[kMfmaClasses];
  v4i_t C0[kMfmaClasses];
#pragma unroll
  for (int q = 0; q < kMfmaClasses; ++q) {
    A[q] = reinterpret_cast<const long*>(a.mfma_a)[q * 64 + lane];
    C0[q] = reinterpret_cast<const v4i_t*>(a.mfma_c)[q * 4 + g];
  }
  const JumpRow second = load_row(a.digits + kShortRun * kJumpMatrixInts + 4 * (lane & 7));  // A^128
  uint32_t ngrp = group_size(0);
  TileInfo ti = lookup(0);
  uint32_t s = jump_group(ti.state[lane & 7], grp < ngrp ? ti.offset : 0, a.digits);
  for (uint64_t r = 0; ngrp != 0; ++r) {
    const bool mine = grp < ngrp;
    const uint32_t s2 = word_of(jump_row(second, centre_word(s)));
    const uint32_t nnext = group_size(r + 1);
    TileInfo tn = ti;
    uint32_t sn = 0;
    if (nnext) {
      tn = lookup(r + 1);
      sn = tn.state[lane & 7];
    }
    const uint64_t alive = __ballot(s != 0u);  // a tile's eight bits are 0: the all-zero state
    const int32_t fmt = __builtin_amdgcn_readfirstlane(ti.fmt);
    const bool plain = __ballot(((alive >> (lane & 56)) & 255u) == 0 || ti.fmt != fmt) == 0;
    uint64_t most = mine ? ti.cnt : 0;
#pragma unroll
    for (int d = 8; d < 64; d *= 2) most = max(most, (uint64_t)__shfl_xor((unsigned long long)most, d));
    most = readlane_u64(most, 0);
    // column n (tile n mod 8, half n / 8): words W(g), W(g) + 1, oldest first
    long B;
    {
      const int hi = (int)(4 * (8 * (n & 7) + 7 - wg)), lo = hi - 4;
      auto from = [](int at, uint32_t v) { return (uint32_t)__builtin_amdgcn_ds_bpermute(at, (int)v); };
      const uint32_t h0 = from(hi, s), h1 = from(hi, s2), l0 = from(lo, s), l1 = from(lo, s2);
      B = mfma_operand(n & 8 ? h1 : h0, n & 8 ? l1 : l0);
    }
    if (r == 0) C0[2] *= 2;  // not before the jump's loads are issued
    uint32_t* const col = stage + n * kShortStride;
    for (uint64_t done = 0;;) {
      const int steps = (int)min<uint64_t>(kShortRun / 16, (most - done + 15) / 16);
#pragma unroll
      for (int step = 0; step < kShortRun / 16; ++step) {
        if (step >= steps) break;
        v4i_t acc[kMfmaClasses];
        mfma_step(acc, A, C0, B);
        uint32_t x[4];
#pragma unroll
        for (int i = 3; i >= 0; --i) x[i] = mfma_step_residue(acc, i);
        B = mfma_operand(x[2] + 1u, x[3] + 1u);
        *reinterpret_cast<u2_t*>(col + 16 * step + 2 * g) = u2_t{x[0], x[1]};
        *reinterpret_cast<u2_t*>(col + 16 * step + 8 + wg) = u2_t{x[2], x[3]};
      }
      // the next group's jumps before this run's stores: they would wait for them
      if (done == 0 && nnext) sn = jump_group(sn, grp < nnext ? tn.offset : 0, a.digits);
      wave_lds_handover();
      if (plain) {
        switch (fmt) {
          case 0: store_runs<0>(ti, ngrp, done, stage); break;
          case 1: store_runs<1>(ti, ngrp, done, stage); break;
          default: store_runs<2>(ti, ngrp, done, stage); break;
        }
      } else {
        for (uint32_t t = 0; t < ngrp; ++t) {
          const uint64_t cnt = readlane_u64(ti.cnt, 8 * t);
          if (done >= cnt) continue;
          void* out = global_pointer(readlane_u64(ti.dst, 8 * t));
          const bool zero = ((alive >> (8 * t)) & 255u) == 0;
          const uint32_t* src = stage + t * kShortStride;
          switch (__builtin_amdgcn_readlane(ti.fmt, 8 * t)) {
            case 0: store_run<0>(out, done, cnt, read_run<0>(src), zero); break;
            case 1: store_run<1>(out, done, cnt, read_run<1>(src), zero); break;
            default: store_run<2>(out, done, cnt, read_run<2>(src), zero); break;
          }
        }
      }
      wave_lds_handover();
      done += 2 * kShortRun;
      if (done >= most) break;
      // every column is at its other half's end of this run: A^128 once more
      v4i_t acc[kMfmaClasses];
#pragma unroll
      for (int q = 0; q < kMfmaClasses; ++q)
        acc[q] = __builtin_amdgcn_mfma_i32_16x16x32_i8(reinterpret_cast<const long*>(a.mfma_skip_a)[q * 64 + lane], B,
                                                       v4i_t{}, 0, 0, 0);
      const u2_t K = reinterpret_cast<const u2_t*>(a.mfma_skip_k)[g];
      B = mfma_operand(mfma_stride_residue(acc, 0, K.x) + 1u, mfma_stride_residue(acc, 1, K.y) + 1u);
    }
    ti = tn;
    s = sn;
    ngrp = nnext;
  }
}

template <int FMT, int PL>
hipError_t fill_one(const FillArgs& a, int block_threads, bool in_step, hipStream_t stream) {
  if (a.n == 0) return hipSuccess;
  const uint64_t waves = fill_waves(a.n, a.head, a.tile);
  const uint64_t wpb = (uint64_t)block_threads / 64;
  const uint64_t blocks = (waves + wpb - 1) / wpb;
  if (blocks * (uint64_t)block_threads > 0xffffffffull) return hipErrorInvalidConfiguration;  // 32-bit grid
  if constexpr (FMT != 2) {
    if (in_step) {
      hipLaunchKernelGGL((k_fill<FMT, PL, true>), dim3((uint32_t)blocks), dim3(block_threads), 0, stream, a);
      return hipGetLastError();
    }
  }
  hipLaunchKernelGGL((k_fill<FMT, PL, false>), dim3((uint32_t)blocks), dim3(block_threads), 0, stream, a);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_fill(const FillArgs& a, int format, int per_lane, int block_threads, bool in_step, hipStream_t stream) {
  switch (format * 8 + per_lane) {
    case 0 * 8 + 1: return fill_one<0, 1>(a, block_threads, in_step, stream);
    case 0 * 8 + 2: return fill_one<0, 2>(a, block_threads, in_step, stream);
    case 0 * 8 + 4: return fill_one<0, 4>(a, block_threads, in_step, stream);
    case 1 * 8 + 1: return fill_one<1, 1>(a, block_threads, in_step, stream);
    case 1 * 8 + 2: return fill_one<1, 2>(a, block_threads, in_step, stream);
    case 1 * 8 + 4: return fill_one<1, 4>(a, block_threads, in_step, stream);
    case 2 * 8 + 1: return fill_one<2, 1>(a, block_threads, in_step, stream);
    case 2 * 8 + 2: return fill_one<2, 2>(a, block_threads, in_step, stream);
    case 2 * 8 + 4: return fill_one<2, 4>(a, block_threads, in_step, stream);
    default: return hipErrorInvalidValue;
  }
}

namespace {

template <int FMT, int COL, int WAVES>
hipError_t fill_mfma_one(const MfmaFillArgs& a, uint64_t blocks, hipStream_t stream) {
  hipLaunchKernelGGL((k_fill_mfma<FMT, COL, WAVES>), dim3((uint32_t)blocks), dim3(64 * WAVES), 0, stream, a);
  return hipGetLastError();
}

template <int FMT, int COL>
hipError_t fill_mfma_waves(const MfmaFillArgs& a, uint64_t blocks, hipStream_t stream) {
  switch (a.waves_per_block) {
    case 4: return fill_mfma_one<FMT, COL, 4>(a, blocks, stream);
    case 8: return fill_mfma_one<FMT, COL, 8>(a, blocks, stream);
    case 16: return fill_mfma_one<FMT, COL, 16>(a, blocks, stream);
    default: return hipErrorInvalidValue;
  }
}

template <int FMT>
hipError_t fill_mfma_column(const MfmaFillArgs& a, uint64_t blocks, hipStream_t stream) {
  return a.column == 64 ? fill_mfma_waves<FMT, 64>(a, blocks, stream) : fill_mfma_waves<FMT, 128>(a, blocks, stream);
}

}  // namespace

hipError_t launch_fill_mfma(const MfmaFillArgs& a, int format, hipStream_t stream) {
  const uint64_t waves = a.waves + a.extra;
  if (waves == 0) return hipSuccess;
  if (a.extra > 2 || a.tiles_per_wave == 0 || a.waves != (a.tiles + a.tiles_per_wave - 1) / a.tiles_per_wave ||
      (a.column != 64 && a.column != 128) || (a.waves_per_block != 4 && a.waves_per_block != 8 && a.waves_per_block != 16))
    return hipErrorInvalidValue;
  const uint64_t blocks = (waves + a.waves_per_block - 1) / a.waves_per_block;
  if (blocks * 64 * a.waves_per_block > 0xffffffffull) return hipErrorInvalidConfiguration;  // 32-bit grid
  switch (format) {
    case 0: return fill_mfma_column<0>(a, blocks, stream);
    case 1: return fill_mfma_column<1>(a, blocks, stream);
    case 2: return fill_mfma_column<2>(a, blocks, stream);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_batch_short(const BatchArgs& a, uint32_t waves, hipStream_t stream) {
  if (!a.mfma_a || waves == 0) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_batch_short, dim3(waves), dim3(64), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_batch(const BatchArgs& a, int grid, int block_threads, hipStream_t stream) {
  hipLaunchKernelGGL(k_batch, dim3(grid), dim3(block_threads), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_batch_queue(const BatchArgs& a, int grid, int block_threads, hipStream_t stream) {
  if (grid <= 0) return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL(k_batch_queue, dim3(grid), dim3(block_threads), 0, stream, a);
  return hipGetLastError();
}

namespace {

template <int G>
hipError_t advance_lds(const AdvanceArgs& a, hipStream_t stream) {
  const uint64_t per = (uint64_t)kAdvanceGroups * G;
  hipLaunchKernelGGL((k_advance_lds<G>), dim3((uint32_t)((a.n + per - 1) / per)), dim3(4 * kAdvanceGroups), 0, stream, a);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_advance(const AdvanceArgs& a, int states, hipStream_t stream) {
  if (a.n == 0) return hipSuccess;
  if (a.n > (0xffffffffull >> 3) || a.words < 1 || a.words > (uint32_t)kAdvanceWords) return hipErrorInvalidValue;
  switch (states) {
    case 0: break;
    case 2: return advance_lds<2>(a, stream);
    case 4: return advance_lds<4>(a, stream);
    case 8: return advance_lds<8>(a, stream);
    default: return hipErrorInvalidValue;
  }
  hipLaunchKernelGGL(k_advance, dim3((uint32_t)((a.n * 8 + 255) / 256)), dim3(256), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_stage(const void* src, void* dst, size_t bytes, hipStream_t stream) {
  if (bytes == 0) return hipSuccess;
  if (bytes % 4 || (reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) % 16)
    return hipErrorInvalidValue;
  const uint64_t n16 = bytes / 16, tail = (bytes % 16) / 4;
  const uint64_t blocks = (n16 + 255) / 256 + (n16 == 0 ? 1 : 0);
  if (blocks > 0xffffffffull) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_stage, dim3((uint32_t)blocks), dim3(256), 0, stream, static_cast<const u4_t*>(src),
                     static_cast<u4_t*>(dst), n16, tail);
  return hipGetLastError();
}

hipError_t launch_batch_tiles(const BatchArgs& a, uint64_t ntiles, int block_threads, hipStream_t stream) {
  if (block_threads > kTileBlockThreads) return hipErrorInvalidConfiguration;
  const uint64_t wpb = (uint64_t)block_threads / 64;
  const uint64_t blocks = (ntiles + wpb - 1) / wpb;
  if (blocks == 0) return hipSuccess;
  if (blocks * (uint64_t)block_threads > 0xffffffffull) return hipErrorInvalidConfiguration;  // 32-bit grid
  hipLaunchKernelGGL(k_batch_tiles, dim3((uint32_t)blocks), dim3(block_threads), 0, stream, a);
  return hipGetLastError();
}

}  // namespace mrg8
