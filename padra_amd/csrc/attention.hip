// Decode attention over a BF16 or q8 KV cache: split-K partial softmax, then a per-head merge.
//
// Reference: gqa8_fragment_validation::SplitBF16 (attention_gqa8_fragment_validation.cuh:
// 79-214) with attention_perhead_exact::Merge (attention_perhead_exact.cuh:7-38); for q8
// caches gqa8_q8_attention::SplitBF16 (attention_gqa8_q8.cuh:112-277), which reads the
// tiles through kv_q8::Decode.  Any number of query heads per KV head up to 8 (the
// reference fixes 8).  One token per sequence, at its DecodeState position; keys are the
// last n positions (n = position + 1, or at most 1024 for a local ring), read from cache
// row (first + offset) % cap.
//
// Split kernel (k_attn_mx): one workgroup per (sequence, KV head, split), over that split's
// 32-key tiles, QK and PV on the matrix cores; the reference's online softmax per row
// (tile maximum, fp32 probabilities for the denominator fmaf(den, alpha, total), BF16
// probabilities for the PV product, scale 1/sqrt(128) applied after the dot product).
// Merge kernel: one wave per (sequence, query head): weights exp(lse_s - max) / sum, then
// out = B(sum_s w_s * partial_s) in split order.
//
// Not bit-identical to the reference: its QK and PV products run on tensor-core MMA with an
// unspecified accumulation order, and its expf/logf are CUDA's.  Products of two BF16
// values are exact in fp32, so only the order of the fp32 sums and the exp/log ulps differ.
// The split kernels take their probabilities from the hardware exponential
// (v_exp_f32(x * log2 e), __expf): for x = score - maximum <= 0 its relative error grows
// with |x| (about 2^-24 |x| from rounding x * log2 e), so it is a few fp32 ulps where the
// probability matters and larger only for probabilities below e^-16.
#include <stdio.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <type_traits>

#include "common.h"
#include "norm_fp8.h"

using namespace padra;

namespace {

constexpr int kD = 128, kKeys = 32;
// Launches of up to this many sequences on a global cache order their splits by window
// length (the ranking reads seqs^2 control records); up to kRankMaxSeqs in the split kernels.
constexpr int kOrderMaxSeqs = 512, kRankMaxSeqs = 16;
constexpr float kScoreScale = .08838834764831845f;

int launched(const char *what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    fprintf(stderr, "padra: %s launch failed: %s\n", what, hipGetErrorString(e));
    return PADRA_INTERNAL;
  }
  return PADRA_OK;
}
bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

struct AttnArgs {
  const void *q; // [seqs][hq][128], activation type
  const uint16_t *kc, *vc;
  void *out; // [seqs][hq][128]
  float *partial, *lse;
  const padra_DecodeState *decode;
  int seqs, hq, hkv, group, cap, local, splits, maximum, vocab;
  long long seq_stride; // cache rows between sequences
  int *bad;
  // q8_0 caches: the coded query (int8 [seqs][hq][128]) and its block scales
  // (fp32 [seqs][hq][4]), both in the scratch.
  int8_t *qcodes;
  float *qscale;
  const float *kvscales; // q8 caches: (k, v) scale pair per row and KV head
  // How a split kernel's workgroup finds its unit (sequence and split): kPlain, from the grid
  // (every sequence's every split); otherwise unit blockIdx.y of the splits that have tiles,
  // longest windows first: kRanked, each wave ranks the sequences itself; kOrdered, from `order`,
  // written by an earlier kernel: the sequence of each rank, and its first unit << 9.
  enum { kPlain, kRanked, kOrdered } units;
  int *order;
};

// The sequence's admission and key window (Admitted, attention_gqa8_fragment_validation.cuh:
// 49-55, with the split count a parameter): n keys from position `first`.
__device__ __forceinline__ bool attn_window(const AttnArgs &a, int seq, int &n, int &first) {
  const padra_DecodeState st = load_state(a.decode + seq);
  const bool ok = decode_ready(st, a.maximum, a.vocab) && a.cap <= st.capacity &&
                  (a.local ? a.cap == min(1024, st.capacity) : a.cap == st.capacity);
  n = a.local ? min(st.position + 1, 1024) : st.position + 1;
  first = st.position + 1 - n;
  return ok;
}

// A split kernel's unit of work: one split of one sequence's window.
struct AttnUnit {
  int seq, split, n, first; // the window: n keys from position `first`
  int begin, end;           // the split's tiles
};

// The splits of an n-key window that have tiles (of TILE keys), and a unit's tiles.
template <int TILE> __device__ __forceinline__ int attn_active(const AttnArgs &a, int n) {
  return min(a.splits, (n + TILE - 1) / TILE);
}
template <int TILE> __device__ __forceinline__ void attn_tiles(const AttnArgs &a, AttnUnit &x) {
  const int tiles = (x.n + TILE - 1) / TILE, active = min(a.splits, tiles);
  x.begin = tiles * x.split / active;
  x.end = tiles * (x.split + 1) / active;
}
template <int TILE> __device__ __forceinline__ bool attn_admitted(const AttnArgs &a, int seq,
                                                                  int &n, int &first) {
  return attn_window(a, seq, n, first) && !(TILE == 128 && a.local && a.cap != 1024);
}

// The unit of (sequence, split), false where the split has no tile.  `raise`: whether this
// thread reports a sequence that is not admitted.
template <int TILE> __device__ __forceinline__ bool attn_unit(const AttnArgs &a, int seq, int split,
                                                              bool raise, AttnUnit &x) {
  x.seq = seq;
  x.split = split;
  if (!attn_admitted<TILE>(a, x.seq, x.n, x.first)) {
    if (split == 0 && raise)
      raise_bad(a.bad);
    return false;
  }
  if (split >= attn_active<TILE>(a, x.n))
    return false;
  attn_tiles<TILE>(a, x);
  return true;
}

// Unit u among all the batch's splits that have tiles, the longest windows' first (ties by
// sequence), so that the longest start first and the shortest fill the end of the launch.  The
// units past the last active one are the end of the grid.  Where each sequence's
// inactive splits (all but n / 32 of 32) came between the others' active ones, their waves, which
// do no more than read the control records, held the slots: 64 sequences of up to 300 keys
// (BF16) 40.4 -> 18.8 us, of up to 1000 keys (q8_0) 83.7 -> 31.8 us.
//
// In the split kernels (2 to 16 sequences, one a lane): saves the launch of k_attn_order, 2-4 us,
// and costs each wave 5 instructions a sequence; at 64 sequences those were 7 us of
// 111 (8000 keys).
template <int TILE> __device__ __forceinline__ bool attn_unit_ranked(const AttnArgs &a, int u,
                                                                     bool raise, AttnUnit &x) {
  const int lane = threadIdx.x & 63;
  int n = 0, first = 0;
  const bool ok = lane < a.seqs && attn_admitted<TILE>(a, lane, n, first);
  if (u == 0 && __ballot(lane < a.seqs && !ok) != 0 && raise)
    raise_bad(a.bad);
  const int active = ok ? attn_active<TILE>(a, n) : 0;
  const int key = ((ok ? n : 0) << 6) + 63 - lane; // distinct
  int before = 0;                                  // active splits of longer windows
  for (int j = 0; j < a.seqs; j += 8)
#pragma unroll
    for (int i = 0; i < 8; ++i)
      before += __builtin_amdgcn_readlane(key, j + i) > key
                    ? __builtin_amdgcn_readlane(active, j + i)
                    : 0;
  const uint64_t mine = __ballot(before <= u && u < before + active);
  if (mine == 0)
    return false; // wave-uniform
  x.seq = (int)__builtin_ctzll(mine);
  x.split = u - __builtin_amdgcn_readlane(before, x.seq);
  x.n = __builtin_amdgcn_readlane(n, x.seq);
  x.first = __builtin_amdgcn_readlane(first, x.seq);
  attn_tiles<TILE>(a, x);
  return true;
}

// More sequences: ranked by an earlier kernel, a 64-lane block per sequence.
template <int TILE> __device__ __forceinline__ void attn_rank(const AttnArgs &a, int seq) {
  int n, first;
  const bool ok = attn_admitted<TILE>(a, seq, n, first);
  if (!ok && threadIdx.x == 0)
    raise_bad(a.bad);
  const int mine = ok ? n : 0;
  int before = 0, units = 0;
  for (int j = threadIdx.x; j < a.seqs; j += 64) {
    const int other = attn_admitted<TILE>(a, j, n, first) ? n : 0;
    if (other > mine || (other == mine && j < seq)) {
      ++before;
      units += attn_active<TILE>(a, other);
    }
  }
  const auto sum = [](int x, int y) { return x + y; };
  before = xor_reduce<32>(before, sum);
  units = xor_reduce<32>(units, sum);
  if (threadIdx.x == 0)
    a.order[before] = seq | (units << 9);
}
template <int TILE> __device__ __forceinline__ bool attn_unit_ordered(const AttnArgs &a, int u,
                                                                      AttnUnit &x) {
  int entry = 0; // of the last rank whose first unit is u or before (rank 0's is 0)
  for (int j = 0; j < a.seqs; j += 64) {
    const int rank = j + (threadIdx.x & 63);
    const int e = a.order[min(rank, a.seqs - 1)];
    const uint64_t m = __ballot(rank < a.seqs && (e >> 9) <= u);
    if (m != 0)
      entry = __builtin_amdgcn_readlane(e, 63 - (int)__builtin_clzll(m));
  }
  return attn_unit<TILE>(a, entry & 511, u - (entry >> 9), false, x);
}

// A workgroup's unit; `raise` as above.
template <int TILE> __device__ __forceinline__ bool attn_find(const AttnArgs &a, bool raise,
                                                              AttnUnit &x) {
  if (a.units == AttnArgs::kPlain)
    return attn_unit<TILE>(a, blockIdx.z, blockIdx.y, raise, x);
  if (a.units == AttnArgs::kRanked)
    return attn_unit_ranked<TILE>(a, blockIdx.y, raise, x);
  return attn_unit_ordered<TILE>(a, blockIdx.y, x);
}

constexpr int kQ8Tile = 128, kRowBytes = 544; // q8_0: keys of a tile, bytes of a row

__global__ __launch_bounds__(64) void k_attn_order(AttnArgs a) {
  attn_rank<kKeys>(a, blockIdx.x);
}

// Hadamard stages on lane bits 0..5, bit 0 first, of two values per lane.
__device__ __forceinline__ void hadamard64_pair(float &x0, float &x1, int lane) {
  x0 = hadamard_lane<1>(x0, lane);
  x1 = hadamard_lane<1>(x1, lane);
  x0 = hadamard_lane<2>(x0, lane);
  x1 = hadamard_lane<2>(x1, lane);
  x0 = hadamard_lane<4>(x0, lane);
  x1 = hadamard_lane<4>(x1, lane);
  x0 = hadamard_lane<8>(x0, lane);
  x1 = hadamard_lane<8>(x1, lane);
  x0 = hadamard_lane<16>(x0, lane);
  x1 = hadamard_lane<16>(x1, lane);
  x0 = hadamard_lane<32>(x0, lane);
  x1 = hadamard_lane<32>(x1, lane);
}
__device__ __forceinline__ float xor_max32(float v) {
  return xor_reduce<16>(v, [](float x, float y) { return fmaxf(x, y); });
}
__device__ __forceinline__ float xor_sum32(float v) {
  return xor_reduce<16>(v, [](float x, float y) { return x + y; });
}

template <class T> __device__ __forceinline__ float act_value(const void *p, size_t i) {
  if constexpr (std::is_same<T, uint16_t>::value)
    return __uint_as_float((uint32_t) static_cast<const uint16_t *>(p)[i] << 16);
  else
    return static_cast<const float *>(p)[i];
}

// ---- Split kernel on the matrix cores --------------------------------------------------
// QK and PV on v_mfma_f32_16x16x32_bf16 (the reference runs both on tensor-core MMA).  One
// workgroup of W waves per (sequence, KV head, split), over the split's tiles in rounds of W;
// query rows are the 16 MFMA columns (rows past the group are zero).
//  - QK, a tile per wave: S[key][row] = K[key][:] . Q[row][:] for the tile's two 16-key halves,
//    4 K-steps of 32 dimensions each.  Lane l then holds row l % 16, keys 16 h + 4 (l / 16) + i.
//  - Softmax: the row's tile maximum and probability sum are the lane's 8 values plus two
//    exchanges between the four lanes of the row.  The tile maxima of a round cross LDS, so
//    that each wave knows the running maximum at its tile: probabilities, rescale factors
//    and the denominator's terms are those of one wave walking the tiles in order.
//  - PV, 8 / W blocks of 16 dimensions per wave, over the round's tiles in order: O[row][dim] +=
//    P[row][key] V[key][dim] with P from the score registers (K-slot i of lane group g is key
//    4g + i, then 16 + 4g + i - 4) and V staged in LDS as 4-key groups per dimension, so that
//    each B operand is two 8-byte LDS reads.  Lane l holds rows 4 (l / 16) + i of dimension
//    16 b + l % 16.  Every sum thus has the order it has with one wave, and the results are
//    the same bits for every W.
//
// What bounds it: with few sequences the bytes in flight (one wave a split: 1.5 TB/s at one
// sequence of 32768 keys), with many the memory rate (5.9 TB/s at 64; a kernel that only reads
// reaches 7.0).  Several waves a split give each its tile's 16 KB of loads at once and divide
// PV: one sequence of 131072 keys 148.9 -> 75.6 us (BF16), 231.5 -> 71.3 us (q8); of 32768 keys
// 45.9 -> 26.4 and 66.4 -> 26.1 us; 8 sequences to 8000 keys 29.9 -> 25.2 and 31.3 -> 24.3 us.
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4_t mfma_bf16(uint4 a, uint4 b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                 __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// Whether every code * scale of a q8 row is finite in BF16 and the scale is valid:
// 0 < scale and 127 * scale below 0x1.ffp127, the least fp32 value that BF16 rounds to
// infinity (|code| <= 127, and rounding is monotonic).  Tiles with a row that fails it
// check each decoded value (q8_check16).
__device__ __forceinline__ bool q8_scale_fast(float scale) {
  return scale > 0.f && 127.f * scale < 0x1.ffp127f;
}

// The values code * scale of a word of four codes (kv_q8::Decode), with the least code seen
// (as a float; -128 is the code the reference rejects).  Keys past the window come with the last
// key's row, whose codes are checked anyway.  Each code is one
// v_cvt_f32_i32 with a sign-extended byte select; min(min(least, a), b) is one v_min3_f32.
__device__ __forceinline__ void q8_values4(uint32_t w, float scale, float *f, float &least) {
#pragma unroll
  for (int b = 0; b < 4; ++b)
    f[b] = (float)(int8_t)((w >> (8 * b)) & 0xffu);
#pragma unroll
  for (int b = 0; b < 4; ++b)
    least = fminf(least, f[b]);
  // Here and not where it is used: sunk to there, it kept every code of the tile in
  // registers (256 VGPRs and more).
  asm volatile("" : "+v"(least));
#pragma unroll
  for (int b = 0; b < 4; ++b)
    f[b] = f[b] * scale;
}
__device__ __forceinline__ void q8_values8(uint32_t w0, uint32_t w1, float scale, float (&f)[8],
                                           float &least) {
  q8_values4(w0, scale, f, least);
  q8_values4(w1, scale, f + 4, least);
}

// kv_q8::Decode's checks on a chunk whose scale failed q8_scale_fast: a valid scale and
// every code * scale finite in BF16, which the largest |code| decides.
__device__ __forceinline__ bool q8_check16(uint4 c, float scale) {
  uint32_t w[4] = {c.x, c.y, c.z, c.w};
  // An opaque copy: the compiler would otherwise keep every decoded value of the tile in
  // registers for this rare path (400 VGPRs).
#pragma unroll
  for (int i = 0; i < 4; ++i)
    asm volatile("" : "+v"(w[i]));
  float most = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int b = 0; b < 4; ++b)
      most = fmaxf(most, fabsf((float)(int8_t)((w[i] >> (8 * b)) & 0xffu)));
  return isfinite(scale) && scale > 0.f && most * scale < 0x1.ffp127f;
}

// Slot of dimension d in a staged V row.  Each staging lane writes its dimension pairs at
// slots rotated by its chunk index (q8: 16-dimension chunks, rotation by the chunk; BF16:
// 8-dimension chunks, rotation by chunk / 4), which spreads a quarter-wave's 16-byte writes
// over all 64 banks.
template <bool Q8> __device__ __forceinline__ int vq_slot(int d) {
  if constexpr (Q8) {
    const int t = d >> 4;
    return 16 * t + 2 * (((d >> 1) + t) & 7) + (d & 1);
  } else {
    const int c = d >> 3;
    return 8 * c + 2 * (((d >> 1) + (c >> 2)) & 3) + (d & 1);
  }
}

// DENSE: for q8 launches of more one-wave workgroups than two on each SIMD (2048), held to the
// registers of three (168 VGPRs, no spill, for 190): the decode is arithmetic, whose waits a third
// wave fills (VALU issue 89% of the cycles then, 64 sequences to 32768 keys).  64 sequences (us): to
// 131072 keys (16 heads) 788 -> 727, to 32768 238 -> 222, to 8000 (32 heads) 96.9 -> 90.0; 24 to
// 8000 keys 50.6 -> 48.5.  In smaller launches two a SIMD is all there is and the order that this
// takes costs 3-5%: 12 sequences to 65536 keys 154 -> 162.
template <class T, bool Q8, int W, bool DENSE = false>
__global__ __launch_bounds__(64 * W, DENSE ? 3 : 1) void k_attn_mx(AttnArgs a) {
  constexpr bool HELD = Q8 && (W > 1 || DENSE);
  constexpr int NB = 8 / W; // 16-dimension blocks of the output per wave
  const int G = a.group;
  // Per tile of the round: (V[4j][d], V[4j+1][d]), (V[4j+2][d], V[4j+3][d]) at slot
  // vq_slot(d) ^ 16 (j % 2) (odd groups half the banks away from even ones); the probabilities in
  // the A operand's layout; per query row, the tile's maximum, its rescale factor and its sum of
  // probabilities.
  __shared__ __align__(16) uint2 vq[W][kKeys / 4][kD];
  __shared__ __align__(16) uint4 pq[W][64];
  __shared__ __align__(16) float tile_max[W][16], tile_alpha[W][16], tile_total[W][16];
  const int lane = threadIdx.x & 63;
  const int wave = W == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, grp = lane >> 4;
  AttnUnit unit;
  if (!attn_find<kKeys>(a, blockIdx.x == 0 && threadIdx.x == 0, unit))
    return; // block-uniform
  int kv = blockIdx.x;
  if (a.units == AttnArgs::kOrdered) {
    // In a large batch a sequence's workgroups go head by head, each head's splits in a row:
    // 64 sequences of 32768 keys (BF16) 360 us, with the heads of a split side by side 370.
    const int active = attn_active<kKeys>(a, unit.n), at = unit.split * a.hkv + kv;
    kv = at / active;
    unit.split = at - kv * active;
    attn_tiles<kKeys>(a, unit);
  }
  const int seq = unit.seq, split = unit.split, n = unit.n, first = unit.first;
  const int begin = unit.begin, end = unit.end;
  const int features = a.hkv * kD;
  constexpr int ES = Q8 ? 1 : 2; // bytes per cache element
  const size_t head_off = ((size_t)seq * a.seq_stride * features + kv * kD) * ES;
  const char *kbytes = reinterpret_cast<const char *>(a.kc) + head_off;
  const char *vbytes = reinterpret_cast<const char *>(a.vc) + head_off;
  const char *sbytes = reinterpret_cast<const char *>(
      reinterpret_cast<const float2 *>(a.kvscales) + (size_t)seq * a.seq_stride * a.hkv + kv);

  // Tile loads, each instruction covering whole rows of the head (BF16: 256 B on 16 lanes;
  // q8: 128 codes on 8 lanes): K straight into the score MFMAs' operand layout, 64 B of 16
  // rows an instruction, reads at half the rate (128 workgroups: 3.3 TB/s against 6.1).
  //  K: load m is key lane / KL + 64 / KL m, 16 bytes at chunk lane % KL of the row.
  //  V: BF16 m = 4 h + p is key 16 h + 4 grp + p, dimensions 8 col ..; q8 m is key
  //  4 (lane / 8) + m, dimensions 16 (lane % 8) ...
  // Window offsets past the last key read the last key's row (the reference zero-fills them);
  // their scores are masked to -inf, so their probabilities are 0, and their V values finite.
  constexpr int KL = Q8 ? 8 : 16, CH = Q8 ? 4 : 8;
  uint4 kw[CH], vw[CH];
  float ksc[2], vsc[4]; // q8: scales of keys 16 h + col (K) and of this lane's V keys
  const uint32_t part = 16 * (lane & (KL - 1)), first_row = (uint32_t)(first % a.cap);
  auto row_of = [&](int tile, int key) { // the window holds at most cap keys: one wrap
    const uint32_t r = first_row + (uint32_t)min(tile * kKeys + key, n - 1);
    return min(r, r - (uint32_t)a.cap); // r - cap is huge when r < cap
  };
  const uint32_t row_bytes = (uint32_t)features * ES, scale_bytes = (uint32_t)a.hkv * 8;
  auto load_k = [&](int tile) {
#pragma unroll
    for (int m = 0; m < CH; ++m)
      kw[m] = ld_nt(reinterpret_cast<const uint4 *>(
          kbytes + part + (size_t)row_of(tile, lane / KL + 64 / KL * m) * row_bytes));
    if constexpr (Q8) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
        ksc[h] = *reinterpret_cast<const float *>(sbytes + (size_t)row_of(tile, 16 * h + col) * scale_bytes);
    }
  };
  auto v_key = [&](int m) { return 4 * (lane / KL) + (Q8 ? m : 16 * (m >> 2) + (m & 3)); };
  auto load_v = [&](int tile) {
#pragma unroll
    for (int m = 0; m < CH; ++m) {
      const uint32_t r = row_of(tile, v_key(m));
      vw[m] = ld_nt(reinterpret_cast<const uint4 *>(vbytes + part + (size_t)r * row_bytes));
      if constexpr (Q8)
        vsc[m] = *reinterpret_cast<const float *>(sbytes + 4 + (size_t)r * scale_bytes);
    }
  };
  if (begin + wave < end) { // wave-uniform
    load_k(begin + wave);
    load_v(begin + wave);
  }
  issue_point();

  // Query operand: row col (zero past G), step t's dimensions as K's chunks hold them;
  // finite and BF16-exact, as the reference requires of its fp32 input.
  uint4 qb[4];
  bool fine = true;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    uint32_t w[4] = {0, 0, 0, 0};
    if (col < G) {
      const size_t o = ((size_t)seq * a.hq + kv * G + col) * kD +
                       (Q8 ? 64 * (t >> 1) + 16 * grp + 8 * (t & 1) : 32 * t + 8 * grp);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x0 = act_value<T>(a.q, o + 2 * e), x1 = act_value<T>(a.q, o + 2 * e + 1);
        fine = fine && isfinite(x0) && isfinite(x1) && (__float_as_uint(x0) & 0xffffu) == 0 &&
               (__float_as_uint(x1) & 0xffffu) == 0;
        w[e] = (__float_as_uint(x0) >> 16) | (__float_as_uint(x1) & 0xffff0000u);
      }
    }
    qb[t] = make_uint4(w[0], w[1], w[2], w[3]);
  }

  float maximum = -INFINITY, den = 0.f; // of row col, over the tiles before this round
  f32x4_t o[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b)
    o[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int round = begin; round < end; round += W) {
    const int count = min(W, end - round), tile = round + wave;
    float sv[8], tmax = -INFINITY;
    // A wave's tile up to its maximum score.  MORE: the wave has a tile in the next round,
    // loaded as soon as the registers are free (K once it is in LDS, V likewise).  The last
    // tile is code of its own: with the loads under a condition the compiler can only wait
    // for all of them at once, which exposed the latency of the tile just issued
    // (W = 1: 148 -> 211 us at 131072 keys).  So is, in BF16, a tile that the window's end cuts
    // (CUT): its keys past the end have no V row, and an infinity of the last key's row, which they
    // read, times their probability 0 would be NaN.  (Cleared in the last tile's code, with a test
    // or for every one, 8 sequences to 8000 keys took 23.5 -> 23.7-23.9 us, so 23.6.)  In q8 a scale
    // of 1 for those keys does it, in the last tile's code: with code of its own 12 sequences to
    // 65536 keys took 154 us, 16 to 8000 35.0, so 152 and 34.7.
    auto scores = [&](auto more, auto cut) {
      constexpr bool MORE = decltype(more)::value, CUT = decltype(cut)::value;
      const int left = n - tile * kKeys; // keys of this tile inside the window (may be >= 32)
      // Scores: lane holds row col, keys 16 h + 4 grp + i.
      f32x4_t s[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};
      // The tile's K rows cross the wave's LDS image (chunks exchanged by key, so that no two
      // lanes of a 16-lane group meet in a bank), then its V rows take the same space: one
      // wave's LDS accesses run in program order, so the K reads come first.
      uint4 *kq = reinterpret_cast<uint4 *>(&vq[wave][0][0]);
      if constexpr (Q8) {
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          const int key = lane / 8 + 8 * m;
          kq[8 * key + ((lane & 7) ^ ((key >> 1) & 7))] = kw[m];
        }
        const float kscale[2] = {ksc[0], ksc[1]};
        if constexpr (MORE) {
          load_k(tile + W);
          issue_point();
        }
        // Decoded a chunk at a time where HELD: the scheduling barriers keep one chunk's values in
        // registers, not all of them.
        float least = 0.f;
        // Whether some key's scale needs every value checked (rare: huge or invalid scales).
        const bool kslow = __ballot(!q8_scale_fast(kscale[0]) || !q8_scale_fast(kscale[1])) != 0;
        const bool vslow = __ballot(!q8_scale_fast(vsc[0]) || !q8_scale_fast(vsc[1]) ||
                                    !q8_scale_fast(vsc[2]) || !q8_scale_fast(vsc[3])) != 0;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const uint4 c = kq[8 * (16 * h + col) + ((4 * u + grp) ^ (col >> 1))];
            uint32_t w[8];
            float f[8];
            q8_values8(c.x, c.y, kscale[h], f, least);
#pragma unroll
            for (int e = 0; e < 4; ++e)
              w[e] = pack2(f[2 * e], f[2 * e + 1]);
            q8_values8(c.z, c.w, kscale[h], f, least);
#pragma unroll
            for (int e = 0; e < 4; ++e)
              w[4 + e] = pack2(f[2 * e], f[2 * e + 1]);
            s[h] = mfma_bf16(make_uint4(w[0], w[1], w[2], w[3]), qb[2 * u], s[h]);
            s[h] = mfma_bf16(make_uint4(w[4], w[5], w[6], w[7]), qb[2 * u + 1], s[h]);
            if constexpr (HELD)
              __builtin_amdgcn_sched_barrier(0);
          }
        if (kslow) { // one rare branch, not one per chunk, which would cut the code above apart
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int u = 0; u < 2; ++u)
              if (!q8_scale_fast(kscale[h]))
                fine = fine && q8_check16(kq[8 * (16 * h + col) + ((4 * u + grp) ^ (col >> 1))],
                                          kscale[h]);
        }
        if constexpr (!MORE) { // keys past the window: a finite value for any scale
#pragma unroll
          for (int m = 0; m < 4; ++m)
            vsc[m] = v_key(m) < left ? vsc[m] : 1.f;
        }
        const int t7 = lane & 7, j = lane >> 3;
        uint2 *dst = &vq[wave][j][(16 * t7) ^ ((j & 1) << 4)];
#pragma unroll
        for (int i = 0; i < 4; ++i) { // dimensions 4 i .. 4 i + 3 of the chunk, four keys
          float f[4][4];
#pragma unroll
          for (int m = 0; m < 4; ++m)
            q8_values4(i == 0 ? vw[m].x : i == 1 ? vw[m].y : i == 2 ? vw[m].z : vw[m].w, vsc[m],
                       f[m], least);
#pragma unroll
          for (int e = 0; e < 4; e += 2)
            *reinterpret_cast<uint4 *>(dst + 2 * ((2 * i + e / 2 + t7) & 7)) =
                make_uint4(pack2(f[0][e], f[1][e]), pack2(f[2][e], f[3][e]),
                           pack2(f[0][e + 1], f[1][e + 1]), pack2(f[2][e + 1], f[3][e + 1]));
          if constexpr (HELD)
            __builtin_amdgcn_sched_barrier(0);
        }
        fine = fine && least > -128.f;
        if (vslow) {
#pragma unroll
          for (int m = 0; m < 4; ++m)
            if (!q8_scale_fast(vsc[m]))
              fine = fine && q8_check16(vw[m], vsc[m]);
        }
      } else {
#pragma unroll
        for (int m = 0; m < 8; ++m) {
          const int key = grp + 4 * m;
          kq[16 * key + (col ^ (key & 15))] = kw[m];
        }
        if constexpr (MORE) {
          load_k(tile + W);
          issue_point();
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int t = 0; t < 4; ++t)
            s[h] = mfma_bf16(kq[16 * (16 * h + col) + ((4 * t + grp) ^ col)], qb[t], s[h]);
        if constexpr (CUT) {
#pragma unroll
          for (int m = 0; m < CH; ++m) {
            const uint32_t keep = v_key(m) < left ? ~0u : 0u;
            vw[m] = make_uint4(vw[m].x & keep, vw[m].y & keep, vw[m].z & keep, vw[m].w & keep);
          }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const uint4 *p = &vw[4 * h];
          const uint32_t w0[4] = {p[0].x, p[0].y, p[0].z, p[0].w}, w1[4] = {p[1].x, p[1].y, p[1].z, p[1].w},
                         w2[4] = {p[2].x, p[2].y, p[2].z, p[2].w}, w3[4] = {p[3].x, p[3].y, p[3].z, p[3].w};
          uint2 *dst = &vq[wave][4 * h + grp][(8 * col) ^ ((grp & 1) << 4)];
#pragma unroll
          for (int e = 0; e < 4; ++e) // dimensions 2e, 2e + 1 of the chunk
            *reinterpret_cast<uint4 *>(dst + 2 * ((e + (col >> 2)) & 3)) = make_uint4(
                __builtin_amdgcn_perm(w1[e], w0[e], 0x05040100u),
                __builtin_amdgcn_perm(w3[e], w2[e], 0x05040100u),
                __builtin_amdgcn_perm(w1[e], w0[e], 0x07060302u),
                __builtin_amdgcn_perm(w3[e], w2[e], 0x07060302u));
        }
      }
      if constexpr (MORE) {
        load_v(tile + W);
        issue_point();
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float v = s[h][i] * kScoreScale;
          if (16 * h + 4 * grp + i < left)
            fine = fine && isfinite(v);
          else
            v = -INFINITY;
          sv[4 * h + i] = v;
          tmax = fmaxf(tmax, v);
        }
      tmax = fmaxf(tmax, lane_xor<16>(tmax));
      tmax = fmaxf(tmax, lane_xor<32>(tmax));
    };
    if (tile + W < end) // wave-uniform, all three
      scores(std::true_type{}, std::false_type{});
    else if (!Q8 && tile * kKeys + kKeys > n && tile < end)
      scores(std::false_type{}, std::true_type{});
    else if (tile < end)
      scores(std::false_type{}, std::false_type{});
    if (W > 1 && grp == 0)
      tile_max[wave][col] = tmax; // -inf without a tile
    // The running maximum at this wave's tile (every tile of the round before it counted),
    // and after the round.
    float before = maximum, after = fmaxf(maximum, tmax);
    if constexpr (W > 1) {
      __syncthreads();
      after = maximum;
#pragma unroll
      for (int t = 0; t < W; ++t) {
        const float m = tile_max[t][col];
        before = fmaxf(before, t < wave ? m : -INFINITY);
        after = fmaxf(after, m);
      }
    }
    uint4 pa;
    float alpha, total = 0.f;
    if (wave < count) {
      const float next = fmaxf(before, tmax);
      alpha = isfinite(before) ? __expf(before - next) : 0.f;
      float p[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        p[k] = isfinite(sv[k]) ? __expf(sv[k] - next) : 0.f;
        total += p[k];
      }
      total += lane_xor<16>(total);
      total += lane_xor<32>(total);
      pa = make_uint4(pack2(p[0], p[1]), pack2(p[2], p[3]), pack2(p[4], p[5]), pack2(p[6], p[7]));
      if constexpr (W > 1)
        pq[wave][lane] = pa;
      if (grp == 0) {
        tile_alpha[wave][col] = alpha;
        tile_total[wave][col] = total;
      }
    }
    maximum = after;
    __syncthreads();
    // PV of this wave's output blocks over the round's tiles, in tile order.
    auto pv = [&](int t) {
      const uint4 pt = W > 1 ? pq[t][lane] : pa;
      const float4 ar = *reinterpret_cast<const float4 *>(&tile_alpha[t][4 * grp]);
      den = __builtin_fmaf(den, W > 1 ? tile_alpha[t][col] : alpha, W > 1 ? tile_total[t][col] : total);
      const f32x4_t rescale = {ar.x, ar.y, ar.z, ar.w}; // 1 unless a row's maximum moved
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const int d = vq_slot<Q8>(16 * (NB * wave + b) + col) ^ ((grp & 1) << 4);
        const uint2 v0 = vq[t][grp][d], v1 = vq[t][4 + grp][d];
        o[b] = mfma_bf16(pt, make_uint4(v0.x, v0.y, v1.x, v1.y), o[b] * rescale);
        if constexpr (HELD)
          if ((b & 3) == 3)
            __builtin_amdgcn_sched_barrier(0);
      }
    };
    if (count == W) { // block-uniform; without a test per tile its LDS reads overlap
#pragma unroll
      for (int t = 0; t < W; ++t)
        pv(t);
    } else {
      for (int t = 0; t < count; ++t)
        pv(t);
    }
    __syncthreads();
  }
  // Rows 4 grp + i: this lane's dimension 16 (NB wave + b) + col of each.
  const int head0 = kv * G;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 4 * grp + i;
    const float d = __shfl(den, r, 64), mx = __shfl(maximum, r, 64);
    if (r < G) {
      float *dst = a.partial + (((size_t)seq * a.splits + split) * a.hq + head0 + r) * kD +
                   16 * NB * wave + col;
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const float v = o[b][i] / d;
        fine = fine && isfinite(v);
        dst[16 * b] = v;
      }
      if (col == 0 && wave == 0) {
        const float l = mx + logf(d);
        fine = fine && isfinite(l);
        a.lse[((size_t)seq * a.splits + split) * a.hq + head0 + r] = l;
      }
    }
  }
  if (__ballot(!fine) != 0 && lane == 0)
    raise_bad(a.bad);
}

// Partial outputs of one (sequence, head), a float2 per lane and split.  The merge kernels are
// bound by their chain of memory round trips (control record, log-sum-exps, partials), so they
// issue every split's load before the first use and, in small launches, before the control record
// is there: the splits that turn out inactive are read in vain,
// inside the scratch.  Launches of more heads read only the active ones: there the bytes count.
// Steps of 1 / 8 / 64 sequences (1000, 8000, 8000 keys), before -> after: BF16 10.3 -> 8.5,
// 25.2 -> 23.8, 103.6 -> 104.2 us; q8_0 21.9 -> 20.3, 39.2 -> 31.6, 107.1 -> 102.6 us.
constexpr int kMaxSplits = 32, kEarlyHeads = 512;

__device__ __forceinline__ void merge_load(const float *src, size_t step, int count,
                                           float2 (&p)[kMaxSplits]) {
#pragma unroll
  for (int g = 0; g < kMaxSplits; g += 4)
    if (g < count) { // wave-uniform
#pragma unroll
      for (int i = g; i < g + 4; ++i)
        p[i] = *reinterpret_cast<const float2 *>(src + min(i, count - 1) * step);
    }
}

// The weighted sum in split order: w holds split sp's weight in lane sp.
__device__ __forceinline__ void merge_sum(const float2 (&p)[kMaxSplits], float w, int active,
                                          float &s0, float &s1) {
  s0 = s1 = 0.f;
#pragma unroll
  for (int sp = 0; sp < kMaxSplits; ++sp)
    if (sp < active) {
      const float ws =
          __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), sp));
      s0 = __builtin_fmaf(ws, p[sp].x, s0);
      s1 = __builtin_fmaf(ws, p[sp].y, s1);
    }
}

template <class T> __global__ __launch_bounds__(64) void k_attn_merge(AttnArgs a) {
  const int head = blockIdx.x, seq = blockIdx.y, lane = threadIdx.x;
  const size_t entry = (size_t)seq * a.splits * a.hq + head, step = (size_t)a.hq * kD;
  const float *src = a.partial + entry * kD + 2 * lane;
  const bool early = gridDim.x * gridDim.y <= kEarlyHeads;
  const float lse = a.lse[entry + (size_t)min(lane, a.splits - 1) * a.hq];
  float2 p[kMaxSplits];
  if (early)
    merge_load(src, step, a.splits, p);
  int n, first;
  if (!attn_window(a, seq, n, first))
    return; // the split kernel raised the flag
  const int active = min(a.splits, (n + kKeys - 1) / kKeys);
  if (!early)
    merge_load(src, step, active, p);
  const float v = lane < active ? lse : -INFINITY;
  const float mx = xor_max32(v);
  const float w = lane < active ? expf(v - mx) : 0.f;
  const float total = xor_sum32(w), weight = w / total;
  bool fine = lane >= active || isfinite(weight);
  float s0, s1;
  merge_sum(p, weight, active, s0, s1);
  const uint32_t word = pack2(s0, s1);
  fine = fine && ((word & 0x7f80u) != 0x7f80u) && ((word & 0x7f800000u) != 0x7f800000u);
  const size_t o = ((size_t)seq * a.hq + head) * kD + 2 * lane;
  if constexpr (std::is_same<T, uint16_t>::value)
    static_cast<uint32_t *>(a.out)[o / 2] = word;
  else
    *reinterpret_cast<float2 *>(static_cast<float *>(a.out) + o) =
        make_float2(lo16(word), hi16(word));
  if (__ballot(!fine) != 0 && lane == 0)
    raise_bad(a.bad);
}

// MergeQuantize (attention_merge_quantize_wide_exact.cuh:9-66), the merge the reference
// runs after its q8 split (attention_gqa8_q8.cuh:278-300) and, with the FP8 output, after
// the BF16 one: k_attn_merge, then this kernel, the E4M3 encoding of each sequence's output
// row (q_heads x 128 values) with scale = max|out| / 448 (1 for a zero row), as
// padra_QuantizeFP8 writes it.  Waves take heads wave, wave + 4, ...; lane l holds
// dimensions 2l, 2l + 1 of each.  The row's maximum needs every head, and one workgroup that
// merges 32 heads of 32 splits (512 KB) for it runs on one compute unit: 24.8 us, where
// the merge on many units takes 4.2 and this kernel 3.9 (8 sequences; the whole step 43.6 ->
// 26.7 us, 1 sequence of 1000 keys 31.0 -> 11.6).
template <class T>
__global__ __launch_bounds__(256) void k_attn_encode_fp8(AttnArgs a, uint8_t *packed,
                                                         float *scales) {
  constexpr int kWaves = 4, kHeads = 32;
  __shared__ float maxima[kWaves];
  const int seq = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int n, first;
  if (!attn_window(a, seq, n, first))
    return; // block-uniform; the split kernel raised the flag
  bool fine = true;
  uint32_t words[kHeads / kWaves];
  float amax = 0.f;
#pragma unroll
  for (int k = 0; k < kHeads / kWaves; ++k) {
    const int head = min(wave + kWaves * k, a.hq - 1); // heads past the row repeat the last
    const size_t o = ((size_t)seq * a.hq + head) * kD + 2 * lane;
    if constexpr (std::is_same<T, uint16_t>::value) {
      words[k] = static_cast<const uint32_t *>(a.out)[o / 2];
    } else {
      const float2 v = *reinterpret_cast<const float2 *>(static_cast<const float *>(a.out) + o);
      words[k] = pack2(v.x, v.y); // BF16-exact
    }
  }
#pragma unroll
  for (int k = 0; k < kHeads / kWaves; ++k) {
    const uint32_t word = words[k];
    fine = fine && ((word & 0x7f80u) != 0x7f80u) && ((word & 0x7f800000u) != 0x7f800000u);
    amax = fmaxf(amax, fmaxf(fabsf(lo16(word)), fabsf(hi16(word))));
  }
  amax = xor_reduce<32>(amax, [](float x, float y) { return fmaxf(x, y); });
  if (lane == 0)
    maxima[wave] = amax;
  const bool row_fine = !__syncthreads_or(!fine); // (k_attn_merge raised the flag)
  amax = fmaxf(fmaxf(maxima[0], maxima[1]), fmaxf(maxima[2], maxima[3]));
  const float scale = amax == 0.f ? 1.f : amax / 448.f;
  const float inverse = 1.f / scale;
  if (threadIdx.x == 0)
    scales[seq] = scale;
  const bool fast = row_fine && fp8_fast_ok(amax, inverse); // block-uniform
#pragma unroll
  for (int k = 0; k < kHeads / kWaves; ++k) {
    const int head = wave + kWaves * k;
    if (head >= a.hq)
      continue;
    const uint32_t word = words[k];
    const uint32_t code =
        fast ? e4m3_pair_fast(fp8_quotient(lo16(word), scale, inverse),
                              fp8_quotient(hi16(word), scale, inverse))
             : e4m3_code(lo16(word) / scale) | (e4m3_code(hi16(word) / scale) << 8);
    *reinterpret_cast<uint16_t *>(packed + ((size_t)seq * a.hq + head) * kD + 2 * lane) =
        (uint16_t)code;
  }
}

// ---- q8_0 caches ------------------------------------------------------------------------
//
// q8_native::EncodeQuery, Split, Merge (kv_q8_native.cuh:103-148, 198-363).  The query is
// rotated like the K rows (128-point Hadamard, bit 0 first) and coded per 32-block with an
// fp32 scale; a score is the integer dot product of codes, block by block, scaled by
// RN(k_scale * q_scale):  four partial sums P_sub over the 4-code groups sub and sub + 4 of
// each block (fmaf in block order), then ((P0 + P1) + (P2 + P3)), times 1/sqrt(128).  Each
// 128-key tile runs as four 32-key online-softmax streams (slice s: keys 32 s .. 32 s + 31),
// each key lane keeping its own denominator; PV multiplies V codes by p * v_scale.  The four
// streams join per split; the merge joins the splits and rotates the result back (two 64-point
// transforms).  Scores and PV run on the matrix cores here.

// One query head's codes and block scales, by a wave: rotated features lane and lane + 64, of
// blocks lane / 32 and 2 + lane / 32.  False (and nothing written) where a value is not finite.
__device__ __forceinline__ bool q8_0_code_query(float x0, float x1, int lane, int8_t *codes,
                                                float *scales) {
  if (__ballot(!isfinite(x0) || !isfinite(x1)) != 0)
    return false;
  // stages on bits 0..5 across lanes, bit 6 in the lane
  hadamard64_pair(x0, x1, lane);
  const float y0 = (x0 + x1) * .08838834764831845f, y1 = (x0 - x1) * .08838834764831845f;
  float m0 = fabsf(y0), m1 = fabsf(y1);
  m0 = xor_max32(m0);
  m1 = xor_max32(m1);
  const float d0 = m0 / 127.f, d1 = m1 / 127.f;
  if (__ballot(!isfinite(d0) || !isfinite(d1)) != 0)
    return false;
  codes[lane] = (int8_t)q8_0_code(y0, d0 == 0.f ? 0.f : 1.f / d0);
  codes[64 + lane] = (int8_t)q8_0_code(y1, d1 == 0.f ? 0.f : 1.f / d1);
  if ((lane & 31) == 0) {
    scales[lane / 32] = d0;
    scales[2 + lane / 32] = d1;
  }
  return true;
}

template <class T> __global__ __launch_bounds__(64) void k_q8_0_query(AttnArgs a) {
  const int head = blockIdx.x, seq = blockIdx.y, lane = threadIdx.x;
  if (a.units == AttnArgs::kOrdered && head == 0) // one sequence per block
    attn_rank<kQ8Tile>(a, seq);
  const size_t row = (size_t)seq * a.hq + head, base = row * kD;
  if (!q8_0_code_query(act_value<T>(a.q, base + lane), act_value<T>(a.q, base + 64 + lane), lane,
                          a.qcodes + base, a.qscale + row * 4) &&
      lane == 0)
    raise_bad(a.bad);
}

__device__ __forceinline__ float f16_bits(uint32_t h) {
  return __half2float(__ushort_as_half((unsigned short)h));
}

// ---- q8_0 split on the matrix cores -----------------------------------------------------
// One workgroup per (sequence, split): four waves, one per KV head, each serving its G query
// heads; the slice's 544-byte rows are staged whole, once for the four heads.  The reference
// keeps four online-softmax streams per split (stream s: keys 32 s .. 32 s + 31 of every
// 128-key tile) and weighs them by exp(lse_s - max) at the end; here each stream runs on its
// own over the split's tiles and is folded into the split's combination when it ends.
// Per 32-key slice:
//  - QK on v_mfma_i32_16x16x64_i8: rows are (head 4 j + r, block b) pairs of a head group j,
//    whose A operand is the head's query codes masked to block b, so that each result is the
//    exact integer dot product of one block; the score is then
//    fma(float(dot_b), RN(k_scale_b * q_scale_b), ..) in block order, times 1/sqrt(128) (the
//    reference sums the same products with its own grouping of the fp32 additions).  Lane l
//    holds head 4 j + l / 16 of key 16 k + l % 16.
//  - Softmax per head with the reference's recurrences (den = fmaf(den, alpha, p) per key
//    position), maxima over the 16 key lanes by DPP row rotations.
//  - PV on v_mfma_f32_16x16x32_bf16: O[head][dim] += (p * v_scale)[head][key] code[key][dim].
//    Codes are exact in BF16; the fp32 factor enters as two BF16 terms (hi + lo, 2^-17
//    relative).  The factor depends on the dimension's block, so rows are (head, block of a
//    block pair): lane l holds rows 4 (l / 16) + i of dimension 16 t + l % 16, of which the
//    rows of the tile's own block are kept.
typedef int i32x4_t __attribute__((ext_vector_type(4)));

constexpr int kStreams = 4;

__device__ __forceinline__ i32x4_t mfma_i8(uint4 a, uint4 b, i32x4_t c) {
  return __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4_t, a),
                                               __builtin_bit_cast(i32x4_t, b), c, 0, 0, 0);
}

// v from lane (l + N) % 16 of the lane's 16-lane row.
template <int N> __device__ __forceinline__ float row_ror(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x120 + N, 0xf, 0xf, false));
}
// The maximum (fmaxf: NaN operands dropped) and the sum over a 16-lane row; every lane of
// the row gets the same value (each step adds the lane's value to its half-row partner's).
__device__ __forceinline__ float row_max16(float v) {
  v = fmaxf(v, row_ror<8>(v));
  v = fmaxf(v, row_ror<4>(v));
  v = fmaxf(v, row_ror<2>(v));
  return fmaxf(v, row_ror<1>(v));
}
__device__ __forceinline__ float row_sum16(float v) {
  v = v + row_ror<8>(v);
  v = v + row_ror<4>(v);
  v = v + row_ror<2>(v);
  return v + row_ror<1>(v);
}

// x as a BF16 pair hi + lo (hi = RN(x), lo = RN(x - hi)): the packed hi and lo words of
// two values.
__device__ __forceinline__ void bf16_split2(float x0, float x1, uint32_t &hi, uint32_t &lo) {
  hi = pack2(x0, x1);
  lo = pack2(x0 - lo16(hi), x1 - hi16(hi));
}

template <int G> __global__ __launch_bounds__(256) void k_q8_0_mx(AttnArgs a) {
  // The 4 KV heads of a row, one wave each: the slice's rows are staged together, whole.  Per
  // head: K codes (32 keys of 8 chunks, chunk c of a key at c ^ (key / 2) % 8), whose space the
  // probabilities take once the wave has its scores; V codes as BF16 (4 keys per dimension and
  // group j, at slot vq_slot<true>(d) ^ 16 ((j ^ j / 2) % 2)); block scales, K's as stored.  The
  // exchanges and the heads' odd half-strides keep every access off the others' banks.
  // Two barriers a slice and 53 KB, where a place of their own for the probabilities and a third
  // barrier took 63 KB: 64 sequences of 8000 keys (32 heads) 98.4-100.5 -> 96.9-97.8 us, of 32768
  // keys (16 heads) 246.6 -> 244.4.  The registers allow two workgroups a compute unit (218 VGPRs);
  // held to three (168), the spills took twice the time.
  __shared__ __align__(16) uint4 kq_all[4][256 + 8];
  __shared__ __align__(16) uint2 vq_all[4][8 * kD + 16];
  __shared__ __align__(8) uint2 ksc_all[4][32];        // K block scales (4 fp16) by key
  __shared__ __align__(16) float vsc_all[4][4][32];    // V block scales by block
  const int tid = threadIdx.x, kv = tid >> 6;
  const int lane = tid & 63, col = lane & 15, grp = lane >> 4;
  auto &kq = kq_all[kv];
  auto &vq = vq_all[kv];
  auto &ksc = ksc_all[kv];
  auto &vsc = vsc_all[kv];
  float(&ps)[8][36] = *reinterpret_cast<float(*)[8][36]>(&kq_all[kv][0]); // by head (rows padded)
  AttnUnit unit;
  if (!attn_find<kQ8Tile>(a, tid == 0, unit))
    return; // block-uniform
  const int seq = __builtin_amdgcn_readfirstlane(unit.seq);
  const int split = __builtin_amdgcn_readfirstlane(unit.split);
  const int n = __builtin_amdgcn_readfirstlane(unit.n);
  const int first = __builtin_amdgcn_readfirstlane(unit.first);
  const int begin = __builtin_amdgcn_readfirstlane(unit.begin);
  const int end = __builtin_amdgcn_readfirstlane(unit.end);
  const int features = a.hkv * kD, dbytes = 2 * (features / 32);
  const uint8_t *krows = static_cast<const uint8_t *>(static_cast<const void *>(a.kc)) +
                         (size_t)seq * a.seq_stride * kRowBytes;
  const uint8_t *vrows = static_cast<const uint8_t *>(static_cast<const void *>(a.vc)) +
                         (size_t)seq * a.seq_stride * kRowBytes;
  const int head0 = kv * G;

  // Query A operands: row col = (head 4 j + col / 4, block col % 4); K-slot group grp of
  // step h covers dimensions 64 h + 16 grp .. + 15, of block 2 h + grp / 2.
  uint4 aq[2][2];
  float qd[2][4]; // block scales of head 4 j + grp
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int hh = 4 * j + (col >> 2);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      aq[j][h] = make_uint4(0, 0, 0, 0);
      if (hh < G && (col & 3) == 2 * h + (grp >> 1))
        aq[j][h] = *reinterpret_cast<const uint4 *>(
            a.qcodes + ((size_t)seq * a.hq + head0 + hh) * kD + 64 * h + 16 * grp);
    }
    const int hq = 4 * j + grp;
#pragma unroll
    for (int b = 0; b < 4; ++b)
      qd[j][b] = hq < G ? a.qscale[((size_t)seq * a.hq + head0 + hq) * 4 + b] : 0.f;
  }

  // Slice loads over whole rows (512 codes = 32 chunks of 16 bytes): K chunk c = tid + 256 m
  // is key c / 32, part c % 32 (head part / 8, codes 16 (part % 8) ..); V chunk m is key
  // 4 (tid / 32) + m, part tid % 32.  Threads 0..127 load the 32-byte scale headers: half
  // tid % 2 (heads 2 (tid % 2), + 1) of K row tid / 2 (tid < 64) or V row tid / 2 - 32.
  // Keys past the window load the window's first row and are zeroed (the reference
  // zero-fills them).
  auto row_at = [&](int o) {
    const int r = o < n ? o : 0;
    return (size_t)(a.local ? (first + r) & 1023 : first + r) * kRowBytes;
  };
  uint4 kw[4], vw[4], hw = make_uint4(0, 0, 0, 0);
  const int hrow = (tid >> 1) & 31;
  // A slice whose 32 rows are inside the window and consecutive in the cache: load m is
  // the slice's first row plus a per-thread offset plus a step common to all threads
  // (K: 8 m rows, V: m rows).
  const uint32_t koff = (uint32_t)((tid >> 5) * kRowBytes + dbytes + 16 * (tid & 31));
  const uint32_t voff = (uint32_t)(4 * (tid >> 5) * kRowBytes + dbytes + 16 * (tid & 31));
  const uint32_t hoff = (uint32_t)(hrow * kRowBytes + 16 * (tid & 1));
  auto load_slice = [&](int tile, int s) {
    const int o0 = tile * kQ8Tile + 32 * s;
    const int r0 = a.local ? (first + o0) & 1023 : first + o0;
    if (o0 + 32 <= n && (!a.local || r0 + 32 <= 1024)) { // block-uniform
      const uint8_t *kt = krows + (size_t)r0 * kRowBytes, *vt = vrows + (size_t)r0 * kRowBytes;
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        kw[m] = ld_nt(reinterpret_cast<const uint4 *>(kt + (size_t)(8 * m) * kRowBytes + koff));
        vw[m] = ld_nt(reinterpret_cast<const uint4 *>(vt + (size_t)m * kRowBytes + voff));
      }
      if (tid < 128)
        hw = *reinterpret_cast<const uint4 *>((tid < 64 ? kt : vt) + hoff);
      return;
    }
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const int c = tid + 256 * m;
      kw[m] = ld_nt(reinterpret_cast<const uint4 *>(krows + row_at(o0 + (c >> 5)) + dbytes) +
                    (c & 31));
      vw[m] = ld_nt(reinterpret_cast<const uint4 *>(vrows + row_at(o0 + 4 * (tid >> 5) + m) +
                                                    dbytes) + (tid & 31));
    }
    if (tid < 128)
      hw = *reinterpret_cast<const uint4 *>((tid < 64 ? krows : vrows) + row_at(o0 + hrow) +
                                            16 * (tid & 1));
  };

  bool fine = true;
  // The split's combination of its streams, for rows 4 grp + i of the PV layout (head
  // (4 grp + i) % 8): the largest stream log-sum-exp, the total weight, and the weighted
  // outputs of this lane's four dimension tiles t = 4 u + 2 (grp / 2) + v.
  float cm[4], ct[4], cs[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    cm[i] = -INFINITY;
    ct[i] = 0.f;
#pragma unroll
    for (int u = 0; u < 4; ++u)
      cs[u][i] = 0.f;
  }
  bool has[2] = {false, false}; // a stream of head 4 j + grp with a finite log-sum-exp
  const int slices = end - begin;
  load_slice(begin, 0);
  for (int s = 0; s < kStreams; ++s) {
    float mx[2] = {-INFINITY, -INFINITY}, den[2][2] = {{0.f, 0.f}, {0.f, 0.f}};
    f32x4_t o[8];
#pragma unroll
    for (int t = 0; t < 8; ++t)
      o[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int it = 0; it < slices; ++it) {
      const int tile = begin + it, o0 = tile * kQ8Tile + 32 * s;
      // Stage the slice.  Keys past the window stage zero codes: only a slice that crosses
      // the window's end (block-uniform test) zeroes them, with a mask per key.
      if (o0 + 32 > n) {
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          const uint32_t kkeep = o0 + ((tid + 256 * m) >> 5) < n ? ~0u : 0u;
          const uint32_t vkeep = o0 + 4 * (tid >> 5) + m < n ? ~0u : 0u;
          kw[m] = make_uint4(kw[m].x & kkeep, kw[m].y & kkeep, kw[m].z & kkeep, kw[m].w & kkeep);
          vw[m] = make_uint4(vw[m].x & vkeep, vw[m].y & vkeep, vw[m].z & vkeep, vw[m].w & vkeep);
        }
      }
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const int key = (tid >> 5) + 8 * m;
        kq_all[(tid >> 3) & 3][8 * key + ((tid & 7) ^ ((key >> 1) & 7))] = kw[m];
      }
      {
        const int t7 = tid & 7, j = tid >> 5;
        uint2 *dst = &vq_all[(tid >> 3) & 3][j * kD + ((16 * t7) ^ (((j ^ (j >> 1)) & 1) << 4))];
        // four dimensions at a time: without the scheduling barriers 251 VGPRs
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float f[4][4];
#pragma unroll
          for (int m = 0; m < 4; ++m) {
            const uint32_t w = i == 0 ? vw[m].x : i == 1 ? vw[m].y : i == 2 ? vw[m].z : vw[m].w;
#pragma unroll
            for (int b = 0; b < 4; ++b)
              f[m][b] = (float)(int8_t)((w >> (8 * b)) & 0xffu);
          }
#pragma unroll
          for (int e = 0; e < 4; e += 2)
            *reinterpret_cast<uint4 *>(dst + 2 * ((2 * i + e / 2 + t7) & 7)) =
                make_uint4(pack2(f[0][e], f[1][e]), pack2(f[2][e], f[3][e]),
                           pack2(f[0][e + 1], f[1][e + 1]), pack2(f[2][e + 1], f[3][e + 1]));
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if (tid < 128) {
        const bool inside = o0 + hrow < n;
        const uint32_t hv[4] = {hw.x, hw.y, hw.z, hw.w};
#pragma unroll
        for (int h2 = 0; h2 < 2; ++h2) { // heads 2 (tid % 2) + h2
          const int hd = 2 * (tid & 1) + h2;
          const uint32_t w0 = inside ? hv[2 * h2] : 0u, w1 = inside ? hv[2 * h2 + 1] : 0u;
          if (tid < 64) {
            ksc_all[hd][hrow] = make_uint2(w0, w1);
          } else {
            vsc_all[hd][0][hrow] = f16_bits(w0 & 0xffffu);
            vsc_all[hd][1][hrow] = f16_bits(w0 >> 16);
            vsc_all[hd][2][hrow] = f16_bits(w1 & 0xffffu);
            vsc_all[hd][3][hrow] = f16_bits(w1 >> 16);
          }
        }
      }
      __syncthreads();
      // The next slice's loads are in flight during this slice's arithmetic: the next tile
      // of this stream, or the next stream's first slice.  After the last slice the loads
      // stay unconditional and repeat the slice just read, which L2 still holds.
      {
        const bool last_tile = it + 1 == slices, last = last_tile && s == kStreams - 1;
        load_slice(last ? tile : (last_tile ? begin : tile + 1), last_tile && !last ? s + 1 : s);
      }

      // Scores: head 4 j + grp, key 16 k + col.
      float sc[2][2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const uint4 b0 = kq[8 * (16 * k + col) + (grp ^ (col >> 1))];
        const uint4 b1 = kq[8 * (16 * k + col) + ((4 + grp) ^ (col >> 1))];
        const uint2 kh = ksc[16 * k + col];
        const float4 kd = make_float4(f16_bits(kh.x & 0xffffu), f16_bits(kh.x >> 16),
                                      f16_bits(kh.y & 0xffffu), f16_bits(kh.y >> 16));
        const bool valid = o0 + 16 * k + col < n;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          i32x4_t d = mfma_i8(aq[j][0], b0, i32x4_t{0, 0, 0, 0});
          d = mfma_i8(aq[j][1], b1, d);
          float dot = 0.f;
          dot = __builtin_fmaf((float)d[0], kd.x * qd[j][0], dot);
          dot = __builtin_fmaf((float)d[1], kd.y * qd[j][1], dot);
          dot = __builtin_fmaf((float)d[2], kd.z * qd[j][2], dot);
          dot = __builtin_fmaf((float)d[3], kd.w * qd[j][3], dot);
          sc[k][j] = valid ? dot * kScoreScale : -INFINITY;
        }
      }
      float alpha[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const float next = fmaxf(mx[j], row_max16(fmaxf(sc[0][j], sc[1][j])));
        alpha[j] = isfinite(mx[j]) ? __expf(mx[j] - next) : 0.f;
        mx[j] = next;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const float p = isfinite(sc[k][j]) ? __expf(sc[k][j] - next) : 0.f;
          den[k][j] = __builtin_fmaf(den[k][j], alpha[j], p);
          ps[4 * j + grp][16 * k + col] = p;
        }
      }
      // Rows 4 grp + i of the PV accumulators are head (4 grp + i) % 8, whose alpha lane 16 i
      // holds (alpha[0] for heads 0..3, alpha[1] for 4..7).
      if (__ballot(alpha[0] != 1.f || alpha[1] != 1.f) != 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float a0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(alpha[0]), 16 * i));
          const float a1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(alpha[1]), 16 * i));
          const float ar = (grp & 1) ? a1 : a0;
#pragma unroll
          for (int t = 0; t < 8; ++t)
            o[t][i] *= ar;
        }
      }
      // (The probabilities are the wave's own: its LDS accesses run in program order.)
      // PV A operands: row col = (head col % 8, block 2 c + col / 8); K-slots of group grp are
      // keys 8 grp .. 8 grp + 7.
      uint4 ahi[2], alo[2];
      {
        const int hh = col & 7;
        const float4 p0 = *reinterpret_cast<const float4 *>(&ps[hh][8 * grp]);
        const float4 p1 = *reinterpret_cast<const float4 *>(&ps[hh][8 * grp + 4]);
        const float pv[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const int b = 2 * c + (col >> 3);
          const float4 v0 = *reinterpret_cast<const float4 *>(&vsc[b][8 * grp]);
          const float4 v1 = *reinterpret_cast<const float4 *>(&vsc[b][8 * grp + 4]);
          const float vv[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
          uint32_t hi[4], lo[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float f0 = hh < G ? pv[2 * e] * vv[2 * e] : 0.f;
            const float f1 = hh < G ? pv[2 * e + 1] * vv[2 * e + 1] : 0.f;
            bf16_split2(f0, f1, hi[e], lo[e]);
          }
          ahi[c] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
          alo[c] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
        }
      }
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const int d = vq_slot<true>(16 * t + col) ^ ((grp & 1) << 4);
        const uint2 v0 = vq[2 * grp * kD + d], v1 = vq[(2 * grp + 1) * kD + (d ^ 16)];
        const uint4 bv = make_uint4(v0.x, v0.y, v1.x, v1.y);
        o[t] = mfma_bf16(ahi[t >> 2], bv, o[t]);
        o[t] = mfma_bf16(alo[t >> 2], bv, o[t]);
      }
      __syncthreads(); // the next slice restages the tiles
    }
    // The stream's log-sum-exp (den over the 32 key positions), folded into the split's
    // combination with weight exp(lse - max): the reference weighs its four streams the
    // same way once all are done; online here, in stream order.  Streams without a finite
    // log-sum-exp carry no weight, as there.
    float dsum[2], lse[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      dsum[j] = row_sum16(den[0][j] + den[1][j]);
      lse[j] = dsum[j] > 0.f ? mx[j] + logf(dsum[j]) : -INFINITY;
      has[j] = has[j] || isfinite(lse[j]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // head (4 grp + i) % 8 is head 4 (grp % 2) + i, whose values lane 16 i holds (in
      // dsum[grp % 2] and lse[grp % 2]: read both, then select per lane)
      const float d0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(dsum[0]), 16 * i));
      const float d1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(dsum[1]), 16 * i));
      const float l0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(lse[0]), 16 * i));
      const float l1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(lse[1]), 16 * i));
      const float d = (grp & 1) ? d1 : d0, l = (grp & 1) ? l1 : l0;
      if (isfinite(l)) {
        const float m2 = fmaxf(cm[i], l);
        const float wa = isfinite(cm[i]) ? expf(cm[i] - m2) : 0.f, wb = expf(l - m2);
        ct[i] = __builtin_fmaf(ct[i], wa, wb);
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int v = 0; v < 2; ++v) {
            // both values first: a conditional over the two array elements would select
            // an address and index the accumulators at run time
            const float xa = o[4 * u + v][i], xb = o[4 * u + 2 + v][i];
            const float x = (grp >> 1) ? xb : xa;
            cs[2 * u + v][i] = __builtin_fmaf(cs[2 * u + v][i], wa, wb * (x / d));
          }
        cm[i] = m2;
      }
    }
  }
  // The split's entry: the combined output and log-sum-exp of each head.
  const size_t entry = (size_t)seq * a.splits + split;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int hh = (4 * grp + i) & 7;
    if (hh < G) {
      float *dst = a.partial + (entry * a.hq + head0 + hh) * kD + col;
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int v = 0; v < 2; ++v)
          dst[16 * (4 * u + 2 * (grp >> 1) + v)] = ct[i] > 0.f ? cs[2 * u + v][i] / ct[i] : 0.f;
      if (col == 0 && grp < 2)
        a.lse[entry * a.hq + head0 + hh] = ct[i] > 0.f ? cm[i] + logf(ct[i]) : -INFINITY;
    }
  }
  // The reference's check of the split's combined weight: it fails when no stream of a
  // head has a finite log-sum-exp (a stream's is finite or -inf).
#pragma unroll
  for (int j = 0; j < 2; ++j)
    if (4 * j + grp < G)
      fine = fine && has[j];
  if (__ballot(!fine) != 0 && lane == 0)
    raise_bad(a.bad);
}

// ---- q8_0 split for few sequences -------------------------------------------------------
// k_q8_0_mx walks the four streams of a split one after the other, with a workgroup per (sequence,
// split) and a wave per KV head: one sequence ran 32 workgroups, 128 waves in all.  Here a
// workgroup takes one (sequence, split, KV head) and its four waves one stream each, so that four
// times the waves walk a quarter of the slices, without a
// barrier on the way; then each wave folds one row of every head's streams.  The query is
// coded here too, while the first slice is on its way, which saves that launch.  Every sum has the
// order it has in k_q8_0_mx: the bits are the same.
// A head's codes are a quarter of each 544-byte row, and the lines at its ends belong to two
// heads: the four heads of a split go to one XCD (workgroup ids 8 apart), whose L2 then holds
// them; the loads are ordinary ones for that.  With many workgroups the whole-row loads of
// k_q8_0_mx are better (the line ends then come from HBM twice).  Steps, k_q8_0_query and
// k_q8_0_mx -> this kernel (us, merge included; workgroups = splits x 4 x sequences):
//   1 sequence, 1000 / 32768 / 131072 keys (128)  20.6 -> 10.3, 71.5 -> 22.9, 237.6 -> 60.2
//   4 sequences, to 8000 keys (512)               29.8 -> 16.7
//   8 sequences (1024); 64 local rings (1024)     31.4 -> 26.8, 30.9 -> 28.4
//   16 sequences, 16 heads (2048)                 39.6 -> 41.4
//   64 sequences, 32768 keys (8192)               245.9 -> 301.9
constexpr int kStreamsMaxGroups = 1024;

// An ordinary 16-byte load as one vector value (a struct copy put the array in scratch memory).
__device__ __forceinline__ uint4 ld_cached(const uint8_t *p) {
  const u32x4_t v = *reinterpret_cast<const u32x4_t *>(p);
  return make_uint4(v.x, v.y, v.z, v.w);
}

template <class T> __global__ __launch_bounds__(256) void k_q8_0_streams(AttnArgs a) {
  // Per wave: the slice's K codes (32 keys of 8 chunks, exchanged by key), then its V codes as
  // BF16 (4 keys per dimension and group, at slot vq_slot<true>(d) ^ 16 flip(group)), then
  // the stream's outputs; block scales; probabilities by head.
  __shared__ __align__(16) uint2 image[kStreams][8][kD];
  __shared__ __align__(16) float ksc_all[kStreams][32][4], vsc_all[kStreams][4][32];
  __shared__ __align__(16) float ps_all[kStreams][8][36];
  __shared__ float dsum_all[kStreams][8], lse_all[kStreams][8];
  __shared__ __align__(16) int8_t qcodes[8][kD];
  __shared__ float qscale[8][4];
  const int lane = threadIdx.x & 63, s = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, grp = lane >> 4, G = a.group;
  const int kv = blockIdx.x >> 3, u = 8 * blockIdx.y + (blockIdx.x & 7);
  AttnUnit unit;
  const bool raise = kv == 0 && threadIdx.x == 0;
  if (a.units == AttnArgs::kRanked ? !attn_unit_ranked<kQ8Tile>(a, u, raise, unit)
                                   : u >= a.seqs * a.splits ||
                                         !attn_unit<kQ8Tile>(a, u / a.splits, u % a.splits, raise, unit))
    return; // block-uniform
  const int n = unit.n, head0 = kv * G;
  const size_t head_off = 32 + kD * (size_t)kv, scale_off = 8 * (size_t)kv;
  const uint8_t *krows = reinterpret_cast<const uint8_t *>(a.kc) +
                         (size_t)unit.seq * a.seq_stride * kRowBytes;
  const uint8_t *vrows = reinterpret_cast<const uint8_t *>(a.vc) +
                         (size_t)unit.seq * a.seq_stride * kRowBytes;
  uint4 *kq = reinterpret_cast<uint4 *>(&image[s][0][0]);
  auto &vq = image[s];
  auto &ksc = ksc_all[s];
  auto &vsc = vsc_all[s];
  auto &ps = ps_all[s];

  // Slice loads: K load m is key lane / 8 + 8 m, codes 16 (lane % 8) ..; V load m is key
  // 4 (lane / 8) + m; the four block scales of K row lane (lanes 0..31) or V row lane - 32.
  // Window offsets past the last key read the last key's row; their scales are zeroed (the
  // reference zero-fills both) and their scores masked.
  const uint32_t first_row = (uint32_t)(unit.first % a.cap);
  auto row_at = [&](int o) { // the window holds at most cap keys: one wrap
    const uint32_t r = first_row + (uint32_t)min(o, n - 1);
    return (size_t)min(r, r - (uint32_t)a.cap) * kRowBytes;
  };
  uint4 kw[4], vw[4];
  uint2 hw;
  auto load_slice = [&](int o0) {
#pragma unroll
    for (int m = 0; m < 4; ++m)
      kw[m] = ld_cached(krows + row_at(o0 + (lane >> 3) + 8 * m) + head_off + 16 * (lane & 7));
#pragma unroll
    for (int m = 0; m < 4; ++m)
      vw[m] = ld_cached(vrows + row_at(o0 + 4 * (lane >> 3) + m) + head_off + 16 * (lane & 7));
    hw = *reinterpret_cast<const uint2 *>((lane < 32 ? krows : vrows) + row_at(o0 + (lane & 31)) +
                                          scale_off);
  };
  // This wave's slices: keys 32 s .. 32 s + 31 of the split's tiles that lie in the window
  // (a slice past it would leave every value as it is).
  const int o_begin = unit.begin * kQ8Tile + 32 * s;
  const int o_end = min(unit.end * kQ8Tile, n);
  if (o_begin < o_end)
    load_slice(o_begin);

  bool fine = true;
#pragma unroll
  for (int k = 0; k < 2; ++k) { // wave s codes heads s and s + 4
    const int h = s + 4 * k;
    if (h < G) {
      const size_t o = ((size_t)unit.seq * a.hq + head0 + h) * kD + lane;
      fine = q8_0_code_query(act_value<T>(a.q, o), act_value<T>(a.q, o + 64), lane, qcodes[h],
                             qscale[h]) &&
             fine;
    }
  }
  __syncthreads();
  // Query A operands: row col = (head 4 j + col / 4, block col % 4); K-slot group grp of
  // step h covers dimensions 64 h + 16 grp .. + 15, of block 2 h + grp / 2.
  uint4 aq[2][2];
  float qd[2][4]; // block scales of head 4 j + grp
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int hh = 4 * j + (col >> 2);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      aq[j][h] = make_uint4(0, 0, 0, 0);
      if (hh < G && (col & 3) == 2 * h + (grp >> 1))
        aq[j][h] = *reinterpret_cast<const uint4 *>(&qcodes[hh][64 * h + 16 * grp]);
    }
#pragma unroll
    for (int b = 0; b < 4; ++b)
      qd[j][b] = 4 * j + grp < G ? qscale[4 * j + grp][b] : 0.f;
  }

  float mx[2] = {-INFINITY, -INFINITY}, den[2][2] = {{0.f, 0.f}, {0.f, 0.f}};
  f32x4_t o[8];
#pragma unroll
  for (int t = 0; t < 8; ++t)
    o[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // One slice; MORE: this wave's next one is loaded once the registers are free.
  auto slice = [&](int o0, auto more) {
    const uint4 va[4] = {vw[0], vw[1], vw[2], vw[3]};
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const int key = (lane >> 3) + 8 * m;
      kq[8 * key + ((lane & 7) ^ ((key >> 1) & 7))] = kw[m];
    }
    {
      const bool inside = o0 + (lane & 31) < n;
      const float4 d = make_float4(inside ? f16_bits(hw.x & 0xffffu) : 0.f,
                                   inside ? f16_bits(hw.x >> 16) : 0.f,
                                   inside ? f16_bits(hw.y & 0xffffu) : 0.f,
                                   inside ? f16_bits(hw.y >> 16) : 0.f);
      if (lane < 32) {
        *reinterpret_cast<float4 *>(&ksc[lane][0]) = d;
      } else {
        vsc[0][lane - 32] = d.x;
        vsc[1][lane - 32] = d.y;
        vsc[2][lane - 32] = d.z;
        vsc[3][lane - 32] = d.w;
      }
    }
    if constexpr (decltype(more)::value) {
      load_slice(o0 + kQ8Tile);
      issue_point();
    }
    // Scores: head 4 j + grp, key 16 k + col.
    float sc[2][2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const uint4 b0 = kq[8 * (16 * k + col) + (grp ^ (col >> 1))];
      const uint4 b1 = kq[8 * (16 * k + col) + ((4 + grp) ^ (col >> 1))];
      const float4 kd = *reinterpret_cast<const float4 *>(&ksc[16 * k + col][0]);
      const bool valid = o0 + 16 * k + col < n;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        i32x4_t d = mfma_i8(aq[j][0], b0, i32x4_t{0, 0, 0, 0});
        d = mfma_i8(aq[j][1], b1, d);
        float dot = 0.f;
        dot = __builtin_fmaf((float)d[0], kd.x * qd[j][0], dot);
        dot = __builtin_fmaf((float)d[1], kd.y * qd[j][1], dot);
        dot = __builtin_fmaf((float)d[2], kd.z * qd[j][2], dot);
        dot = __builtin_fmaf((float)d[3], kd.w * qd[j][3], dot);
        sc[k][j] = valid ? dot * kScoreScale : -INFINITY;
      }
    }
    // V takes the K codes' place (a wave's LDS accesses run in program order).
    {
      float f[4][16];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const uint32_t w[4] = {va[m].x, va[m].y, va[m].z, va[m].w};
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int b = 0; b < 4; ++b)
            f[m][4 * i + b] = (float)(int8_t)((w[i] >> (8 * b)) & 0xffu);
      }
      const int t7 = lane & 7, j = lane >> 3;
      uint2 *dst = &vq[j][(16 * t7) ^ (((j ^ (j >> 1)) & 1) << 4)];
#pragma unroll
      for (int e = 0; e < 16; e += 2)
        *reinterpret_cast<uint4 *>(dst + 2 * ((e / 2 + t7) & 7)) =
            make_uint4(pack2(f[0][e], f[1][e]), pack2(f[2][e], f[3][e]),
                       pack2(f[0][e + 1], f[1][e + 1]), pack2(f[2][e + 1], f[3][e + 1]));
    }
    float alpha[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float next = fmaxf(mx[j], row_max16(fmaxf(sc[0][j], sc[1][j])));
      alpha[j] = isfinite(mx[j]) ? __expf(mx[j] - next) : 0.f;
      mx[j] = next;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const float p = isfinite(sc[k][j]) ? __expf(sc[k][j] - next) : 0.f;
        den[k][j] = __builtin_fmaf(den[k][j], alpha[j], p);
        ps[4 * j + grp][16 * k + col] = p;
      }
    }
    // Rows 4 grp + i of the PV accumulators are head (4 grp + i) % 8, whose alpha lane 16 i
    // holds (alpha[0] for heads 0..3, alpha[1] for 4..7).
    if (__ballot(alpha[0] != 1.f || alpha[1] != 1.f) != 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float a0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(alpha[0]), 16 * i));
        const float a1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(alpha[1]), 16 * i));
        const float ar = (grp & 1) ? a1 : a0;
#pragma unroll
        for (int t = 0; t < 8; ++t)
          o[t][i] *= ar;
      }
    }
    // PV A operands: row col = (head col % 8, block 2 c + col / 8); K-slots of group grp are
    // keys 8 grp .. 8 grp + 7.
    uint4 ahi[2], alo[2];
    {
      const int hh = col & 7;
      const float4 p0 = *reinterpret_cast<const float4 *>(&ps[hh][8 * grp]);
      const float4 p1 = *reinterpret_cast<const float4 *>(&ps[hh][8 * grp + 4]);
      const float pv[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int b = 2 * c + (col >> 3);
        const float4 v0 = *reinterpret_cast<const float4 *>(&vsc[b][8 * grp]);
        const float4 v1 = *reinterpret_cast<const float4 *>(&vsc[b][8 * grp + 4]);
        const float vv[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
        uint32_t hi[4], lo[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float f0 = hh < G ? pv[2 * e] * vv[2 * e] : 0.f;
          const float f1 = hh < G ? pv[2 * e + 1] * vv[2 * e + 1] : 0.f;
          bf16_split2(f0, f1, hi[e], lo[e]);
        }
        ahi[c] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
        alo[c] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
      }
    }
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const int d = vq_slot<true>(16 * t + col) ^ ((grp & 1) << 4);
      const uint2 v0 = vq[2 * grp][d], v1 = vq[2 * grp + 1][d ^ 16];
      const uint4 bv = make_uint4(v0.x, v0.y, v1.x, v1.y);
      o[t] = mfma_bf16(ahi[t >> 2], bv, o[t]);
      o[t] = mfma_bf16(alo[t >> 2], bv, o[t]);
    }
  };
  int o0 = o_begin;
  for (; o0 + kQ8Tile < o_end; o0 += kQ8Tile)
    slice(o0, std::true_type{});
  if (o0 < o_end)
    slice(o0, std::false_type{});

  // Each stream's log-sum-exp (den over the 32 key positions) and outputs, for the fold.
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const float dsum = row_sum16(den[0][j] + den[1][j]);
    if (col == 0) {
      dsum_all[s][4 * j + grp] = dsum;
      lse_all[s][4 * j + grp] = dsum > 0.f ? mx[j] + logf(dsum) : -INFINITY;
    }
  }
  float *out = reinterpret_cast<float *>(&image[s][0][0]); // [8 tiles][4 rows][64 lanes]
#pragma unroll
  for (int t = 0; t < 8; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      out[64 * (4 * t + i) + lane] = o[t][i];
  __syncthreads();
  // Wave i = s folds row i of the PV layout (head (4 grp + i) % 8) over the streams in order,
  // with weight exp(lse - max), for this lane's four dimension tiles t = 4 u + 2 (grp / 2) + v;
  // streams without a finite log-sum-exp carry no weight.
  const int i = s, hh = (4 * grp + i) & 7;
  float cm = -INFINITY, ct = 0.f, cs[4] = {0.f, 0.f, 0.f, 0.f};
  bool has = false;
  for (int st = 0; st < kStreams; ++st) {
    const float d = dsum_all[st][hh], l = lse_all[st][hh];
    const float *from = reinterpret_cast<const float *>(&image[st][0][0]) + 64 * i + lane;
    float x[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      x[k] = from[256 * (4 * (k >> 1) + 2 * (grp >> 1) + (k & 1))];
    if (isfinite(l)) {
      has = true;
      const float m2 = fmaxf(cm, l);
      const float wa = isfinite(cm) ? expf(cm - m2) : 0.f, wb = expf(l - m2);
      ct = __builtin_fmaf(ct, wa, wb);
#pragma unroll
      for (int k = 0; k < 4; ++k)
        cs[k] = __builtin_fmaf(cs[k], wa, wb * (x[k] / d));
      cm = m2;
    }
  }
  // The split's entry: the combined output and log-sum-exp of each head.
  const size_t entry = (size_t)unit.seq * a.splits + unit.split;
  if (hh < G) {
    float *dst = a.partial + (entry * a.hq + head0 + hh) * kD + col;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      dst[16 * (4 * (k >> 1) + 2 * (grp >> 1) + (k & 1))] = ct > 0.f ? cs[k] / ct : 0.f;
    if (col == 0 && grp < 2)
      a.lse[entry * a.hq + head0 + hh] = ct > 0.f ? cm + logf(ct) : -INFINITY;
    // The reference's check of the split's combined weight: it fails when no stream of a
    // head has a finite log-sum-exp (a stream's is finite or -inf).
    fine = fine && has;
  }
  if (__ballot(!fine) != 0 && lane == 0)
    raise_bad(a.bad);
}

template <class T> __global__ __launch_bounds__(64) void k_q8_0_mx_merge(AttnArgs a) {
  const int head = blockIdx.x, seq = blockIdx.y, lane = threadIdx.x;
  const size_t entry = (size_t)seq * a.splits * a.hq + head, step = (size_t)a.hq * kD;
  const float *src = a.partial + entry * kD + 2 * lane;
  const bool early = gridDim.x * gridDim.y <= kEarlyHeads;
  const float lse = a.lse[entry + (size_t)min(lane & 31, a.splits - 1) * a.hq];
  float2 p[kMaxSplits];
  if (early)
    merge_load(src, step, a.splits, p);
  int n, first;
  if (!attn_window(a, seq, n, first) || (a.local && a.cap != 1024))
    return; // the split kernel raised the flag
  // One entry per active split (at most 32: lanes 0..31).
  const int active = min(a.splits, (n + kQ8Tile - 1) / kQ8Tile), l32 = lane & 31;
  if (!early)
    merge_load(src, step, active, p);
  const float v = l32 < active ? lse : -INFINITY;
  float mxv = v;
  mxv = xor_max32(mxv);
  const float e = isfinite(v) ? expf(v - mxv) : 0.f;
  float den = e;
  den = xor_sum32(den);
  const float weight = e / den;
  float s0, s1;
  merge_sum(p, weight, active, s0, s1);
  // Lane l has features 2l, 2l + 1; the transforms take l and l + 64.
  const int from = (lane >> 1), odd = lane & 1;
  const float a0 = __shfl(s0, from, 64), a1 = __shfl(s1, from, 64);
  const float b0 = __shfl(s0, from + 32, 64), b1 = __shfl(s1, from + 32, 64);
  float x0 = odd ? a1 : a0, x1 = odd ? b1 : b0;
  // back from the V rotation: two 64-point transforms (features lane and lane + 64)
  hadamard64_pair(x0, x1, lane);
  x0 *= .125f;
  x1 *= .125f;
  const uint32_t word = pack2(x0, x1); // lo: feature lane, hi: feature lane + 64
  if (__ballot(!isfinite(x0) || !isfinite(x1) || !(den > 0.f)) != 0 && lane == 0)
    raise_bad(a.bad);
  const size_t o = ((size_t)seq * a.hq + head) * kD;
  if constexpr (std::is_same<T, uint16_t>::value) {
    static_cast<uint16_t *>(a.out)[o + lane] = (uint16_t)(word & 0xffffu);
    static_cast<uint16_t *>(a.out)[o + 64 + lane] = (uint16_t)(word >> 16);
  } else {
    static_cast<float *>(a.out)[o + lane] = lo16(word);
    static_cast<float *>(a.out)[o + 64 + lane] = hi16(word);
  }
}

} // namespace

extern "C" long long padra_DecodeAttentionScratch(int format, int seqs, int q_heads,
                                                  int splits) {
  if (seqs < 1 || q_heads < 1 || splits < 1 || splits > 32 ||
      (format != PADRA_KV_BF16 && format != PADRA_KV_Q8 && format != PADRA_KV_Q8_0))
    return -1;
  // partial outputs and log-sum-exps per split, rounded up to 16 bytes
  const long long base = ((long long)seqs * splits * q_heads * (kD + 1) + 3) & ~3ll;
  // q8_0: the coded query (128 bytes) and its 4 block scales per head, after the lse
  const long long query = format == PADRA_KV_Q8_0 ? (long long)seqs * q_heads * (kD / 4 + 4) : 0;
  // then the split kernels' dispatch order, one int per sequence, rounded up to 16 bytes
  return base + query + ((seqs + 3) & ~3ll);
}

namespace {
// The reference's split counts: q8_0 16 (local) or 32; otherwise one per 32 keys of the
// ring, at most 16 (local) or 32.
int reference_splits(const padra_KVCache *kv, int local) {
  if (kv->format == PADRA_KV_Q8_0)
    return local ? 16 : 32;
  return std::min((kv->cap + kKeys - 1) / kKeys, local ? 16 : 32);
}

// The split count for splits = -1.  Global windows keep the reference's count (within 1.5% of the
// best of 8-32 at 64 sequences).  A local ring's 1024-key windows take fewer splits the more
// sequences there are: about 1,024 one-wave splits for BF16 and q8_0 and 2,048 for q8, which was the
// best of a sweep when every split was one wave.  It is kept as callers' results and scratch sizes
// follow it.  This count against the reference's 16 as the kernels are (us, 32 query heads; 1, 8,
// 12, 24, 64 sequences):
//   BF16   9.1 :  9.1  12.7 : 12.7  14.7 : 14.8  19.6 : 21.0  32.7 : 40.5
//   q8    10.0 : 10.0  13.9 : 13.2  17.2 : 14.9  22.5 : 20.7  28.4 : 34.9
//   q8_0  11.0 : 11.6  15.5 : 15.6  16.4 : 16.4  23.1 : 29.1  33.9 : 51.2
// For q8 it is thus the slower choice from 4 to 32 sequences, as it was with one wave a split
// (12: 17.7 : 15.2).
int tuned_splits(const padra_KVCache *kv, int local, int seqs, int kv_heads) {
  if (!local)
    return reference_splits(kv, local);
  const int per_seq = std::max(1, seqs);
  if (kv->format == PADRA_KV_Q8_0)
    return std::clamp(256 / per_seq, 4, 16);
  const int waves = kv->format == PADRA_KV_Q8 ? 2048 : 1024;
  const int cap_splits = std::min((kv->cap + kKeys - 1) / kKeys, kv->format == PADRA_KV_Q8 ? 32 : 16);
  return std::clamp(waves / (per_seq * std::max(1, kv_heads)), std::min(2, cap_splits), cap_splits);
}

// splits as passed (1..32), 0: the reference's count, -1: the tuned count; 0 if invalid.
int resolve_splits(const padra_KVCache *kv, int local, int seqs, int kv_heads, int splits) {
  if (splits == 0)
    return reference_splits(kv, local);
  if (splits == -1)
    return tuned_splits(kv, local, seqs, kv_heads);
  return splits >= 1 && splits <= 32 ? splits : 0;
}

// Both entry points: packed/scales non-null selects the merge with the FP8 encoding.
int decode_attention(void *stream, const void *q, const padra_KVCache *kv, void *out,
                     uint8_t *packed, float *scales, const padra_Positions *pos, int seqs,
                     int q_heads, int kv_heads, int local, int splits, float *scratch,
                     long long scratch_floats, int *bad, int act) {
  if (!q || !kv || !out || !pos || !bad || !scratch || seqs < 1 || q_heads < 1 ||
      kv_heads < 1 || q_heads % kv_heads || !kv->k || !kv->v || kv->cap < 1 ||
      kv->cap > 131072 || pos->mode != PADRA_POS_DECODE || !pos->decode || pos->maximum < 1 ||
      pos->maximum > 131072 || pos->vocab < 1 || (seqs > 1 && kv->seq_stride < kv->cap) ||
      (act != PADRA_ACT_BF16 && act != PADRA_ACT_F32) || !aligned16(kv->k) ||
      !aligned16(kv->v) || !aligned16(scratch) || splits < -1 || splits > 32)
    return PADRA_INVALID_ARGUMENT;
  if (kv->format != PADRA_KV_BF16 && kv->format != PADRA_KV_Q8 && kv->format != PADRA_KV_Q8_0)
    return PADRA_UNSUPPORTED;
  if (kv->format == PADRA_KV_Q8 && !kv->scales)
    return PADRA_INVALID_ARGUMENT;
  const bool fp8 = packed != nullptr;
  if (fp8 && (!scales || q_heads > 32 || (reinterpret_cast<uintptr_t>(packed) & 1) ||
              (reinterpret_cast<uintptr_t>(scales) & 3)))
    return PADRA_INVALID_ARGUMENT;
  if (fp8 && kv->format == PADRA_KV_Q8_0)
    return PADRA_UNSUPPORTED; // the reference's q8_0 merge has no FP8 form
  const bool q8 = kv->format == PADRA_KV_Q8_0, q8s = kv->format == PADRA_KV_Q8;
  if (q8 && kv_heads * kD != 512)
    return PADRA_UNSUPPORTED; // the 544-byte q8_0 row of 4 KV heads
  splits = resolve_splits(kv, local, seqs, kv_heads, splits);
  const long long need = padra_DecodeAttentionScratch(kv->format, seqs, q_heads, splits);
  if (scratch_floats < need)
    return PADRA_INVALID_ARGUMENT;
  AttnArgs a{};
  a.q = q;
  a.kc = static_cast<const uint16_t *>(kv->k);
  a.vc = static_cast<const uint16_t *>(kv->v);
  a.out = out;
  // scratch: partial [seqs][splits][hq][128], lse [seqs][splits][hq], then (q8_0 only,
  // from the next 16-byte boundary) coded query [seqs][hq][128] bytes and query block
  // scales [seqs][hq][4]; the end is exactly padra_DecodeAttentionScratch's count
  const long long entries = (long long)seqs * splits * q_heads;
  const long long qbase = (entries * (kD + 1) + 3) & ~3ll;
  a.partial = scratch;
  a.lse = scratch + entries * kD;
  a.qcodes = reinterpret_cast<int8_t *>(scratch + qbase);
  a.qscale = scratch + qbase + (long long)seqs * q_heads * (kD / 4);
  // Units longest first, without the inactive ones, when the lengths can differ much: several
  // sequences on a global cache (a local ring's windows are at most 1024 keys).
  const long long obase = qbase + (q8 ? (long long)seqs * q_heads * (kD / 4 + 4) : 0);
  a.order = reinterpret_cast<int *>(scratch + obase);
  a.units = seqs < 2 || seqs > kOrderMaxSeqs || local ? AttnArgs::kPlain
            : seqs <= kRankMaxSeqs                    ? AttnArgs::kRanked
                                                      : AttnArgs::kOrdered;
  a.decode = pos->decode;
  a.seqs = seqs;
  a.hq = q_heads;
  a.hkv = kv_heads;
  a.group = q_heads / kv_heads;
  a.cap = kv->cap;
  a.local = local ? 1 : 0;
  a.splits = splits;
  a.maximum = pos->maximum;
  a.vocab = pos->vocab;
  a.seq_stride = seqs > 1 ? kv->seq_stride : 0;
  a.bad = bad;
  a.kvscales = static_cast<const float *>(kv->scales);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  // The heads of a split side by side: with the heads outermost each would bring its own tail
  // of inactive splits (8 sequences of 8000 keys 24.1 -> 25.9 us).
  const bool plain = a.units == AttnArgs::kPlain;
  const dim3 split_grid = plain ? dim3(kv_heads, splits, seqs) : dim3(kv_heads, splits * seqs);
  const dim3 q8_grid = plain ? dim3(1, splits, seqs) : dim3(1, splits * seqs);
  const dim3 merge_grid(q_heads, seqs);
  const int group = q_heads / kv_heads;
  if (group != 1 && group != 2 && group != 4 && group != 8)
    return PADRA_UNSUPPORTED;
  auto launch = [&](auto tag) -> int {
    using T = decltype(tag);
    if (a.units == AttnArgs::kOrdered && !q8) // (the q8_0 query kernel ranks them itself)
      hipLaunchKernelGGL(k_attn_order, dim3(seqs), dim3(64), 0, s, a);
    if (q8 && splits * kv_heads * seqs <= kStreamsMaxGroups) {
      hipLaunchKernelGGL((k_q8_0_streams<T>), dim3(8 * kv_heads, (splits * seqs + 7) / 8), dim3(256),
                         0, s, a);
      hipLaunchKernelGGL((k_q8_0_mx_merge<T>), merge_grid, dim3(64), 0, s, a);
      return launched("DecodeAttention");
    }
    if (q8) {
      hipLaunchKernelGGL((k_q8_0_query<T>), merge_grid, dim3(64), 0, s, a);
      switch (group) {
      case 1:
        hipLaunchKernelGGL((k_q8_0_mx<1>), q8_grid, dim3(256), 0, s, a);
        break;
      case 2:
        hipLaunchKernelGGL((k_q8_0_mx<2>), q8_grid, dim3(256), 0, s, a);
        break;
      case 4:
        hipLaunchKernelGGL((k_q8_0_mx<4>), q8_grid, dim3(256), 0, s, a);
        break;
      default:
        hipLaunchKernelGGL((k_q8_0_mx<8>), q8_grid, dim3(256), 0, s, a);
        break;
      }
      hipLaunchKernelGGL((k_q8_0_mx_merge<T>), merge_grid, dim3(64), 0, s, a);
      return launched("DecodeAttention");
    }
    auto split = [&](auto q8tag, auto wtag) {
      constexpr bool Q8 = decltype(q8tag)::value;
      constexpr int W = decltype(wtag)::value;
      hipLaunchKernelGGL((k_attn_mx<T, Q8, W>), split_grid, dim3(64 * W), 0, s, a);
    };
    // Waves per workgroup, by how many workgroups the launch has: with few of them one wave
    // each leaves most of the chip idle, with many the round's barriers cost more than its
    // waves bring.  Measured (us, split and merge, W = 1 / 2 / 4 / 8; BF16, then q8):
    //   1 sequence, 32768 keys, 32 heads (128 workgroups)  45.7/36.2/27.5/26.4  72.0/47.4/29.7/25.9
    //   4 sequences, to 8000 keys, 32 heads (512)          21.9/19.3/17.9/21.8  27.7/21.3/17.2/21.5
    //   8 sequences, the same (1024)                       27.2/25.3/27.8/36.4  29.1/24.9/25.9/36.8
    //   16 sequences, 16 heads (2048)                      36.6/37.0/43.6/62.9  32.2/34.6/38.4/64.0
    // and on local rings, whose splits have two tiles (waves without a tile still divide PV):
    //   1 ring, 32 heads (64)                              10.5/9.5/9.2/9.1     12.5/10.4/10.1/10.0
    //   4 rings (256)                                      11.3/10.8/10.4/10.4  12.9/11.2/10.9/10.8
    //   8 rings (512)                                      13.4/13.4/13.1/16.6  14.0/13.5/13.2/16.8
    //   12 rings (768)                                     14.8/15.2/18.5/22.6  15.1/14.8/15.1/23.2
    const int wgs = splits * kv_heads * seqs;
    auto split_w = [&](auto q8tag) {
      if (wgs <= 256)
        split(q8tag, std::integral_constant<int, 8>{});
      else if (wgs <= 512)
        split(q8tag, std::integral_constant<int, 4>{});
      else if (wgs <= 1024 && !local) // a local ring's split has two tiles or so: 15.2 us
                                      // with two waves, 14.9 with one (12 sequences)
        split(q8tag, std::integral_constant<int, 2>{});
      else if (decltype(q8tag)::value && wgs > 2048) // (k_attn_mx, DENSE)
        hipLaunchKernelGGL((k_attn_mx<T, true, 1, true>), split_grid, dim3(64), 0, s, a);
      else
        split(q8tag, std::integral_constant<int, 1>{});
    };
    if (q8s)
      split_w(std::true_type{});
    else
      split_w(std::false_type{});
    hipLaunchKernelGGL((k_attn_merge<T>), merge_grid, dim3(64), 0, s, a);
    if (fp8)
      hipLaunchKernelGGL((k_attn_encode_fp8<T>), dim3(seqs), dim3(256), 0, s, a, packed, scales);
    return launched("DecodeAttention");
  };
  return act == PADRA_ACT_BF16 ? launch(uint16_t{}) : launch(float{});
}
} // namespace

extern "C" int padra_DecodeAttentionSplits(const padra_KVCache *kv, int seqs, int kv_heads,
                                           int local, int splits) {
  if (!kv || seqs < 1 || kv_heads < 1 || kv->cap < 1 || splits < -1 || splits > 32 ||
      (kv->format != PADRA_KV_BF16 && kv->format != PADRA_KV_Q8 && kv->format != PADRA_KV_Q8_0))
    return -1;
  return resolve_splits(kv, local, seqs, kv_heads, splits);
}


extern "C" int padra_DecodeAttention(void *stream, const void *q, const padra_KVCache *kv,
                                     void *out, const padra_Positions *pos, int seqs,
                                     int q_heads, int kv_heads, int local, int splits,
                                     float *scratch, long long scratch_floats, int *bad,
                                     int act) {
  return decode_attention(stream, q, kv, out, nullptr, nullptr, pos, seqs, q_heads, kv_heads,
                          local, splits, scratch, scratch_floats, bad, act);
}

extern "C" int padra_DecodeAttentionFP8(void *stream, const void *q, const padra_KVCache *kv,
                                        void *out, uint8_t *packed, float *scales,
                                        const padra_Positions *pos, int seqs, int q_heads,
                                        int kv_heads, int local, int splits, float *scratch,
                                        long long scratch_floats, int *bad, int act) {
  if (!packed)
    return PADRA_INVALID_ARGUMENT;
  return decode_attention(stream, q, kv, out, packed, scales, pos, seqs, q_heads, kv_heads,
                          local, splits, scratch, scratch_floats, bad, act);
}

// ---- the entry point that allocates nothing ---------------------------------------------
//
// padra_DecodeAttentionNoAlloc's workspace: a fixed array in device memory, one copy per
// GPU the library runs on, held until the process ends.  Its name is a host-side
// stand-in, not a device address: host code uses only the address hipGetSymbolAddress
// returns for the current device (scratch_address below).
static __device__ __align__(256) float scratch[PADRA_DECODE_ATTENTION_STATIC_FLOATS];

namespace {
constexpr int kMaxDevices = 64;
std::atomic<float *> g_scratch_address[kMaxDevices];
std::mutex g_scratch_mutex;

// The array's device address on the current device, looked up on the first call there;
// null when the lookup fails.
float *scratch_address() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return nullptr;
  float *p = g_scratch_address[dev].load(std::memory_order_acquire);
  if (p)
    return p;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  p = g_scratch_address[dev].load(std::memory_order_relaxed);
  if (!p) {
    void *address = nullptr;
    const hipError_t e = hipGetSymbolAddress(&address, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !address) {
      fprintf(stderr, "padra: DecodeAttentionNoAlloc: workspace lookup failed: %s\n",
              hipGetErrorString(e));
      return nullptr;
    }
    p = static_cast<float *>(address);
    g_scratch_address[dev].store(p, std::memory_order_release);
  }
  return p;
}
} // namespace

extern "C" int padra_DecodeAttentionNoAlloc(void *stream, const void *q, const padra_KVCache *kv,
                                            void *out, const padra_Positions *pos, int seqs,
                                            int q_heads, int kv_heads, int local, int splits,
                                            int *bad, int act) {
  if (!kv || splits < -1 || splits > 32)
    return PADRA_INVALID_ARGUMENT;
  splits = resolve_splits(kv, local, seqs, kv_heads, splits);
  const long long need = padra_DecodeAttentionScratch(kv->format, seqs, q_heads, splits);
  if (need < 0)
    return PADRA_INVALID_ARGUMENT;
  if (need > PADRA_DECODE_ATTENTION_STATIC_FLOATS) {
    fprintf(stderr,
            "padra: DecodeAttentionNoAlloc: %lld workspace floats needed (%d sequences, %d "
            "query heads), the fixed workspace holds %d; use padra_DecodeAttention\n",
            need, seqs, q_heads, PADRA_DECODE_ATTENTION_STATIC_FLOATS);
    return PADRA_INVALID_ARGUMENT;
  }
  float *ws = scratch_address();
  if (!ws)
    return PADRA_INTERNAL;
  return decode_attention(stream, q, kv, out, nullptr, nullptr, pos, seqs, q_heads, kv_heads,
                          local, splits, ws, PADRA_DECODE_ATTENTION_STATIC_FLOATS, bad, act);
}
