// GPU decode of the reference's own rANS-family bf16 formats:
//   bf16_parallel_v1   (bigsmall/codecs/bf16_parallel.py:262-352, streams via rans.py:165-207)
//   bf16_se_tans       (bigsmall/codecs/bf16_tans.py:121-167, streams via numba_rans.py:168-192)
//   bf16_se_single_kernel (bigsmall/codecs/single_kernel.py:431-580)
//
// All three code a bf16 word as a sign+exponent ("SE", 9-bit) symbol with
// rANS M = 4096, plus the 7-bit mantissa with a per-exponent rANS table
// (M = 1024), in "buckets": the mantissas of the elements that share an
// exponent, in element order (a stable sort by exponent). The state machine is
// the same everywhere: 32-bit state, L = 2^16, 16-bit renormalisation,
//   slot = x & (M-1); s = sym(slot); x = f*(x >> log2 M) + slot - cf;
//   while (x < L && words remain) x = (x << 16) | next_word;
// The formats differ only in framing, which the host resolves into the
// stream descriptors below (initial state, word array, optional odd trailing
// byte that reads as one more word).
//
// Decoding is two launches on one stream:
//   1. se_kernel: one lane per SE stream (bf16_parallel_v1 has N interleaved
//      streams, the other two formats one). Writes sign<<15 | exp<<7 of every
//      element, and the element's index into `perm` at the next free position
//      of its (stream, exponent) bucket: per-lane cursors in LDS give the
//      stable-sort rank without any sort.
//   2. mant_kernel: one lane per bucket. Decodes the bucket's mantissas in
//      order and ORs mantissa r into element perm[bucket_begin + r].
// The SE decode tables sit in LDS; mantissa tables (1024 entries per
// exponent, up to 256 of them) are read through the caches.
#include <stdint.h>

#include <type_traits>

#include "simt.h"

#include "../../include/bigsmall_hip.h"
#include "lds_limit.h"

namespace {


constexpr uint32_t kL = 1u << 16;
constexpr int kWave = 64;
constexpr int kSeLanes = 64;        // SE streams per workgroup (one wavefront)
constexpr int kMantThreads = 64;

__device__ __forceinline__ uint32_t word_at(const GLB uint8_t* w, uint32_t i) {
  return (uint32_t)w[2 * i] | ((uint32_t)w[2 * i + 1] << 8);   // byte loads: any alignment
}

// One renormalisation with the reference's loop: while the state is below L
// and words remain, shift one in. The optional tail is the last "word".
__device__ __forceinline__ void renorm(uint32_t& x, uint32_t& pos, uint32_t n_eff, const GLB uint8_t* w,
                                       uint32_t n_words, uint32_t tail) {
  while (x < kL && pos < n_eff) {
    const uint32_t v = pos < n_words ? word_at(w, pos) : (tail & 0xFFFFu);
    x = (x << 16) | v;
    ++pos;
  }
}

__device__ __forceinline__ void flag(int32_t* status, int32_t bits) { atomicOr(status, bits); }

// SE table (LDS): slot -> {f | (slot - cf) << 13, symbol}
__global__ __launch_bounds__(kSeLanes) void se_kernel(const bs_se_stream* __restrict__ streams, uint32_t n_streams,
                                                      const uint32_t* __restrict__ se_table,
                                                      const uint32_t* __restrict__ bstart, uint64_t n_out,
                                                      uint16_t* __restrict__ out, uint32_t* __restrict__ perm,
                                                      int32_t* __restrict__ status) {
  BS_DYNAMIC_LDS(smem);
  LDS uint64_t* s_tbl = (LDS uint64_t*)smem;                   // 4096 entries
  LDS uint32_t* s_cur = (LDS uint32_t*)(smem + 4096 * 8);      // cursor of exponent e for lane l at e*64 + l
  const uint32_t lane = threadIdx.x;
  for (uint32_t i = lane; i < 4096; i += kSeLanes)
    s_tbl[i] = (uint64_t)se_table[2 * i] | ((uint64_t)se_table[2 * i + 1] << 32);
  const uint32_t sid = blockIdx.x * kSeLanes + lane;
  const bool live = sid < n_streams;
  const GLB uint32_t* bs = (const GLB uint32_t*)bstart + (uint64_t)(live ? sid : 0) * 257;
  for (uint32_t e = 0; e < 256; ++e) s_cur[e * kSeLanes + lane] = live ? bs[e] : 0u;
  __syncthreads();
  if (!live) return;

  const bs_se_stream S = streams[sid];
  const GLB uint8_t* w = (const GLB uint8_t*)S.words;
  const uint32_t n_eff = S.n_words + ((S.tail >> 16) & 1u);
  uint32_t x = S.x0, pos = 0;
  uint64_t idx = S.first;
  const uint32_t pend = bs[256];   // the stream's perm region ends here: no write goes past it
  bool bad = false;
  for (uint32_t i = 0; i < S.n; ++i, idx += S.stride) {
    const uint64_t ent = s_tbl[x & 4095u];
    const uint32_t lo = (uint32_t)ent, sym = (uint32_t)(ent >> 32);
    x = (lo & 0x1FFFu) * (x >> 12) + (lo >> 13);
    renorm(x, pos, n_eff, w, S.n_words, S.tail);
    const uint32_t e = sym & 0xFFu;
    const uint32_t p = s_cur[e * kSeLanes + lane];
    if (idx < n_out && p < pend) {
      out[idx] = (uint16_t)((((sym >> 8) & 1u) << 15) | (e << 7));
      perm[p] = (uint32_t)idx;
      s_cur[e * kSeLanes + lane] = p + 1;
    } else {
      bad = true;   // more elements than the stream's buckets hold, or a bad index
    }
  }
  // every bucket must be exactly full: the header's bucket sizes match the
  // decoded exponents (a bucket overfilled into its neighbour leaves one short)
  for (uint32_t e = 0; e < 256; ++e) bad |= s_cur[e * kSeLanes + lane] != bs[e + 1];
  if (bad) flag(status, BS_DEV_ERR_COUNT);
  if (x != kL || pos != n_eff) flag(status, BS_DEV_ERR_STREAM);
}

// Mantissa table (global): table*1024 + slot -> f | (slot - cf) << 11 | symbol << 21
__global__ __launch_bounds__(kMantThreads) void mant_kernel(const bs_mant_bucket* __restrict__ buckets,
                                                            uint32_t n_buckets, const uint32_t* __restrict__ tables,
                                                            uint32_t n_tables, const uint32_t* __restrict__ perm,
                                                            uint64_t n_perm, uint64_t n_out,
                                                            uint16_t* __restrict__ out, int32_t* __restrict__ status) {
  const uint32_t bid = blockIdx.x * kMantThreads + threadIdx.x;
  if (bid >= n_buckets) return;
  const bs_mant_bucket B = buckets[bid];
  if (B.table >= n_tables || B.perm_begin + B.n > n_perm) {
    flag(status, BS_DEV_ERR_HEADER);
    return;
  }
  const GLB uint32_t* tbl = (const GLB uint32_t*)tables + (uint64_t)B.table * 1024;
  const GLB uint8_t* w = (const GLB uint8_t*)B.words;
  const uint32_t n_eff = B.n_words + ((B.tail >> 16) & 1u);
  uint32_t x = B.x0, pos = 0;
  bool bad = false;
  for (uint32_t r = 0; r < B.n; ++r) {
    const uint32_t ent = tbl[x & 1023u];
    x = (ent & 0x7FFu) * (x >> 10) + ((ent >> 11) & 0x3FFu);
    renorm(x, pos, n_eff, w, B.n_words, B.tail);
    const uint32_t idx = perm[B.perm_begin + r];
    if (idx < n_out) out[idx] |= (uint16_t)((ent >> 21) & 0x7Fu);
    else bad = true;
  }
  if (bad) flag(status, BS_DEV_ERR_COUNT);
  if (x != kL || pos != n_eff) flag(status, BS_DEV_ERR_STREAM);
}

// ---- wave-serial path: every SE stream (one for bf16_se_tans and
// bf16_se_single_kernel, N interleaved ones for bf16_parallel_v1) is a chain
// decoded by its own wavefront, and so is every mantissa bucket unless many
// buckets share a table (lane_chains, below).
//
// A wavefront's chain keeps its state in a scalar register and its symbols
// spread over the lanes (serial_chain), or, with many symbols, reads a table
// (table_chain); the lanes also load the word stream 1 KB at a time into an LDS
// byte ring one segment ahead of use, hold a 64-word window of it, and keep the
// symbols of 64 steps (lane j: step j) for one coalesced store. The SE chain
// writes sign<<15 | exp<<7 of every element and counts the exponents of each tile of kTile symbols of its
// stream; the mantissa chains, which do not depend on it, run at the same time
// in other workgroups and write their bucket's mantissas in bucket order. Two
// parallel passes then give every element its position in its (stream,
// exponent) bucket (a stable counting sort by exponent within each stream: a
// scan of the tile counts over the stream's tiles, then per-tile ranks by
// wavefront ballots) and OR in its mantissa.

constexpr uint32_t kRingB = 2048;     // word-stream byte ring per chain (two segments: one landed, one in flight)
constexpr uint32_t kSegB = 1024;      // bytes per cooperative load (64 lanes x 16 B)
constexpr uint32_t kTile = 16384;     // elements per tile of the placement passes
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// This lane's 16 bytes of ring segment q of a stream whose bytes are
// [s_off, e_off) relative to the 16-byte aligned address A. Bytes outside that
// range are never read (they come back as zero).
__device__ __forceinline__ u32x4 seg_block(const GLB uint8_t* A, uint64_t q, uint32_t lane, uint64_t s_off,
                                           uint64_t e_off) {
  const uint64_t b0 = q * kSegB + lane * 16u;
  if (b0 >= s_off && b0 + 16u <= e_off) return *(const GLB u32x4*)(A + b0);
  u32x4 r = {0u, 0u, 0u, 0u};
#pragma unroll
  for (uint32_t k = 0; k < 16; ++k) {
    const uint64_t b = b0 + k;
    if (b >= s_off && b < e_off) r[k >> 2] |= (uint32_t)A[b] << (8u * (k & 3u));
  }
  return r;
}

__device__ __forceinline__ void seg_land(LDS uint8_t* ring, uint64_t q, uint32_t lane, u32x4 v) {
  *(LDS u32x4*)(ring + ((q * kSegB + lane * 16u) & (kRingB - 1u))) = v;
}

// A stream descriptor every pass of the serial path may use: at most max_len
// symbols (what the placement tiles cover) and every element index inside the
// output. The chain and placement kernels check it alike, so a bad
// descriptor is reported and skipped, never followed.
__device__ __forceinline__ bool stream_ok(const bs_se_stream& S, uint64_t max_len, uint64_t n_out) {
  return S.n <= max_len && S.stride != 0 && (S.n == 0 || S.first + (uint64_t)(S.n - 1) * S.stride < n_out);
}

// Exponent counts of an SE chain, kept in the wave's own 256 LDS bins for
// the current tile of kTile symbols and written to ghist[tile][256] when the
// tile ends (symbols [i0, i0 + cnt) are this batch, lane j holding output
// word j; a stream of n symbols). Counting here, one LDS add per lane per 64
// steps, replaced a pass that read every output word back with a stride of
// n_streams elements (1.6 of 39 ms for an 8B layer in bf16_parallel_v1).
__device__ __forceinline__ void tile_count(LDS uint32_t* hist, GLB uint32_t* ghist, uint32_t word, uint32_t lane,
                                           uint32_t i0, uint32_t cnt, uint32_t n) {
  if (cnt == (uint32_t)kWave || lane < cnt) BS_LDS_ADD(hist + ((word >> 7) & 0xFFu), 1u);
  const uint32_t end = i0 + cnt;
  if (end % kTile == 0 || end == n) {
    wave_sync();
    GLB uint32_t* g = ghist + (uint64_t)(i0 / kTile) * 256u;
    for (uint32_t b = lane; b < 256; b += kWave) {
      g[b] = hist[b];
      hist[b] = 0;
    }
    wave_sync();
  }
}
// Before an SE chain: empty bins. After it: zero counts for the tiles its n
// symbols do not reach (of the task's tps per stream).
__device__ __forceinline__ void tile_count_begin(LDS uint32_t* hist, uint32_t lane) {
  for (uint32_t b = lane; b < 256; b += kWave) hist[b] = 0;
  wave_sync();
}
__device__ __forceinline__ void tile_count_end(GLB uint32_t* ghist, uint32_t lane, uint32_t n, uint32_t tps) {
  for (uint64_t i = ((uint64_t)n + kTile - 1) / kTile * 256u + lane; i < (uint64_t)tps * 256u; i += kWave) ghist[i] = 0;
}

__device__ __forceinline__ uint32_t uni32(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ uint64_t uni64(uint64_t v) {
  return (uint64_t)uni32((uint32_t)v) | ((uint64_t)uni32((uint32_t)(v >> 32)) << 32);
}

// A chain's words: its bytes go through the wave's LDS ring, loaded a segment
// ahead of use, into a window of 64 words: lane l of `win` holds word base + l
// (past the stream: the tail word). A step takes at most one word, so a window
// moved on when the chain has taken kHalf of it lasts another kHalf steps.
constexpr uint32_t kHalf = 32;           // steps between looks at the window
struct WordWindow {
  const GLB uint8_t* A;                  // the stream starts at A + s_off, A 16-byte aligned
  uint32_t s_off, n_words, tail_word;
  uint64_t e_off;
  LDS uint8_t* ring;
  uint64_t landed = 0;                   // stream bytes [.., landed) are in the ring (relative to A)
  bool inflight = false;                 // segment `landed / kSegB` is being loaded into `seg`
  u32x4 seg = {0u, 0u, 0u, 0u};
  uint32_t base = 0, win = 0;
  __device__ __forceinline__ WordWindow(const GLB uint8_t* words, uint32_t n, uint32_t tail, LDS uint8_t* r)
      : n_words(n), tail_word(tail & 0xFFFFu), ring(r) {
    const uint64_t wa = uni64((uint64_t)words);
    A = (const GLB uint8_t*)(wa & ~15ull);
    s_off = (uint32_t)(wa & 15u);
    e_off = s_off + 2ull * n_words;
  }
  // moves the window on by `taken` words
  __device__ __forceinline__ void move(uint32_t taken, uint32_t lane) {
    base = uni32(base + taken);
    const uint64_t consumed = s_off + 2ull * base;
    if (inflight) {
      seg_land(ring, landed / kSegB, lane, seg);
      landed += kSegB;
      inflight = false;
    }
    while (landed < e_off && landed < consumed + 2u * kWave + 2u) {
      seg_land(ring, landed / kSegB, lane, seg_block(A, landed / kSegB, lane, s_off, e_off));
      landed += kSegB;
    }
    if (landed < e_off && landed + kSegB <= consumed + kRingB) {
      seg = seg_block(A, landed / kSegB, lane, s_off, e_off);
      inflight = true;
    }
    wave_sync();
    const uint32_t b = s_off + 2u * (base + lane);
    win = (uint32_t)ring[b & (kRingB - 1u)] | ((uint32_t)ring[(b + 1u) & (kRingB - 1u)] << 8);
    win = base + lane < n_words ? win : tail_word;
  }
};

// Decode one chain of n symbols with the symbols spread over the lanes: lane l
// holds symbols l*R .. l*R + R-1 (in slot order: f and cf of each), and no table
// is read. A step forms in every lane the state its symbol would give,
//   c = f * (x >> log2 M) + (x mod M) - cf  =  x - cf - (M - f) * (x >> log2 M),
// and that state renormalised with the chain's next word; the one lane whose
// interval [cf, cf + sum of its f) holds the slot is found by a ballot, and a
// readlane takes its state as the wave's next (x is uniform, in a scalar
// register). The interval test runs on the slot shifted to the top of the word
// (x << (32 - log2 M)), so it needs no mask and covers f = M.
//
// What bounds it: one wavefront's in-order issue (about 4.2 cycles per
// instruction, 8.3 where one uses the last one's result, about 21 from a vector
// instruction that writes a scalar register to the next scalar instruction),
// since a chain is serial by its format. Hence no branch in the step (34 cycles
// taken, 20 not taken, and a renormalisation every sixth step behind it) and no
// table read (a scalar load through its cache 60 cycles and more, an LDS read 56).
// MI355X, ns per step with everything around it: 31 with at most 64 symbols, 45 with
// up to 128 (54-57 with a table in the scalar cache, 68-77 with one in LDS). A layer of
// 2048 x 5632 in bf16_parallel_v1 5.62 -> 3.57 ms, 4096 x 14336 28.3 -> 17.7 ms, a layer
// of 512 x 1408 in bf16_se_tans 44.9 -> 22.6 ms (the lane-wise mantissas included).
//
// Renormalisation: the reference loops `while x < L and words remain`. From a
// state x >= L one decode step leaves x >= 2^4 (SE) or 2^6 (mantissa), so one
// shifted-in word restores x >= L: a valid stream never takes the loop twice,
// and an initial state below L, which no encoder writes, is reported as a
// corrupt stream. A corrupt stream that runs out of words shifts in its tail
// word (zero when it has none) and fails the end-of-stream check.

// A symbol of a chain's table in LDS: f | cf << 16, and its output (SE: the
// word sign<<15 | exp<<7; mantissa: the 7 bits).
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// This lane's symbols, from the list in LDS (`live` of them, in slot order).
template <int R, bool SE>
struct LaneSyms {
  int32_t nf[R];         // f - M
  uint32_t cf[R];
  uint32_t first;        // -(cf of the first) << (32 - log2 M)
  uint32_t last;         // (the lane's slots << (32 - log2 M)) - 1: the interval test's bound
  uint32_t bound[R];     // states below this renormalise: the symbol's decode is below L for x < the encode of L
  uint32_t begin[R];     // (cf - first cf) << (32 - log2 M) of symbols 1 .. R-1
  __device__ __forceinline__ void load(const LDS u32x2* syms, uint32_t live, uint32_t lane) {
    constexpr uint32_t kM = SE ? 4096u : 1024u, kTop = SE ? 20u : 22u;
    uint32_t slots = 0, cf0 = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const uint32_t i = lane * R + r;
      const uint32_t e = syms[min(i, live - 1u)].x;
      const uint32_t f = i < live ? e & 0xFFFFu : 0u;
      cf[r] = e >> 16;
      nf[r] = (int32_t)f - (int32_t)kM;
      bound[r] = f ? ((kL / f) << (32u - kTop)) + kL % f + cf[r] : 0u;
      if (r == 0) cf0 = cf[0];
      // an absent symbol begins where no slot is (a shifted slot has zero low bits)
      begin[r] = i < live ? (cf[r] - cf0) << kTop : 0xFFFFFFFFu;
      slots += f;
    }
    // a lane without symbols matches no slot: its shifted slot is odd, its bound zero
    first = slots ? 0u - (cf0 << kTop) : 1u;
    last = slots ? (slots << kTop) - 1u : 0u;
  }
};

template <int R, bool SE>
__device__ __forceinline__ void serial_chain(const GLB uint8_t* words, uint32_t n_words, uint32_t tail, uint32_t x0,
                                             uint32_t n, const LDS u32x2* syms, uint32_t live, LDS uint8_t* ring,
                                             GLB uint8_t* __restrict__ out, uint32_t stride, LDS uint32_t* hist,
                                             GLB uint32_t* ghist, uint32_t tps, int32_t* status) {
  constexpr uint32_t kLog = SE ? 12u : 10u, kTop = 32u - kLog;
  // the descriptor's fields are the same in every lane: say so, so that the
  // chain's state and word position stay scalar
  n_words = uni32(n_words);
  tail = uni32(tail);
  n = uni32(n);
  const uint32_t lane = __lane_id();
  const uint32_t n_eff = n_words + ((tail >> 16) & 1u);
  uint32_t x = uni32(x0);
  if (x < kL) {
    if (lane == 0) flag(status, BS_DEV_ERR_STREAM);
    return;
  }
  if (SE) tile_count_begin(hist, lane);
  LaneSyms<R, SE> S;
  S.load(syms, live, lane);
  WordWindow W(words, n_words, tail, ring);
  uint32_t at = kWave, win = 0;          // the next word is lane `at`'s; kWave: no window yet
  auto window = [&]() {
    W.move(at == kWave ? 0u : at, lane);
    at = 0;
    win = W.win;
  };
  uint32_t acc = 0;            // lane j: the symbol index (lane * R + r) of step j of the batch
  // One step: x becomes the next state, and lane j of acc takes the symbol's
  // index. On the GPU the step is one asm block per R, in this order because
  // issue is in order: a scalar instruction waits some 21 cycles for every
  // vector instruction before it that writes a scalar register (compares,
  // readlanes), whichever register it reads itself, so the compares come first,
  // the arithmetic fills the wait, and the scalar instructions follow together.
  // Wait states the hardware does not keep itself: two instructions between a
  // vector write of a scalar register and a vector read of it (x: writelane and
  // the next step's readlane of w; w, need, second: the arithmetic), one between
  // a vector write and a readlane of it (y: s_addc). settle() keeps those of the first
  // step of a run, whose operands the compiler wrote: without it nothing but the
  // compiler's choice of scalar instructions for them did (0.3 % of a chain's time).
#ifdef BS_SIMT_CPU
  // every lane finds the slot's symbol in the list by itself (an emulated
  // ballot or readlane costs 64 fiber switches)
  auto step = [&](uint32_t j) {
    const uint32_t slot = x & ((1u << kLog) - 1u);
    uint32_t lo = 0, hi = live;
    while (hi - lo > 1) {
      const uint32_t mid = (lo + hi) >> 1;
      if ((syms[mid].x >> 16) <= slot) lo = mid; else hi = mid;
    }
    const uint32_t c = (syms[lo].x & 0xFFFFu) * (x >> kLog) + slot - (syms[lo].x >> 16);
    if (c < kL) x = (c << 16) | (uint32_t)__builtin_amdgcn_readlane((int)win, (int)at++);
    else x = c;
    acc = lane == j ? lo : acc;
  };
#define BS_STEP(j) step(j)
#else
#define BS_STEP1(j)                                                                                              \
  {                                                                                                                   \
    uint32_t w, l, t, h, c, y;                                                                                        \
    uint64_t need;                                                                                                    \
    asm volatile("v_readlane_b32 %[w], %[win], %[at]\n\t"                                                             \
                 "v_lshl_add_u32 %[t], %[x], %[top], %[first]\n\t"                                                    \
                 "v_cmp_gt_u32 %[need], %[xb], %[x]\n\t"                                                              \
                 "v_cmp_le_u32 vcc, %[t], %[last]\n\t"                                                                \
                 "v_lshrrev_b32 %[h], %[log], %[x]\n\t"                                                               \
                 "v_sub_u32 %[c], %[x], %[cf]\n\t"                                                                    \
                 "v_mad_i32_i24 %[c], %[nf], %[h], %[c]\n\t"                                                          \
                 "v_lshl_or_b32 %[y], %[c], 16, %[w]\n\t"                                                             \
                 "v_cndmask_b32 %[y], %[c], %[y], %[need]\n\t"                                                        \
                 "s_ff1_i32_b64 %[l], vcc\n\t"                                                                        \
                 "s_bitcmp1_b64 %[need], %[l]\n\t"                                                                    \
                 "s_addc_u32 %[at], %[at], 0\n\t"                                                                     \
                 "v_readlane_b32 %[x], %[y], %[l]\n\t"                                                                \
                 "v_writelane_b32 %[acc], %[l], %[step]"                                                              \
                 : [x] "+s"(x), [at] "+s"(at), [acc] "+v"(acc), [w] "=&s"(w), [l] "=&s"(l), [t] "=&v"(t), [h] "=&v"(h), \
                   [c] "=&v"(c), [y] "=&v"(y), [need] "=&s"(need)                                                     \
                 : [cf] "v"(S.cf[0]), [nf] "v"(S.nf[0]), [xb] "v"(S.bound[0]), [first] "v"(S.first),                  \
                   [last] "v"(S.last), [win] "v"(win), [log] "i"(kLog), [top] "i"(kTop), [step] "i"(j)                \
                 : "vcc", "scc");                                                                                     \
  }
#define BS_STEP2(j)                                                                                              \
  {                                                                                                                   \
    uint32_t w, l, o, t, h, c, d, y;                                                                                  \
    uint64_t need, second;                                                                                            \
    asm volatile("v_readlane_b32 %[w], %[win], %[at]\n\t"                                                             \
                 "v_lshl_add_u32 %[t], %[x], %[top], %[first]\n\t"                                                    \
                 "v_lshrrev_b32 %[h], %[log], %[x]\n\t"                                                               \
                 "v_cmp_ge_u32 %[second], %[t], %[begin]\n\t"                                                         \
                 "v_cmp_le_u32 vcc, %[t], %[last]\n\t"                                                                \
                 "v_sub_u32 %[c], %[x], %[cf]\n\t"                                                                    \
                 "v_cndmask_b32 %[y], %[xb], %[xb1], %[second]\n\t"                                                   \
                 "v_sub_u32 %[d], %[x], %[cf1]\n\t"                                                                   \
                 "v_cmp_gt_u32 %[need], %[y], %[x]\n\t"                                                               \
                 "v_mad_i32_i24 %[c], %[nf], %[h], %[c]\n\t"                                                          \
                 "v_mad_i32_i24 %[d], %[nf1], %[h], %[d]\n\t"                                                         \
                 "v_cndmask_b32 %[c], %[c], %[d], %[second]\n\t"                                                      \
                 "v_lshl_or_b32 %[y], %[c], 16, %[w]\n\t"                                                             \
                 "v_cndmask_b32 %[y], %[c], %[y], %[need]\n\t"                                                        \
                 "s_ff1_i32_b64 %[l], vcc\n\t"                                                                        \
                 "s_bitcmp1_b64 %[second], %[l]\n\t"                                                                  \
                 "s_addc_u32 %[o], %[l], %[l]\n\t"                                                                    \
                 "s_bitcmp1_b64 %[need], %[l]\n\t"                                                                    \
                 "s_addc_u32 %[at], %[at], 0\n\t"                                                                     \
                 "v_readlane_b32 %[x], %[y], %[l]\n\t"                                                                \
                 "v_writelane_b32 %[acc], %[o], %[step]"                                                              \
                 : [x] "+s"(x), [at] "+s"(at), [acc] "+v"(acc), [w] "=&s"(w), [l] "=&s"(l), [o] "=&s"(o),             \
                   [t] "=&v"(t), [h] "=&v"(h), [c] "=&v"(c), [d] "=&v"(d), [y] "=&v"(y), [need] "=&s"(need),          \
                   [second] "=&s"(second)                                                                             \
                 : [cf] "v"(S.cf[0]), [cf1] "v"(S.cf[R - 1]), [nf] "v"(S.nf[0]), [nf1] "v"(S.nf[R - 1]),              \
                   [xb] "v"(S.bound[0]), [xb1] "v"(S.bound[R - 1]), [first] "v"(S.first), [last] "v"(S.last),         \
                   [begin] "v"(S.begin[R - 1]), [win] "v"(win), [log] "i"(kLog), [top] "i"(kTop), [step] "i"(j)       \
                 : "vcc", "scc");                                                                                     \
  }
#define BS_STEP(j)                  \
  if constexpr (R == 1) BS_STEP1(j) \
  else BS_STEP2(j)
#endif
  auto settle = [&]() {
    x = uni32(x);
    at = uni32(at);
    BS_LANE_SETTLE(x, at, win);
  };
  // this lane's step of a batch at i0 out (cnt steps), its exponent into the tile's counts
  auto emit = [&](uint32_t i0, uint32_t cnt) {
    const uint32_t word = syms[min(acc, live - 1u)].y;
    if (cnt == (uint32_t)kWave || lane < cnt) {
      if (SE) ((GLB uint16_t*)out)[(uint64_t)(i0 + lane) * stride] = (uint16_t)word;
      else out[i0 + lane] = (uint8_t)word;
    }
    if (SE) tile_count(hist, ghist, word, lane, i0, cnt, n);
  };
  const uint32_t whole = n & ~(uint32_t)(kWave - 1);
  for (uint32_t i0 = 0; i0 < whole; i0 += kWave) {
#pragma unroll
    for (uint32_t h0 = 0; h0 < kWave; h0 += kHalf) {
      if (at >= kHalf) window();                         // uniform
      settle();
#pragma unroll
      for (uint32_t j = 0; j < kHalf; ++j) {
        BS_STEP(h0 + j);
      }
    }
    emit(i0, kWave);
  }
  if (whole < n) {                                       // the last, partial batch (a step's lane is a constant: 0)
    uint32_t kept = 0;
    for (uint32_t j = 0; j < n - whole; ++j) {
      if (at >= kHalf) window();
      settle();
      BS_STEP(0);
      BS_VGPR_SETTLE(acc);
      const uint32_t o = (uint32_t)__builtin_amdgcn_readlane((int)acc, 0);
      kept = lane == j ? o : kept;
    }
    acc = kept;
    emit(whole, n - whole);
  }
#undef BS_STEP
  if (SE) tile_count_end(ghist, lane, n, tps);
  if (at == kWave) at = 0;                               // an empty chain never opened its window
  if (x != kL || W.base + at != n_eff) {
    if (lane == 0) flag(status, BS_DEV_ERR_STREAM);
  }
}

// The SE chain of a tensor with more than 128 live symbols (a checkpoint's weights
// have 60 or so), of which a lane would hold four or more: each of those costs a
// step five instructions more in every lane, a table read costs one LDS latency.
// The table is the task's own, in LDS as 4-byte entries {f | (slot - cf) << 13}
// beside the slots' output words, shared by the workgroup's chains. The state and the word position stay in vector registers,
// the same in every lane, so that no step waits for a scalar register; the next
// word comes by ds_bpermute as soon as its position is known, under the next table
// read; a step's slot goes to its place in the wave's stage, which lane j reads
// after 64 steps. MI355X, 250 symbols: 54 ns a step on one chain (132 with eight symbols
// per lane), 70 with 128 chains (146); held by the lanes, 120 symbols take 45 and 59.
__device__ __forceinline__ void table_chain(const GLB uint8_t* words, uint32_t n_words, uint32_t tail, uint32_t x0,
                                            uint32_t n, const LDS uint32_t* tbl, const LDS uint16_t* slot_words,
                                            LDS uint16_t* stage, LDS uint8_t* ring, GLB uint16_t* __restrict__ out,
                                            uint32_t stride, LDS uint32_t* hist, GLB uint32_t* ghist, uint32_t tps,
                                            int32_t* status) {
  n_words = uni32(n_words);
  tail = uni32(tail);
  n = uni32(n);
  const uint32_t lane = __lane_id();
  const uint32_t n_eff = n_words + ((tail >> 16) & 1u);
  if (uni32(x0) < kL) {
    if (lane == 0) flag(status, BS_DEV_ERR_STREAM);
    return;
  }
  tile_count_begin(hist, lane);
  WordWindow W(words, n_words, tail, ring);
  uint32_t x = x0, at4 = 0, w = 0;       // at4: 4 * the next word's lane
  auto window = [&]() {
    W.move(uni32(at4) >> 2, lane);
    at4 = 0;
    w = (uint32_t)__builtin_amdgcn_ds_bpermute(0, (int)W.win);
  };
  window();
  BS_OPAQUE(x);
  auto step = [&](uint32_t j) {
    const uint32_t slot = x & 4095u, e = tbl[slot];
    const uint32_t c = __umul24(e & 0x1FFFu, x >> 12) + (e >> 13);
    *(volatile LDS uint16_t*)(stage + j) = (uint16_t)slot;
#ifdef BS_SIMT_CPU     // an emulated exchange costs 64 fiber switches: one where a word is taken
    x = c < kL ? (c << 16) | (uint32_t)__builtin_amdgcn_readlane((int)W.win, (int)(at4 >> 2)) : c;
    at4 += c < kL ? 4u : 0u;
#else
    x = c < kL ? (c << 16) | w : c;
    at4 += c < kL ? 4u : 0u;
    BS_OPAQUE(x);
    BS_OPAQUE(at4);
    w = (uint32_t)__builtin_amdgcn_ds_bpermute((int)at4, (int)W.win);
#endif
  };
  for (uint32_t i0 = 0; i0 < n; i0 += kWave) {
    const uint32_t cnt = min((uint32_t)kWave, n - i0);
    for (uint32_t h0 = 0; h0 < cnt; h0 += kHalf) {
      if (uni32(at4) >= 4u * kHalf) window();
      if (cnt - h0 >= kHalf) {
#pragma unroll
        for (uint32_t j = 0; j < kHalf; ++j) step(h0 + j);
      } else {
        for (uint32_t j = h0; j < cnt; ++j) step(j);
      }
    }
    wave_sync();
    const uint32_t word = slot_words[stage[lane] & 4095u];
    if (lane < cnt) out[(uint64_t)(i0 + lane) * stride] = (uint16_t)word;
    tile_count(hist, ghist, word, lane, i0, cnt, n);
    wave_sync();
  }
  tile_count_end(ghist, lane, n, tps);
  if (uni32(x) != kL || W.base + (uni32(at4) >> 2) != n_eff) {
    if (lane == 0) flag(status, BS_DEV_ERR_STREAM);
  }
}

// ---- mantissa chains, one per lane. The buckets of one exponent (one per stream of
// a bf16_parallel_v1 tensor) share a decode table, so a wavefront decodes up to
// 64 of them at once from one or two tables in LDS. A step costs more time than a
// wave-wide chain's (an LDS read on the state's path), but it advances 64
// chains, so the mantissas take a few wavefronts and leave the issue slots to the
// SE chains. The host lists the buckets table by table; a wavefront whose buckets
// have more than two tables takes two at a time.
//
// The SE chains set the launch's time where no exponent holds half of a stream, as
// in weights. A bucket as long as its stream does instead (73 ns a step): MI355X,
// 8 M elements in 128 streams, ms with a wavefront per bucket and LDS tables / now:
// normal weights 3.90 / 2.30, one exponent in all 5.80 / 4.78, 90 % one exponent
// 5.39 / 4.45, values around 1 (two exponents) 3.43 / 2.54; seven such tensors of 1 M
// elements with one exponent 0.85 / 0.82.
constexpr uint32_t kLaneRing = 32;                        // words in a lane's ring
constexpr uint32_t kLaneTables = 2;                       // decode tables of a wavefront
constexpr uint32_t kLaneB = kLaneTables * 4096 + kLaneRing * 2 * kWave;   // LDS bytes of a wavefront
constexpr uint32_t kLaneSteps = 16;                       // steps between looks at the ring

// Chains with at least this many buckets per table run one per lane: below it a
// wavefront would hold buckets of three tables or more, and takes them in turns.
constexpr uint32_t kLaneMin = 32;

__device__ __forceinline__ void lane_chains(const bs_mant_bucket* __restrict__ buckets, uint32_t n_buckets,
                                            uint32_t first, const uint32_t* __restrict__ tables, uint32_t n_tables,
                                            uint64_t n_out, uint8_t* __restrict__ mant, LDS uint8_t* area,
                                            int32_t* status) {
  const uint32_t lane = __lane_id();
  LDS uint32_t* tbl = (LDS uint32_t*)area;                // [table][slot]
  LDS uint32_t* ring = (LDS uint32_t*)(area + kLaneTables * 4096);   // word p of a lane: half p & 1 of dword (p/2)*64 + lane
  const bool have = first + lane < n_buckets;
  const bs_mant_bucket B = buckets[have ? first + lane : first];
  bool bad = have && (B.table >= n_tables || B.perm_begin + B.n > n_out);
  if (bad) flag(status, BS_DEV_ERR_HEADER);
  bool todo = have && !bad;
  if (todo && B.x0 < kL) {
    flag(status, BS_DEV_ERR_STREAM);
    todo = false;
  }
  const GLB uint8_t* w = (const GLB uint8_t*)B.words;
  const uint32_t n_eff = B.n_words + ((B.tail >> 16) & 1u), tail_word = B.tail & 0xFFFFu;
  // words p .. p+7 (p a multiple of 8) as four dwords; past the stream its tail word
  auto words8 = [&](uint32_t p) -> u32x4 {
    u32x4 v;
    if ((uint64_t)p + 8u <= B.n_words) {
      typedef u32x4 __attribute__((aligned(1))) unaligned4;
      v = *(const GLB unaligned4*)(w + 2ull * p);
    } else {
      for (uint32_t k = 0; k < 4; ++k) {
        const uint32_t a = p + 2 * k, b = a + 1;
        v[k] = (a < B.n_words ? word_at(w, a) : tail_word) | (b < B.n_words ? word_at(w, b) : tail_word) << 16;
      }
    }
    return v;
  };
  auto put8 = [&](uint32_t p, u32x4 v) {
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) ring[(((p >> 1) + k) & (kLaneRing / 2 - 1)) * kWave + lane] = v[k];
  };
  while (true) {
    // the next tables still wanted, and whose lanes run now
    uint64_t left = __ballot(todo);
    if (left == 0) break;
    bool run = false;
    uint32_t slot0 = 0;
#pragma unroll
    for (uint32_t k = 0; k < kLaneTables; ++k) {
      if (left == 0) break;                               // uniform
      const uint32_t t = (uint32_t)__builtin_amdgcn_readlane((int)B.table, (int)__builtin_ctzll(left));
      const bool mine = todo && !run && B.table == t;
      for (uint32_t i = lane; i < 1024; i += kWave) tbl[k * 1024 + i] = tables[(uint64_t)t * 1024u + i];
      if (mine) {
        run = true;
        slot0 = k * 1024;
      }
      left &= ~__ballot(mine);
    }
    wave_sync();
    todo = todo && !run;
    if (run) {
      uint32_t x = B.x0, pos = 0, ld = kLaneRing, r = 0;   // the ring holds words [pos, ld)
      for (uint32_t p = 0; p < kLaneRing; p += 8) put8(p, words8(p));
      GLB uint8_t* out = (GLB uint8_t*)(mant + B.perm_begin);
      // the word at pos, read when pos moves: its latency passes under the next table read
      auto next_word = [&]() {
        return (uint32_t)((const LDS uint16_t*)ring)[2u * (((pos >> 1) & (kLaneRing / 2 - 1)) * kWave + lane) + (pos & 1u)];
      };
      uint32_t wnext = next_word();
      auto step = [&]() -> uint32_t {
        const uint32_t e = tbl[slot0 + (x & 1023u)];
        const uint32_t c = __umul24(e & 0x7FFu, x >> 10) + ((e >> 11) & 0x3FFu);
        const bool need = c < kL;
        x = need ? (c << 16) | wnext : c;
        pos += need ? 1u : 0u;
        wnext = next_word();
        return e >> 21;
      };
      for (; r + kLaneSteps <= B.n; r += kLaneSteps) {
        while (ld - pos < kLaneSteps) {                   // rare: a block may take a word per step
          put8(ld, words8(ld));
          ld += 8;
          wnext = next_word();
        }
        const uint32_t room = kLaneRing - (ld - pos);
        u32x4 f0 = {0u, 0u, 0u, 0u}, f1 = {0u, 0u, 0u, 0u};
        if (room >= 8) f0 = words8(ld);                   // in flight under the block, landed after it
        if (room >= 16) f1 = words8(ld + 8);
        u32x4 o;
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
          uint32_t v = 0;
#pragma unroll
          for (uint32_t j = 0; j < 4; ++j) v |= (step() & 0x7Fu) << (8 * j);
          o[k] = v;
        }
        if (room >= 8) put8(ld, f0);
        if (room >= 16) put8(ld + 8, f1);
        ld += room >= 16 ? 16u : room >= 8 ? 8u : 0u;
        typedef u32x4 __attribute__((aligned(1))) unaligned4;
        *(GLB unaligned4*)(out + r) = o;
        wnext = next_word();                              // the word at pos may have landed only now
      }
      while (ld - pos < kLaneSteps) {
        put8(ld, words8(ld));
        ld += 8;
      }
      wnext = next_word();
      for (; r < B.n; ++r) out[r] = (uint8_t)(step() & 0x7Fu);
      if (x != kL || pos != n_eff) flag(status, BS_DEV_ERR_STREAM);
    }
    wave_sync();                                          // every lane is done with the tables
  }
}

// List the live symbols of a decode table in LDS, in slot order: the slots
// whose offset in their symbol is zero. `entry` gives slot i's {f | cf offset
// (slot - cf), output}; one wavefront runs it. Returns their number (at most cap).
template <uint32_t M, class Entry>
__device__ __forceinline__ uint32_t list_symbols(LDS u32x2* syms, uint32_t cap, uint32_t lane, Entry entry) {
  uint32_t live = 0;
#pragma unroll 8
  for (uint32_t i0 = 0; i0 < M; i0 += kWave) {
    const uint32_t i = i0 + lane;
    uint32_t f, off, out;
    entry(i, f, off, out);
    const bool starts = off == 0 && f != 0;
    const uint64_t m = __ballot(starts);
    const uint32_t r = live + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
    if (starts && r < cap) syms[r] = u32x2{f | (i << 16), out};
    live += (uint32_t)__popcll(m);
  }
  return min(live, cap);
}

// ---- tasks of a wave-serial launch. Every tensor of a batch is one task; its
// chain groups, tiles and streams occupy consecutive workgroups of the grids
// (se_group_begin, mant_group_begin, tile_begin, stream_begin), so one launch
// of each kernel covers the whole batch and the chains of all its tensors run
// side by side. The single-tensor entry point passes its one task by value
// (tasks == nullptr).

__host__ __device__ inline uint64_t serial_max_len(uint64_t n_out, uint32_t n_streams) {
  return (n_out + n_streams - 1) / n_streams;
}
__host__ __device__ inline uint32_t serial_tiles(uint64_t n_out, uint32_t n_streams) {
  return (uint32_t)((serial_max_len(n_out, n_streams) + kTile - 1) / kTile);
}
__host__ __device__ inline uint64_t serial_work(uint64_t n_out, uint32_t n_streams) {
  return ((n_out + 255) & ~255ull) + (uint64_t)n_streams * serial_tiles(n_out, n_streams) * 256 * 4;
}

// A task every kernel may follow: 1 <= n_out < 2^32, at least one stream, a
// tile count that fits 32 bits, and its scratch inside the work buffer. Every
// kernel checks it alike, so a bad task is reported once and skipped by all.
__device__ __forceinline__ bool task_ok(const bs_ref_task& T, uint64_t work_bytes) {
  if (T.n_out == 0 || T.n_out > 0xFFFFFFFFull || T.n_streams == 0 || (T.work_offset & 255u)) return false;
  if ((uint64_t)T.n_streams * serial_tiles(T.n_out, T.n_streams) > 0xFFFFFFFFull) return false;
  return T.work_offset <= work_bytes && serial_work(T.n_out, T.n_streams) <= work_bytes - T.work_offset;
}

enum { kSeGrid = 0, kMantGrid = 1, kTileGrid = 2, kStreamGrid = 3 };
template <int G>
__device__ __forceinline__ uint32_t grid_begin(const bs_ref_task& t) {
  return G == kSeGrid ? t.se_group_begin : G == kMantGrid ? t.mant_group_begin
                                         : G == kTileGrid ? t.tile_begin : t.stream_begin;
}
// The task whose range of grid G holds workgroup b (binary search over the
// ascending begins; wave-uniform).
template <int G>
__device__ __forceinline__ bs_ref_task pick_task(const bs_ref_task* __restrict__ tasks, uint32_t n_tasks,
                                                 const bs_ref_task& single, uint32_t b) {
  if (tasks == nullptr) return single;
  uint32_t lo = 0, hi = n_tasks;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (grid_begin<G>(tasks[mid]) <= b) lo = mid; else hi = mid;
  }
  return tasks[lo];
}

// Chain grid: workgroups of kSerWaves wavefronts, one chain each. The first
// xcd_slots(se_groups) workgroups serve the SE groups (task by
// se_group_begin; their order is below): wave w of group j decodes SE stream
// j*kSerWaves + w (element first + i*stride for symbol i) with the task's SE
// symbols, listed once per workgroup and shared.
// The rest are mantissa groups (task by mant_group_begin): wave w decodes
// bucket j*kSerWaves + w into mant[perm_begin ...], or, with kLaneMin buckets per
// table or more, buckets 64 * (j*kSerWaves + w) .. + 63 (the groups past the
// last such bucket exit at once).
// The host lists buckets longest first, so the four buckets of a group end at
// about the same time and the longest start first.
//
// The SE part of the grid has xcd_slots(se_groups) workgroups, a multiple of
// kXcds: workgroup p serves SE group (p % kXcds) * (slots / kXcds) + p / kXcds
// (none past the last group). Workgroups go to the XCDs round-robin, so each
// XCD decodes one contiguous run of groups.
constexpr uint32_t kSerWaves = 4;
constexpr uint32_t kXcds = 8;
// A grid part of `count` workgroups dealt to the XCDs in contiguous blocks:
// count rounded up to a multiple of kXcds.
__host__ __device__ constexpr uint64_t xcd_slots(uint32_t count) {
  return ((uint64_t)count + kXcds - 1) / kXcds * kXcds;
}
constexpr uint32_t kSeSyms = 512, kMantSyms = 128;
constexpr uint32_t kSymB = kSeSyms * 8;   // one SE symbol list, or kSerWaves mantissa lists
static_assert(kSerWaves * kMantSyms <= kSeSyms, "mantissa lists exceed the symbol area");
constexpr uint32_t kHistB = 256 * 4;   // per SE chain: the exponent counts of its current tile
constexpr uint32_t kTblOff = kSerWaves * kRingB + kSymB + kSerWaves * kHistB;
// 48 KB: rings | symbols | tile counts (16 KB) | table_chain's table, output words and stages
// (24.5 KB), or the lane-wise chains' tables and rings
constexpr uint32_t kSerLds = kSerWaves * kLaneB;
static_assert(kSerLds >= kTblOff + 4096 * 6 + kSerWaves * kWave * 2, "chain LDS");

__global__ __launch_bounds__(kSerWaves * kWave) void serial_kernel(const bs_ref_task* __restrict__ tasks,
                                                                   uint32_t n_tasks, bs_ref_task single,
                                                                   uint32_t se_groups, uint8_t* __restrict__ work,
                                                                   uint64_t work_bytes, int32_t* __restrict__ status) {
  BS_DYNAMIC_LDS(smem);
  const uint32_t tid = threadIdx.x, lane = tid % kWave;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  LDS uint8_t* ring = (LDS uint8_t*)smem + wave * kRingB;
  LDS u32x2* syms = (LDS u32x2*)(smem + kSerWaves * kRingB);
  LDS uint32_t* hist = (LDS uint32_t*)(smem + kSerWaves * kRingB + kSymB + wave * kHistB);
  const uint32_t slots = (uint32_t)xcd_slots(se_groups);  // the launch checked that it fits
  const bool se = blockIdx.x < slots;                     // uniform over the workgroup
  const uint32_t g = se ? (blockIdx.x % kXcds) * (slots / kXcds) + blockIdx.x / kXcds : blockIdx.x - slots;
  if (se && g >= se_groups) return;
  const bs_ref_task T = se ? pick_task<kSeGrid>(tasks, n_tasks, single, g)
                           : pick_task<kMantGrid>(tasks, n_tasks, single, g);
  const uint32_t begin = se ? T.se_group_begin : T.mant_group_begin;
  if (g < begin) return;
  const uint32_t local = g - begin, count = se ? T.n_streams : T.n_buckets;
  const bool lanes = !se && T.n_buckets / kLaneMin >= T.n_tables;   // mantissa chains one per lane: 64 buckets a wave
  if ((uint64_t)local * kSerWaves * (lanes ? kWave : 1u) >= count) return;
  if (!task_ok(T, work_bytes)) {
    if (local == 0 && tid == 0) flag(status, BS_DEV_ERR_HEADER);
    return;
  }
  const uint32_t c = local * kSerWaves + wave;            // this wave's stream or bucket (none when >= count)
  const uint64_t max_len = (uint64_t)serial_tiles(T.n_out, T.n_streams) * kTile;
  uint8_t* mant = work + T.work_offset;
  if (se) {
    // every wave lists the symbols alike (the same values to the same places)
    const GLB u32x2* t = (const GLB u32x2*)T.se_table;
    const uint32_t live = list_symbols<4096>(syms, kSeSyms, lane, [&](uint32_t i, uint32_t& f, uint32_t& off, uint32_t& o) {
      const u32x2 e = t[i];
      f = e.x & 0x1FFFu;
      off = e.x >> 13;
      o = (((e.y >> 8) & 1u) << 15) | ((e.y & 0xFFu) << 7);
    });
    const bool table = live > 128;                        // uniform over the workgroup
    LDS uint32_t* tbl = (LDS uint32_t*)(smem + kTblOff);
    LDS uint16_t* slot_words = (LDS uint16_t*)(smem + kTblOff + 4096 * 4);
    if (table) {
      for (uint32_t i = tid; i < 4096; i += kSerWaves * kWave) {
        const u32x2 e = t[i];
        tbl[i] = e.x;
        slot_words[i] = (uint16_t)((((e.y >> 8) & 1u) << 15) | ((e.y & 0xFFu) << 7));
      }
    }
    __syncthreads();
    if (c >= count) return;
    const bs_se_stream S = T.streams[c];
    if (!stream_ok(S, max_len, T.n_out) || live == 0) {
      if (lane == 0) flag(status, BS_DEV_ERR_HEADER);
      return;
    }
    __builtin_amdgcn_s_setprio(3);                        // the longest chains: issue before the mantissas'
    // the stream's tile counts: tps x 256 after the task's mantissa area
    const uint32_t tps = serial_tiles(T.n_out, T.n_streams);
    GLB uint32_t* ghist = (GLB uint32_t*)(work + T.work_offset + ((T.n_out + 255) & ~255ull)) + (uint64_t)c * tps * 256u;
    auto run = [&](auto r) {
      serial_chain<decltype(r)::value, true>((const GLB uint8_t*)S.words, S.n_words, S.tail, S.x0, S.n, syms, live, ring,
                                             (GLB uint8_t*)(T.out + S.first), S.stride, hist, ghist, tps, status);
    };
    if (table)
      table_chain((const GLB uint8_t*)S.words, S.n_words, S.tail, S.x0, S.n, tbl, slot_words,
                  (LDS uint16_t*)(smem + kTblOff + 4096 * 6) + wave * kWave, ring, (GLB uint16_t*)(T.out + S.first), S.stride,
                  hist, ghist, tps, status);
    else if (live <= 64) run(std::integral_constant<int, 1>{});
    else run(std::integral_constant<int, 2>{});
  } else if (lanes) {
    if ((uint64_t)c * kWave >= count) return;
    lane_chains(T.buckets, T.n_buckets, c * kWave, T.mant_tables, T.n_tables, T.n_out, mant,
                (LDS uint8_t*)smem + wave * kLaneB, status);
  } else {
    if (c >= count) return;
    const bs_mant_bucket B = T.buckets[c];
    if (B.table >= T.n_tables || B.perm_begin + B.n > T.n_out) {
      if (lane == 0) flag(status, BS_DEV_ERR_HEADER);
      return;
    }
    const GLB uint32_t* t = (const GLB uint32_t*)T.mant_tables + (uint64_t)B.table * 1024u;
    syms += wave * kMantSyms;
    const uint32_t live = list_symbols<1024>(syms, kMantSyms, lane, [&](uint32_t i, uint32_t& f, uint32_t& off, uint32_t& o) {
      const uint32_t e = t[i];
      f = e & 0x7FFu;
      off = (e >> 11) & 0x3FFu;
      o = (e >> 21) & 0x7Fu;
    });
    wave_sync();
    if (live == 0) {
      if (lane == 0) flag(status, BS_DEV_ERR_HEADER);
      return;
    }
    serial_chain<2, false>((const GLB uint8_t*)B.words, B.n_words, B.tail, B.x0, B.n, syms, live, ring,
                           (GLB uint8_t*)(mant + B.perm_begin), 1u, nullptr, nullptr, 0u, status);
  }
}

// Stream grid, one workgroup per stream k of a task, thread e: turn stream
// k's tile counts of exponent e into each tile's first position in the
// bucket (bstart[k][e] + counts of the earlier tiles), and check that the
// decoded exponents fill every bucket exactly.
__global__ __launch_bounds__(256) void scan_kernel(const bs_ref_task* __restrict__ tasks, uint32_t n_tasks,
                                                   bs_ref_task single, uint8_t* __restrict__ work,
                                                   uint64_t work_bytes, int32_t* __restrict__ status) {
  const uint32_t e = threadIdx.x;
  const bs_ref_task T = pick_task<kStreamGrid>(tasks, n_tasks, single, blockIdx.x);
  if (blockIdx.x < T.stream_begin || !task_ok(T, work_bytes)) return;
  const uint32_t k = blockIdx.x - T.stream_begin;
  if (k >= T.n_streams) return;
  const uint32_t tps = serial_tiles(T.n_out, T.n_streams);
  const uint32_t* bs = T.bstart + (uint64_t)k * 257;
  uint32_t* hk = (uint32_t*)(work + T.work_offset + ((T.n_out + 255) & ~255ull)) + (uint64_t)k * tps * 256;
  uint32_t run = bs[e];
  for (uint32_t t = 0; t < tps; ++t) {
    const uint32_t c = hk[(uint64_t)t * 256 + e];
    hk[(uint64_t)t * 256 + e] = run;
    run += c;
  }
  if (run != bs[e + 1]) flag(status, BS_DEV_ERR_COUNT);
}

// Tile grid, one wavefront per (stream k, tile t) of a task: the position of
// each element in its bucket, from the tile's first positions plus its rank
// among the equal exponents before it (64 elements at a time: lanes with the
// same exponent found with eight ballots); then OR the element's mantissa
// into it.
//
// A 128-byte line of output holds one symbol of 64 streams, so the waves of
// one tile column (tile t of every stream of a task) share their lines. The
// grid (a multiple of kXcds workgroups) is dealt like the SE part of the
// chain grid: workgroup p takes tile slot (p % kXcds) * (grid / kXcds) + p /
// kXcds of the tile grid, in which a task's tiles run streams fastest, so
// each XCD works through whole columns one after another and a line's 64
// writers meet in one L2. Tile order (stream, tile) spread every column
// over all XCDs: the batched 8B layer placed in 4.5 ms against 2.4 ms in
// column order (loading up to eight batches of 64 words at once, instead of
// one, made no difference in column order).
__global__ __launch_bounds__(kWave) void place_kernel(const bs_ref_task* __restrict__ tasks, uint32_t n_tasks,
                                                      bs_ref_task single, uint32_t n_tiles, uint8_t* __restrict__ work,
                                                      uint64_t work_bytes, int32_t* __restrict__ status) {
  __shared__ uint32_t cnt[256];
  const uint32_t lane = threadIdx.x;
  const uint32_t v = (blockIdx.x % kXcds) * (gridDim.x / kXcds) + blockIdx.x / kXcds;
  if (v >= n_tiles) return;
  const bs_ref_task T = pick_task<kTileGrid>(tasks, n_tasks, single, v);
  if (v < T.tile_begin || !task_ok(T, work_bytes)) return;
  const uint32_t tps = serial_tiles(T.n_out, T.n_streams), local = v - T.tile_begin;
  if (local >= T.n_streams * tps) return;
  const uint32_t t = local / T.n_streams, k = local % T.n_streams;
  const uint64_t n = T.n_out;
  const uint8_t* mant = work + T.work_offset;
  const uint32_t* first = (const uint32_t*)(mant + ((n + 255) & ~255ull));
  uint16_t* out = T.out;
  const bs_se_stream S = T.streams[k];
  if (!stream_ok(S, (uint64_t)tps * kTile, n)) return;     // reported by serial_kernel
  const uint64_t kt = (uint64_t)k * tps + t;               // the scan's (stream, tile) order
  for (uint32_t e = lane; e < 256; e += kWave) cnt[e] = first[kt * 256 + e];
  wave_sync();
  const uint32_t lo = t * kTile, hi = (uint32_t)min((uint64_t)S.n, (uint64_t)lo + kTile);
  const uint64_t lt = (1ull << lane) - 1ull;
  bool bad = false;
  for (uint32_t k0 = lo; k0 < hi; k0 += kWave) {
    const uint32_t i = k0 + lane;
    const bool valid = i < hi;
    const uint64_t el = S.first + (uint64_t)i * S.stride;
    const uint32_t word = valid ? out[el] : 0u;
    const uint32_t e = (word >> 7) & 0xFFu;
    uint64_t m = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const bool bit = (e >> b) & 1u;
      const uint64_t bb = __ballot(bit);
      m &= bit ? bb : ~bb;
    }
    const uint32_t rank = (uint32_t)__popcll(m & lt), total = (uint32_t)__popcll(m);
    const uint32_t base = cnt[e];
    wave_sync();
    if (valid && rank == 0) cnt[e] = base + total;
    if (valid) {
      const uint32_t p = base + rank;
      if (p < n) out[el] = (uint16_t)(word | mant[p]);
      else bad = true;
    }
    wave_sync();
  }
  if (__ballot(bad) != 0 && lane == 0) flag(status, BS_DEV_ERR_COUNT);
}

int launch_serial(const bs_ref_task* tasks, uint32_t n_tasks, const bs_ref_task& single, uint32_t se_groups,
                  uint32_t mant_groups, uint32_t tiles, uint32_t streams, uint8_t* work, uint64_t work_bytes,
                  int32_t* status, hipStream_t s) {
  if (xcd_slots(se_groups) + mant_groups > 0xFFFFFFFFull || xcd_slots(tiles) > 0xFFFFFFFFull) return BS_ERR_ARG;
  hipLaunchKernelGGL(serial_kernel, dim3((uint32_t)xcd_slots(se_groups) + mant_groups), dim3(kSerWaves * kWave),
                     kSerLds, s, tasks, n_tasks, single, se_groups, work, work_bytes, status);
  if (hipGetLastError() != hipSuccess) return BS_ERR_HIP;
  hipLaunchKernelGGL(scan_kernel, dim3(streams), dim3(256), 0, s, tasks, n_tasks, single, work, work_bytes, status);
  if (hipGetLastError() != hipSuccess) return BS_ERR_HIP;
  hipLaunchKernelGGL(place_kernel, dim3((uint32_t)xcd_slots(tiles)), dim3(kWave), 0, s, tasks, n_tasks, single, tiles,
                     work, work_bytes, status);
  return hipGetLastError() == hipSuccess ? BS_OK : BS_ERR_HIP;
}

}  // namespace

extern "C" {

int bs_refcodec_decode(const bs_se_stream* d_streams, uint32_t n_streams, const uint32_t* d_se_table,
                       const uint32_t* d_bstart, const bs_mant_bucket* d_buckets, uint32_t n_buckets,
                       const uint32_t* d_mant_tables, uint32_t n_tables, uint16_t* d_out, uint64_t n_out,
                       uint32_t* d_perm, int32_t* d_status, void* stream) {
  if (!d_status || (n_streams && (!d_streams || !d_se_table || !d_bstart)) ||
      (n_buckets && (!d_buckets || !d_mant_tables)) || (n_out && (!d_out || !d_perm)))
    return BS_ERR_ARG;
  if (n_out == 0 || n_streams == 0) return BS_OK;
  hipStream_t s = (hipStream_t)stream;
  constexpr uint32_t kSeLds = 4096 * 8 + 256 * kSeLanes * 4;
  static std::atomic<uint64_t> lds_set{0};
  bs_internal::ensure_lds_limit((const void*)se_kernel, kSeLds, lds_set);
  hipLaunchKernelGGL(se_kernel, dim3((n_streams + kSeLanes - 1) / kSeLanes), dim3(kSeLanes), kSeLds, s, d_streams,
                     n_streams, d_se_table, d_bstart, n_out, d_out, d_perm, d_status);
  if (hipGetLastError() != hipSuccess) return BS_ERR_HIP;
  if (n_buckets) {
    hipLaunchKernelGGL(mant_kernel, dim3((n_buckets + kMantThreads - 1) / kMantThreads), dim3(kMantThreads), 0, s,
                       d_buckets, n_buckets, d_mant_tables, n_tables, d_perm, n_out, n_out, d_out, d_status);
    if (hipGetLastError() != hipSuccess) return BS_ERR_HIP;
  }
  return BS_OK;
}

uint64_t bs_refcodec_serial_work_bytes(uint64_t n_out, uint32_t n_streams) {
  if (n_streams == 0) return 0;
  return serial_work(n_out, n_streams);
}

uint32_t bs_refcodec_serial_tiles(uint64_t n_out, uint32_t n_streams) {
  if (n_streams == 0 || n_out == 0) return 0;
  return serial_tiles(n_out, n_streams);
}

int bs_refcodec_decode_serial(const bs_se_stream* d_streams, uint32_t n_streams, const uint32_t* d_se_table,
                              const uint32_t* d_bstart, const bs_mant_bucket* d_buckets, uint32_t n_buckets,
                              const uint32_t* d_mant_tables, uint32_t n_tables, uint16_t* d_out, uint64_t n_out,
                              void* d_work, uint64_t work_bytes, int32_t* d_status, void* stream) {
  if (!d_status || (n_out && (!d_streams || !d_se_table || !d_bstart || !d_out || !d_work || !n_streams)) ||
      (n_buckets && (!d_buckets || !d_mant_tables)) || n_out > 0xFFFFFFFFull)
    return BS_ERR_ARG;
  if (n_out == 0) return BS_OK;
  if (work_bytes < bs_refcodec_serial_work_bytes(n_out, n_streams) || ((uintptr_t)d_work & 255u)) return BS_ERR_ARG;
  const uint64_t tiles = (uint64_t)n_streams * serial_tiles(n_out, n_streams);
  if ((uint64_t)n_streams + n_buckets > 0xFFFFFFFFull || tiles > 0xFFFFFFFFull) return BS_ERR_ARG;
  bs_ref_task t{};
  t.streams = d_streams;
  t.se_table = d_se_table;
  t.bstart = d_bstart;
  t.buckets = d_buckets;
  t.mant_tables = d_mant_tables;
  t.out = d_out;
  t.n_out = n_out;
  t.work_offset = 0;
  t.n_streams = n_streams;
  t.n_buckets = n_buckets;
  t.n_tables = n_tables;
  return launch_serial(nullptr, 0u, t, (n_streams + kSerWaves - 1) / kSerWaves,
                       (uint32_t)(((uint64_t)n_buckets + kSerWaves - 1) / kSerWaves), (uint32_t)tiles, n_streams,
                       (uint8_t*)d_work, work_bytes, d_status, (hipStream_t)stream);
}

uint32_t bs_refcodec_serial_chains_per_group(void) { return kSerWaves; }

int bs_refcodec_decode_serial_batch(const bs_ref_task* d_tasks, uint32_t n_tasks, uint32_t total_se_groups,
                                    uint32_t total_mant_groups, uint32_t total_tiles, uint32_t total_streams,
                                    void* d_work, uint64_t work_bytes, int32_t* d_status, void* stream) {
  if (!d_status || (n_tasks && (!d_tasks || !d_work)) || ((uintptr_t)d_work & 255u)) return BS_ERR_ARG;
  if (n_tasks == 0) return BS_OK;
  if (total_se_groups == 0 || total_tiles == 0 || total_streams == 0) return BS_ERR_ARG;
  bs_ref_task dummy{};
  return launch_serial(d_tasks, n_tasks, dummy, total_se_groups, total_mant_groups, total_tiles, total_streams,
                       (uint8_t*)d_work, work_bytes, d_status, (hipStream_t)stream);
}

}  // extern "C"
