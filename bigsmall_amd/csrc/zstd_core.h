// Zstandard frame decoding (RFC 8878), written once for a team of lanes that
// run it together: a 256-lane workgroup on the GPU (zstd_decode.hip). The
// frame, block and section headers are parsed by every lane alike (the same
// bytes, the same branches); table descriptions are read by one lane, tables
// are built and Huffman streams decoded by all lanes, with the tables in shared
// memory; long copies are spread over all lanes, short sequences run by the
// leading ones.
//
// A Team provides lane() (0 .. size-1), size and sync() (a barrier that also
// makes every lane's earlier global and shared-memory writes visible to the
// team), and its leading lanes, 0 .. lead_size-1 (one wavefront on the GPU):
// leads() (true in them, the same in a whole wavefront) and lead_sync(), the
// same among them alone.
//
// Every read of the input is bounds-checked; malformed input ends the task
// with an error code, never with an out-of-bounds access. Not supported:
// dictionaries (a frame naming a dictionary is an error) and checking the
// optional content checksum (its 4 bytes are skipped).
#pragma once

#include <stdint.h>

namespace bs_zstd {

constexpr uint32_t kBlockMax = 128u << 10;     // RFC 8878 3.1.1.2.4: Block_Maximum_Size
constexpr uint32_t kHufLogMax = 12;
constexpr uint32_t kLLLog = 9, kMLLog = 9, kOFLog = 8, kWeightLog = 6;
constexpr uint32_t kLLMax = 35, kMLMax = 52, kOFMax = 31;
constexpr uint32_t kStageBytes = 24u << 10;    // compressed blocks up to this size are read from shared memory
constexpr uint32_t kHufGroups = 64;            // pieces of a literal section's streams decoded side by side
constexpr uint32_t kHufQuarterMax = 128;       // stream bits of a quarter of a piece at most
constexpr uint32_t kFewSequences = 32;         // a block of fewer is run by all lanes alike, of more by the leading ones
constexpr uint32_t kLongSequence = 128;        // literals or match bytes from which all lanes copy a sequence in either case
static_assert((kLongSequence & (kLongSequence - 1)) == 0, "run_sequences tests literals and match bytes together");

enum : int32_t {
  kOk = 0,
  kErrTruncated = 1,     // a header or section runs past the input
  kErrFormat = 2,        // bad magic, reserved bits or block type, dictionary frame
  kErrTable = 3,         // invalid FSE or Huffman table description
  kErrStream = 4,        // a bitstream does not end where it must
  kErrOutput = 5,        // output past the destination capacity, or a size check failed
  kErrOffset = 6,        // a match reaches before the start of its frame
};

struct FseCell {
  uint16_t base;     // next state = base + (nb bits read)
  uint8_t sym;
  uint8_t nb;
};

// Repeat offsets (RFC 8878 3.1.2.5), kept from block to block in a frame.
struct Rep {
  uint32_t r0, r1, r2;
};

// Scratch of the table builds (dead before a Huffman decode starts).
struct BuildScratch {
  int16_t norm[64];
  uint16_t start[64];                 // FSE construction: cells of the symbols before this one
  alignas(16) uint8_t weight[256];
  alignas(16) uint8_t spread[1u << kLLLog];   // FSE construction: symbol of each cell
};
// Per piece of a Huffman stream and bit of its start that a code may begin at:
// where the walk from there leaves the piece (bits past its end) | its symbols << 4.
struct HufScratch {
  uint16_t hop[kHufGroups * kHufLogMax];
};

// Per-task state: the decode tables kept between the blocks of a frame. Four of
// these fit a CU's 160 KB of LDS.
struct ZState {
  alignas(16) uint16_t huf[1u << kHufLogMax];   // symbol | bits << 8, indexed by the next huf_log bits
  FseCell ll[1u << kLLLog], ml[1u << kMLLog], of[1u << kOFLog];
  FseCell wt[1u << kWeightLog];       // Huffman-weight table
  uint32_t ll_base[kLLMax + 1], ml_base[kMLMax + 1];
  uint8_t ll_bits[kLLMax + 1], ml_bits[kMLMax + 1];
  union {
    BuildScratch b;
    HufScratch h;
  };
  uint32_t entry[kHufGroups];         // per piece: its first code's bit in it | symbols before it << 4
  uint16_t mark[kHufGroups][3];       // the same within a piece at its second, third and last quarter
  struct {
    uint32_t bits, off, count;        // a Huffman stream: its bits, first byte, symbols
    uint32_t at;                      // the same as `entry` for the pieces still to come
  } hs[4];
  uint32_t huf_log;                   // 0: no Huffman table yet in this frame
  uint32_t ll_log, ml_log, of_log;
  uint32_t have_ll, have_ml, have_of; // a table exists for the Repeat mode
  uint32_t val[3];                    // broadcast: results of single-lane work
  int32_t err;                        // broadcast: error of single-lane work
  struct {                            // from the leading lanes: a long sequence, or (more == 0) the end of them
    uint64_t op;
    uint32_t lp, ll, ml, off, more;
    int32_t err;
    Rep rep;
  } seq;
  uint8_t stage[kStageBytes];         // the current compressed block, when it fits
};
static_assert(sizeof(ZState) <= 160u * 1024u / 4, "four tasks per CU");

__host__ __device__ constexpr uint32_t highbit(uint32_t v) { return 31u - (uint32_t)__builtin_clz(v); }
__host__ __device__ __forceinline__ uint64_t mask64(uint32_t n) { return n >= 64 ? ~0ull : ((1ull << n) - 1ull); }

// Little-endian value of p[i .. i+8), bytes at or past `len` read as zero.
__host__ __device__ inline uint64_t load_le(const uint8_t* p, uint64_t len, uint64_t i) {
  uint64_t v = 0;
  for (uint32_t k = 0; k < 8; ++k)
    if (i + k < len) v |= (uint64_t)p[i + k] << (8 * k);
  return v;
}

// Forward bit reader (FSE table descriptions): bits taken from the least
// significant end of each byte, bytes in increasing order.
struct FwdBits {
  const uint8_t* p;
  uint64_t len;
  uint64_t pos;      // bits consumed
  __host__ __device__ uint32_t peek(uint32_t n) const {
    return (uint32_t)((load_le(p, len, pos >> 3) >> (pos & 7)) & mask64(n));
  }
  __host__ __device__ uint32_t read(uint32_t n) {
    const uint32_t v = peek(n);
    pos += n;
    return v;
  }
};

// Backward bit reader (Huffman and FSE-coded streams, RFC 8878 4.1, 4.2.2):
// the stream is read from its last byte towards its first; the highest set
// bit of the last byte marks the end and is skipped. Reading n bits yields the
// next n unread bits from the top as one number; past the start of the stream
// the missing bits read as zeros and `bits` goes negative (overflow). The next
// unread bits sit left-aligned in a 64-bit register, refilled a byte at a time.
struct BackBits {
  const uint8_t* p;
  uint64_t acc;      // the top `have` unread bits, most significant first; zeros below
  int32_t have;      // negative once reads have gone past the start of the stream
  uint32_t lo;       // bytes [0, lo) are not yet in acc
  __host__ __device__ bool init(const uint8_t* q, uint64_t n) {
    p = q;
    acc = 0;
    have = 0;
    lo = 0;
    if (n == 0 || n > 0xFFFFFFFFull || q[n - 1] == 0) return false;
    const uint32_t hb = highbit(q[n - 1]);
    acc = hb ? (uint64_t)(q[n - 1] & ((1u << hb) - 1u)) << (64 - hb) : 0ull;
    have = (int32_t)hb;
    lo = (uint32_t)(n - 1);
    refill();
    return true;
  }
  // Unread bits; negative after an overflow.
  __host__ __device__ int64_t bits() const { return (int64_t)lo * 8 + have; }
  __host__ __device__ void refill() {         // as many whole bytes as fit, loaded together
    if (have > 56 || lo == 0) return;
    if (lo >= 8 && have >= 0) {
      // one load; a byte of which only the top bits fit is read again by the next refill, the same bits
      uint64_t v;
      __builtin_memcpy(&v, p + lo - 8, 8);
      acc |= v >> have;
      const uint32_t k = (uint32_t)(64 - have) >> 3;
      have += (int32_t)(8 * k);
      lo -= k;
      return;
    }
    const uint32_t want = (uint32_t)(64 - have) >> 3;
    const uint32_t k = lo < want ? lo : want;
    uint64_t v = 0;
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i)
      if (i < k) v |= (uint64_t)p[lo - 1 - i] << (56 - 8 * i);
    acc |= v >> have;
    have += (int32_t)(8 * k);
    lo -= k;
  }
  __host__ __device__ uint32_t peek(uint32_t n) {             // n <= 32
    if (have < (int32_t)n) refill();
    return n ? (uint32_t)(acc >> (64 - n)) : 0u;
  }
  __host__ __device__ void skip(uint32_t n) {                 // after a peek of >= n bits
    acc = n < 64 ? acc << n : 0ull;
    have -= (int32_t)n;
  }
  __host__ __device__ uint32_t read(uint32_t n) {
    const uint32_t v = peek(n);
    skip(n);
    return v;
  }
};

// Default distributions (RFC 8878 3.1.1.3.2.2), 3 bits per symbol holding
// count + 1, 21 symbols per word.
__host__ __device__ constexpr int16_t default_norm(uint32_t kind, uint32_t s) {
  uint64_t w = 0;
  const uint32_t k = s / 21, sh = 3 * (s % 21);
  if (kind == 0)
    w = k == 0 ? 0x36DB4936DB6DB6E5ull : 0x000000009249C6DBull;                  // literal lengths, 36
  else if (kind == 1)
    w = k == 0 ? 0x24924924936DB72Aull : k == 1 ? 0x2492492492492492ull : 0x0000000000000492ull;  // match lengths, 53
  else
    w = k == 0 ? 0x24924924936D2492ull : 0x0000000000000092ull;                  // offsets, 29
  return (int16_t)((w >> sh) & 7u) - 1;
}

// Extra-bit counts of the literal- and match-length codes (RFC 8878
// 3.1.1.3.2.1.1); each baseline is the previous one plus 2^(previous bits).
__host__ __device__ constexpr uint32_t ll_code_bits(uint32_t c) {
  return c < 16 ? 0u : c < 20 ? 1u : c < 22 ? 2u : c < 24 ? 3u : c == 24 ? 4u : c - 19u;
}
__host__ __device__ constexpr uint32_t ml_code_bits(uint32_t c) {
  return c < 32 ? 0u : c < 36 ? 1u : c < 38 ? 2u : c < 40 ? 3u : c < 42 ? 4u : c == 42 ? 5u : c - 36u;
}

// Tables that the format fixes, made by the compiler: the length codes and the
// predefined sequence tables (RFC 8878 appendix A). Building them on one lane
// of every task took a fifth of a small frame's time.
struct FixedTables {
  uint32_t ll_base[kLLMax + 1], ml_base[kMLMax + 1];
  uint8_t ll_bits[kLLMax + 1], ml_bits[kMLMax + 1];
  FseCell ll[64], ml[64], of[32];
};
// Decode table of default_norm(kind) at accuracy log (RFC 8878 4.1.1, "FSE Table Construction").
constexpr void fixed_fse(FseCell* t, uint32_t kind, uint32_t nsym, uint32_t log) {
  const uint32_t size = 1u << log, mask = size - 1, step = (size >> 1) + (size >> 3) + 3;
  uint32_t next[64] = {}, high = size - 1, pos = 0;
  for (uint32_t s = 0; s < nsym; ++s) {
    const int16_t n = default_norm(kind, s);
    next[s] = n < 0 ? 1u : (uint32_t)n;
    if (n < 0) t[high--].sym = (uint8_t)s;
  }
  for (uint32_t s = 0; s < nsym; ++s)
    for (int32_t i = 0; i < default_norm(kind, s); ++i) {
      t[pos].sym = (uint8_t)s;
      do pos = (pos + step) & mask;
      while (pos > high);
    }
  for (uint32_t u = 0; u < size; ++u) {
    const uint32_t x = next[t[u].sym]++, nb = log - highbit(x);
    t[u].nb = (uint8_t)nb;
    t[u].base = (uint16_t)((x << nb) - size);
  }
}
constexpr FixedTables fixed_tables() {
  FixedTables f{};
  uint32_t b = 0;
  for (uint32_t c = 0; c <= kLLMax; ++c) {
    f.ll_bits[c] = (uint8_t)ll_code_bits(c);
    f.ll_base[c] = c < 16 ? c : b;
    b = (c < 16 ? c : b) + (1u << ll_code_bits(c));
  }
  b = 0;
  for (uint32_t c = 0; c <= kMLMax; ++c) {
    f.ml_bits[c] = (uint8_t)ml_code_bits(c);
    f.ml_base[c] = c < 32 ? c + 3 : b;
    b = (c < 32 ? c + 3 : b) + (1u << ml_code_bits(c));
  }
  fixed_fse(f.ll, 0, 36, 6);
  fixed_fse(f.ml, 1, 53, 6);
  fixed_fse(f.of, 2, 29, 5);
  return f;
}
constexpr FixedTables kFixed = fixed_tables();

template <class Team>
__host__ __device__ inline void load_length_codes(const Team& tm, ZState& z) {
  for (uint32_t c = tm.lane(); c <= kMLMax; c += Team::size) {
    z.ml_base[c] = kFixed.ml_base[c];
    z.ml_bits[c] = kFixed.ml_bits[c];
    if (c <= kLLMax) {
      z.ll_base[c] = kFixed.ll_base[c];
      z.ll_bits[c] = kFixed.ll_bits[c];
    }
  }
}

// FSE table description (RFC 8878 4.1.1) at p[0, len) into norm[]; returns
// the bytes it takes, 0 if it is invalid.
__host__ __device__ inline uint32_t read_ncount(const uint8_t* p, uint64_t len, int16_t* norm, uint32_t max_sym,
                                                uint32_t max_log, uint32_t& log, uint32_t& nsym) {
  if (len == 0) return 0;
  FwdBits br{p, len, 0};
  log = br.read(4) + 5;
  if (log > max_log) return 0;
  int32_t remaining = (1 << log) + 1, threshold = 1 << log;
  uint32_t nb = log + 1, sym = 0;
  bool prev0 = false;
  while (remaining > 1 && sym <= max_sym) {
    if (prev0) {                        // a zero count is followed by 2-bit repeat flags
      uint32_t n0 = sym;
      for (;;) {
        const uint32_t r = br.read(2);
        n0 += r;
        if (r != 3 || n0 > max_sym) break;
      }
      if (n0 > max_sym) return 0;
      while (sym < n0) norm[sym++] = 0;
    }
    const int32_t maxv = (2 * threshold - 1) - remaining;
    const uint32_t v = br.peek(nb);
    int32_t count;
    if ((int32_t)(v & (uint32_t)(threshold - 1)) < maxv) {
      count = (int32_t)(v & (uint32_t)(threshold - 1));
      br.pos += nb - 1;
    } else {
      count = (int32_t)(v & (uint32_t)(2 * threshold - 1));
      if (count >= threshold) count -= maxv;
      br.pos += nb;
    }
    --count;                            // -1: a "less than one" probability
    remaining -= count < 0 ? -count : count;
    norm[sym++] = (int16_t)count;
    prev0 = count == 0;
    while (remaining < threshold) {
      --nb;
      threshold >>= 1;
    }
  }
  if (remaining != 1 || br.pos > 8 * len) return 0;
  nsym = sym;
  return (uint32_t)((br.pos + 7) >> 3);
}

// Decode table for z.b.norm[0, nsym) at accuracy `log` (RFC 8878 4.1.1, "FSE
// Table Construction"). False if the counts do not fill the table. Every lane
// calls it after a sync; it ends with one. The format spreads the symbols with
// a fixed step over the cells below the "less than one" symbols', which are the
// last ones; here each cell finds its symbol by itself: cell (i * step) mod size
// is the walk's i-th, less the skipped cells before it.
template <class Team>
__host__ __device__ inline bool build_fse(const Team& tm, ZState& z, FseCell* t, uint32_t nsym, uint32_t log) {
  const uint32_t size = 1u << log, mask = size - 1, step = (size >> 1) + (size >> 3) + 3;
  if (nsym > 64) return false;
  BuildScratch& B = z.b;
  uint32_t total = 0, low = 0;
  for (uint32_t s = 0; s < nsym; ++s) {
    const int32_t v = B.norm[s];
    total += v < 0 ? 1u : (uint32_t)v;
    low += v < 0;
  }
  if (total != size) return false;
  const uint32_t cells = size - low;                   // cells of the walk; the rest hold the low symbols
  for (uint32_t s = tm.lane(); s < nsym; s += Team::size) {
    uint32_t before = 0, lows = 0;
    for (uint32_t r = 0; r < s; ++r) {
      const int32_t v = B.norm[r];
      before += v < 0 ? 0u : (uint32_t)v;
      lows += v < 0;
    }
    B.start[s] = (uint16_t)before;
    if (B.norm[s] < 0) B.spread[size - 1 - lows] = (uint8_t)s;
  }
  tm.sync();
  uint32_t inv = step;                                 // step's inverse modulo 2^32 (step is odd)
  for (int i = 0; i < 4; ++i) inv *= 2u - step * inv;
  for (uint32_t i = tm.lane(); i < size; i += Team::size) {
    const uint32_t p = (i * step) & mask;
    if (p >= cells) continue;
    uint32_t k = i;                                    // the cell's place among the symbols' occurrences
    for (uint32_t m = cells; m < size; ++m) k -= ((m * inv) & mask) < i;
    uint32_t lo = 0, hi = nsym;                        // the last symbol that starts at or before k
    while (hi - lo > 1) {
      const uint32_t mid = (lo + hi) >> 1;
      if (B.start[mid] <= k) lo = mid; else hi = mid;
    }
    B.spread[p] = (uint8_t)lo;
  }
  tm.sync();
  // a symbol's cells take its states in ascending order: a lane per symbol
  for (uint32_t s = tm.lane(); s < nsym; s += Team::size) {
    const int32_t v = B.norm[s];
    uint32_t x = v < 0 ? 1u : (uint32_t)v;
    if (x == 0) continue;
    for (uint32_t u = 0; u < size; u += 16) {          // sixteen cells read at a time
      uint32_t w[4];
      __builtin_memcpy(w, __builtin_assume_aligned(B.spread + u, 16), 16);
#pragma unroll
      for (uint32_t i = 0; i < 16; ++i) {
        if (((w[i >> 2] >> (8 * (i & 3))) & 0xFFu) != s) continue;
        const uint32_t nb = log - highbit(x);
        t[u + i] = FseCell{(uint16_t)((x << nb) - size), (uint8_t)s, (uint8_t)nb};
        ++x;
      }
    }
  }
  tm.sync();
  return true;
}

// Size in bytes of a Huffman tree description starting at q (RFC 8878 4.2.1).
__host__ __device__ inline uint32_t huf_desc_bytes(uint8_t h) { return h < 128 ? 1u + h : 1u + (h - 127u + 1u) / 2u; }

// Weights of an FSE-coded tree description, from the bits after its table
// (one lane): how many, or 0 if the stream is invalid.
__host__ __device__ inline uint32_t read_weights(ZState& z, const uint8_t* q, uint64_t n, uint32_t log) {
  BackBits br;
  if (!br.init(q, n)) return 0;
  uint32_t nw = 0, s1 = br.read(log), s2 = br.read(log);
  for (;;) {                            // two interleaved states until the stream overflows
    if (nw >= 255) return 0;
    z.b.weight[nw++] = z.wt[s1].sym;
    s1 = z.wt[s1].base + br.read(z.wt[s1].nb);
    if (br.bits() < 0) {
      z.b.weight[nw++] = z.wt[s2].sym;
      break;
    }
    if (nw >= 255) return 0;
    z.b.weight[nw++] = z.wt[s2].sym;
    s2 = z.wt[s2].base + br.read(z.wt[s2].nb);
    if (br.bits() < 0) {
      z.b.weight[nw++] = z.wt[s1].sym;
      break;
    }
  }
  return nw > 255 ? 0 : nw;
}

// Weights i .. i+15 (i a multiple of 16) as four words, zeros from nw on.
__host__ __device__ inline void load_weights(const uint8_t* weight, uint32_t nw, uint32_t i, uint32_t (&w)[4]) {
  __builtin_memcpy(w, __builtin_assume_aligned(weight + i, 16), 16);
#pragma unroll
  for (uint32_t k = 0; k < 4; ++k) {
    const uint32_t left = nw > i + 4 * k ? nw - (i + 4 * k) : 0u;
    if (left < 4) w[k] &= (1u << (8 * left)) - 1u;
  }
}

// Builds z.huf from the tree description at q, whose size is inside the
// section: the weights, the implied last weight, then codes assigned by weight
// and symbol. Every lane calls it; it ends with a sync, except on an error.
template <class Team>
__host__ __device__ inline int32_t build_huffman(const Team& tm, ZState& z, const uint8_t* q) {
  const uint8_t h = q[0];
  uint8_t* weight = z.b.weight;
  tm.sync();                            // the scratch's earlier use is over
  uint32_t nw;
  if (h >= 128) {
    nw = h - 127u;
    for (uint32_t i = tm.lane(); i < nw; i += Team::size) {
      const uint8_t b = q[1 + i / 2];
      weight[i] = (uint8_t)((i & 1) ? (b & 15u) : (b >> 4));
    }
    tm.sync();
  } else {
    if (tm.lane() == 0) z.val[0] = read_ncount(q + 1, h, z.b.norm, kHufLogMax, kWeightLog, z.val[1], z.val[2]);
    tm.sync();
    const uint32_t used = z.val[0], log = z.val[1], nsym = z.val[2];
    if (!used || used >= h || !build_fse(tm, z, z.wt, nsym, log)) return kErrTable;
    if (tm.lane() == 0) z.val[0] = read_weights(z, q + 1 + used, h - used, log);
    tm.sync();
    nw = z.val[0];
    if (!nw) return kErrTable;
  }
  // read sixteen at a time (zeros after the last): a read at a time waits for each
  uint32_t total = 0, top = 0;
  for (uint32_t i = 0; i < nw; i += 16) {
    uint32_t w4[4];
    load_weights(weight, nw, i, w4);
#pragma unroll
    for (uint32_t k = 0; k < 16; ++k) {
      const uint32_t w = (w4[k >> 2] >> (8 * (k & 3))) & 0xFFu;
      total += (1u << (w & 31u)) >> 1;
      top = w > top ? w : top;
    }
  }
  if (top > kHufLogMax || total == 0) return kErrTable;
  const uint32_t log = highbit(total) + 1;
  if (log > kHufLogMax) return kErrTable;
  const uint32_t rest = (1u << log) - total;
  if (rest & (rest - 1)) return kErrTable;
  const uint32_t nsym = nw + 1, last = highbit(rest) + 1;
  // A symbol of weight w has 2^(w-1) entries, after those of all lower weights
  // and of the symbols of its own weight before it. A run starts at a multiple
  // of its length (the runs from it on are multiples of it, and all together
  // fill the table), so runs of four and more are written four at a time.
  for (uint32_t s = tm.lane(); s < nsym; s += Team::size) {
    const uint32_t w = s < nw ? weight[s] : last;
    if (!w) continue;
    uint32_t pos = s < nw && last < w ? 1u << (last - 1) : 0u;
    for (uint32_t r = 0; r < nw; r += 16) {
      uint32_t w4[4];
      load_weights(weight, nw, r, w4);
#pragma unroll
      for (uint32_t k = 0; k < 16; ++k) {
        const uint32_t v = (w4[k >> 2] >> (8 * (k & 3))) & 0xFFu;
        pos += v < w + (r + k < s) ? (1u << v) >> 1 : 0u;
      }
    }
    const uint32_t e = s | ((log + 1 - w) << 8), run = 1u << (w - 1);
    if (run < 4) {
      for (uint32_t k = 0; k < run; ++k) z.huf[pos + k] = (uint16_t)e;
    } else {
      const uint64_t e4 = (uint64_t)e * 0x0001000100010001ull;
      for (uint32_t k = 0; k < run; k += 4) __builtin_memcpy(__builtin_assume_aligned(z.huf + pos + k, 8), &e4, 8);
    }
  }
  if (tm.lane() == 0) z.huf_log = log;
  tm.sync();
  return kOk;
}

// Bits [o, o + 32) of s[0, n) as one little-endian number (bit 0: the lowest
// bit of s[0]); bits outside it read as zeros.
__host__ __device__ inline uint32_t bits32(const uint8_t* s, uint32_t n, int32_t o) {
  const int32_t j = o >> 3;
  uint64_t v = 0;
#pragma unroll
  for (int32_t i = 0; i < 5; ++i)
    if ((uint32_t)(j + i) < n) v |= (uint64_t)s[j + i] << (8 * i);
  return (uint32_t)(v >> (o & 7));
}

// Walks NJ chains of codes of a stream q[0, n) of T bits through windows of 32
// bits from bit `at` to `to` (`at` plus a multiple of 32; the stream may end
// before it). `win` holds the 64 bits from `at` on, p[j] the bit of chain j's
// next code in them, c[j] its symbols so far.
template <uint32_t NJ>
__host__ __device__ __forceinline__ void huf_walk(const ZState& z, const uint8_t* q, uint32_t n, uint32_t T, uint32_t at,
                                                  uint32_t to, uint32_t log, uint64_t& win, uint32_t (&p)[NJ],
                                                  uint32_t (&c)[NJ]) {
  const uint32_t mask = (1u << log) - 1, sh = 64 - log;
  for (; at < to && at < T; at += 32) {
    const uint32_t lim = T - at < 32 ? T - at : 32, next = bits32(q, n, (int32_t)(T - at) - 96);
    if (NJ == 1) {
      while (p[0] < lim) {
        p[0] += z.huf[(uint32_t)(win >> (sh - p[0])) & mask] >> 8;
        ++c[0];
      }
    } else {
      for (;;) {
        bool any = false;
#pragma unroll
        for (uint32_t j = 0; j < NJ; ++j) any = any || p[j] < lim;
        if (!any) break;
#pragma unroll
        for (uint32_t j = 0; j < NJ; ++j) {
          const uint32_t bits = z.huf[(uint32_t)(win >> (sh - p[j])) & mask] >> 8;
          const bool on = p[j] < lim;
          p[j] += on ? bits : 0u;
          c[j] += on;
        }
      }
    }
#pragma unroll
    for (uint32_t j = 0; j < NJ; ++j) p[j] -= lim;
    win = (win << 32) | next;
  }
}

// The 64 bits of stream q from bit `at` on.
__host__ __device__ __forceinline__ uint64_t huf_window(const uint8_t* q, uint32_t n, uint32_t T, uint32_t at) {
  return ((uint64_t)bits32(q, n, (int32_t)(T - at) - 32) << 32) | bits32(q, n, (int32_t)(T - at) - 64);
}

// Chains o, o + 4, .. of NJ of one piece (quarters of gq bits from bit p0): their
// ends into hop[], their places at the piece's inner quarters into m[j][].
template <uint32_t NJ>
__host__ __device__ __forceinline__ void huf_piece(const ZState& z, const uint8_t* q, uint32_t n, uint32_t T, uint32_t p0,
                                                   uint32_t gq, uint32_t o, uint16_t* hop, uint16_t (&m)[3][3]) {
  const uint32_t log = z.huf_log;
  uint32_t p[NJ], c[NJ];
#pragma unroll
  for (uint32_t j = 0; j < NJ; ++j) {
    p[j] = o + 4 * j;
    c[j] = 0;
  }
  uint64_t win = huf_window(q, n, T, p0);
#pragma unroll
  for (uint32_t k = 0; k < 4; ++k) {
    huf_walk<NJ>(z, q, n, T, p0 + k * gq, p0 + (k + 1) * gq, log, win, p, c);
#pragma unroll
    for (uint32_t j = 0; j < NJ; ++j) {
      const uint16_t v = (uint16_t)(p[j] | (c[j] << 4));
      if (k < 3) m[j][k < 3 ? k : 0] = v;
      else if (o + 4 * j < log) hop[o + 4 * j] = v;
    }
  }
}

// The Huffman streams z.hs[0, ns) of one literal section at `s` (their sizes
// checked), stream i's symbols to out + i * seg. Every lane calls it after a
// sync; returns whether every stream ends where it must, after a sync.
//
// A code's place is known only once all codes before it are, so a stream is a
// serial chain: one lane per stream took 60 % of a small frame's time. But a code
// is at most 12 bits long, so a piece of a stream can be entered at one of at
// most 12 bits. The streams are cut into kHufGroups pieces, and four lanes (of as
// many wavefronts) walk a piece from every such bit, up to three chains a lane;
// then the true walk hops from piece to piece, one step each; the lane that
// walked the true chain tells where it was at the piece's quarters, and four
// lanes walk a quarter each and write its symbols. Walking counts symbols of at
// least one bit, so a stream is right exactly when the walk ends on its last bit
// with the expected count. MI355X, 65 frames of 4,096 four-bit indices: 220 -> 74 us
// with tables built by all lanes and one wavefront per frame, 44 to 50 us with four
// and the literals in LDS.
template <class Team>
__host__ __device__ __forceinline__ bool huf_streams(const Team& tm, ZState& z, const uint8_t* s, uint32_t ns,
                                                     uint32_t seg, uint8_t* out) {
  constexpr uint32_t kItems = 4 * kHufGroups, kPerLane = (kItems + Team::size - 1) / Team::size;
  const uint32_t log = z.huf_log, per = kHufGroups / ns;
  uint32_t most = 0;
  for (uint32_t i = 0; i < ns; ++i) most = z.hs[i].bits > most ? z.hs[i].bits : most;
  for (uint32_t base = 0; base < most;) {
    // the pieces of this pass: four quarters of whole 32-bit windows
    const uint32_t even = ((most - base + 4 * per - 1) / (4 * per) + 31u) & ~31u;
    const uint32_t gq = even < kHufQuarterMax ? even : kHufQuarterMax;
    uint16_t m[kPerLane][3][3];
#pragma unroll
    for (uint32_t i = 0; i < kPerLane; ++i) {
      const uint32_t it = i * Team::size + tm.lane(), g = it % kHufGroups, o = it / kHufGroups;
      if (it >= kItems || o >= log) continue;
      const uint32_t st = g / per, T = z.hs[st].bits, p0 = base + (g - st * per) * 4 * gq;
      if (p0 >= T) continue;
      const uint8_t* q = s + z.hs[st].off;
      const uint32_t n = (T >> 3) + 1;
      uint16_t* hop = z.h.hop + g * kHufLogMax;
      if (log <= 4) huf_piece<1>(z, q, n, T, p0, gq, o, hop, m[i]);
      else if (log <= 8) huf_piece<2>(z, q, n, T, p0, gq, o, hop, m[i]);
      else huf_piece<3>(z, q, n, T, p0, gq, o, hop, m[i]);
    }
    tm.sync();
    for (uint32_t st = tm.lane(); st < ns; st += Team::size) {
      const uint32_t bits = z.hs[st].bits;
      uint32_t at = z.hs[st].at;
      for (uint32_t g = 0; g < per && base + g * 4 * gq < bits; ++g) {
        z.entry[st * per + g] = at;
        // the low fields: the new bit, and symbols added above it
        at = (at & ~15u) + z.h.hop[(st * per + g) * kHufLogMax + (at & 15u)];
      }
      z.hs[st].at = at;
    }
    tm.sync();
#pragma unroll
    for (uint32_t i = 0; i < kPerLane; ++i) {
      const uint32_t it = i * Team::size + tm.lane(), g = it % kHufGroups, o = it / kHufGroups;
      if (it >= kItems || o >= log) continue;
      const uint32_t st = g / per;
      if (base + (g - st * per) * 4 * gq >= z.hs[st].bits) continue;
      const uint32_t e = z.entry[g] & 15u;
#pragma unroll
      for (uint32_t j = 0; j < 3; ++j)
        if (o + 4 * j == e)
          for (uint32_t k = 0; k < 3; ++k) z.mark[g][k] = m[i][j][k];
    }
    tm.sync();
    for (uint32_t it = tm.lane(); it < kItems; it += Team::size) {
      const uint32_t g = it % kHufGroups, k = it / kHufGroups, st = g / per, T = z.hs[st].bits;
      const uint32_t a = base + ((g - st * per) * 4 + k) * gq;
      if (a >= T) continue;
      const uint32_t n = (T >> 3) + 1, count = z.hs[st].count, mask = (1u << log) - 1, sh = 64 - log;
      const uint8_t* q = s + z.hs[st].off;
      uint8_t* d = out + (uint64_t)st * seg;
      const uint32_t e = z.entry[g], v = k ? z.mark[g][k - 1] : e & 15u;
      uint32_t p = v & 15u, j = (e >> 4) + (v >> 4);
      uint64_t win = huf_window(q, n, T, a);
      for (uint32_t at = a; at < a + gq && at < T; at += 32) {
        const uint32_t lim = T - at < 32 ? T - at : 32, next = bits32(q, n, (int32_t)(T - at) - 96);
        while (p < lim) {
          const uint32_t h = z.huf[(uint32_t)(win >> (sh - p)) & mask];
          if (j < count) d[j] = (uint8_t)h;
          ++j;
          p += h >> 8;
        }
        p -= lim;
        win = (win << 32) | next;
      }
    }
    tm.sync();
    base += per * 4 * gq;
  }
  bool ok = true;
  for (uint32_t i = 0; i < ns; ++i) ok = ok && z.hs[i].at == z.hs[i].count << 4;
  return ok;
}

// Sets up one sequence table (literal lengths 0, offsets 1, match lengths 2)
// for `mode` from b[0, n); returns the bytes taken or -1. Every lane calls it
// after a sync; the table and its log are visible after the next one.
template <class Team>
__host__ __device__ inline int32_t seq_table(const Team& tm, ZState& z, uint32_t kind, uint32_t mode, const uint8_t* b,
                                             uint64_t n) {
  FseCell* t = kind == 0 ? z.ll : kind == 1 ? z.of : z.ml;
  uint32_t* log = kind == 0 ? &z.ll_log : kind == 1 ? &z.of_log : &z.ml_log;
  uint32_t* have = kind == 0 ? &z.have_ll : kind == 1 ? &z.have_of : &z.have_ml;
  const uint32_t max_sym = kind == 0 ? kLLMax : kind == 1 ? kOFMax : kMLMax;
  const uint32_t max_log = kind == 0 ? kLLLog : kind == 1 ? kOFLog : kMLLog;
  if (mode == 3) return *have ? 0 : -1; // repeat
  uint32_t lg = 0, used = 0;
  if (mode == 0) {                      // predefined
    const FseCell* f = kind == 0 ? kFixed.ll : kind == 1 ? kFixed.of : kFixed.ml;
    lg = kind == 1 ? 5u : 6u;
    for (uint32_t u = tm.lane(); u < 1u << lg; u += Team::size) t[u] = f[u];
  } else if (mode == 1) {               // RLE: one symbol
    if (n < 1 || b[0] > max_sym) return -1;
    if (tm.lane() == 0) t[0] = FseCell{0, b[0], 0};
    used = 1;
  } else {                              // FSE-compressed
    if (tm.lane() == 0) z.val[0] = read_ncount(b, n, z.b.norm, max_sym, max_log, z.val[1], z.val[2]);
    tm.sync();
    used = z.val[0];
    lg = z.val[1];
    if (!used || !build_fse(tm, z, t, z.val[2], lg)) return -1;
  }
  if (tm.lane() == 0) {
    *log = lg;
    *have = 1;
  }
  return (int32_t)used;
}

// Output positions are frame-relative inside dst; `frame0` is where the frame
// starts. Every lane holds the same values.
struct Out {
  uint8_t* dst;
  uint64_t cap;
  uint64_t op;
  uint64_t frame0;
};

template <class Team>
__host__ __device__ inline void team_fill(const Team& tm, uint8_t* d, uint8_t v, uint64_t n) {
  for (uint64_t i = tm.lane(); i < n; i += Team::size) d[i] = v;
}
// N lanes copy s[0, n) to d, which it does not overlap: four bytes per lane in
// flight (past the end, the last byte again).
template <uint32_t N>
__host__ __device__ inline void copy_bytes(uint32_t lane, uint8_t* d, const uint8_t* s, uint64_t n) {
  for (uint64_t i = lane; i < n; i += 4 * N) {
    uint8_t v[4];
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
      const uint64_t j = i + k * N;
      v[k] = s[j < n ? j : n - 1];
    }
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k)
      if (i + k * N < n) d[i + k * N] = v[k];
  }
}
template <class Team>
__host__ __device__ inline void team_copy(const Team& tm, uint8_t* d, const uint8_t* s, uint64_t n) {
  copy_bytes<Team::size>(tm.lane(), d, s, n);
}

// One sequence at dst + op by N lanes: ll literals from lit, then ml bytes from
// `off` before them. Match byte i is d[ll - off + i % off]: earlier output, or
// this sequence's literals (then read from the literal buffer).
template <uint32_t N>
__host__ __device__ inline void run_sequence(uint32_t lane, uint8_t* dst, uint64_t op, const uint8_t* lit, uint32_t ll,
                                             uint32_t ml, uint32_t off) {
  if (ll > N) copy_bytes<N>(lane, dst + op, lit, ll);
  else if (lane < ll) dst[op + lane] = lit[lane];
  const uint64_t from = op + ll - off;
  if (off >= ml) {
    for (uint32_t j = lane; j < ml; j += N) {
      const uint64_t src = from + j;
      dst[op + ll + j] = src >= op ? lit[src - op] : dst[src];
    }
  } else {
    // j mod off kept incrementally: j grows by N each round (off < ml < 2^32, so
    // this is 32-bit arithmetic and two divisions per sequence instead of one
    // 64-bit modulo per byte)
    const uint32_t step = N % off;
    uint32_t r = lane % off;
    for (uint32_t j = lane; j < ml; j += N) {
      const uint64_t src = from + r;
      dst[op + ll + j] = src >= op ? lit[src - op] : dst[src];
      r += step;
      if (r >= off) r -= off;
    }
  }
}

// The sequences of a block: nseq of them from the bitstream b[pos, n), literals
// from lit[0, lsize); o.op and lp move on. LEAD: run by the team's leading lanes,
// who share the long ones with the others (below); else by all lanes alike.
template <bool LEAD, class Team>
__host__ __device__ __forceinline__ int32_t run_sequences(const Team& tm, ZState& z, const uint8_t* b, uint64_t n,
                                                          uint64_t pos, uint32_t nseq, Out& o, Rep& rep,
                                                          const uint8_t* lit, uint32_t lsize, uint64_t& lp) {
  BackBits br;
  if (pos >= n || !br.init(b + pos, n - pos)) return kErrStream;
  uint32_t sll = br.read(z.ll_log), sof = br.read(z.of_log), sml = br.read(z.ml_log);
  uint64_t visible = o.op;              // output below this is visible to every lane
  for (uint32_t i = 0; i < nseq; ++i) {
    const FseCell cl = z.ll[sll], co = z.of[sof], cm = z.ml[sml];
    const uint32_t ofc = co.sym & 31u;
    const uint32_t ofv = (1u << ofc) + br.read(ofc);
    const uint32_t ml = z.ml_base[cm.sym] + br.read(z.ml_bits[cm.sym]);
    const uint32_t ll = z.ll_base[cl.sym] + br.read(z.ll_bits[cl.sym]);
    uint32_t off;
    if (ofv > 3) {
      off = ofv - 3;
      rep.r2 = rep.r1;
      rep.r1 = rep.r0;
      rep.r0 = off;
    } else {                            // a repeat: shifted by one when the literal length is 0
      const uint32_t r = ofv - 1 + (ll == 0 ? 1u : 0u);
      if (r == 0) {
        off = rep.r0;
      } else {
        off = r == 1 ? rep.r1 : r == 2 ? rep.r2 : rep.r0 - 1;
        if (r != 1) rep.r2 = rep.r1;
        rep.r1 = rep.r0;
        rep.r0 = off;
      }
    }
    if (i + 1 < nseq) {                 // state updates: literal lengths, match lengths, offsets
      sll = cl.base + br.read(cl.nb);
      sml = cm.base + br.read(cm.nb);
      sof = co.base + br.read(co.nb);
    }
    // One branch for all that may be wrong: a block of short sequences is bound by
    // the instructions between two of them, and a branch costs 20 cycles and more.
    // With 32-bit copy loops, MI355X: consecutive int64 numbers (a sequence per 8
    // bytes), 300 KB 37.3 -> 35.5 ms, text of 300 KB 30.5 -> 28.8 ms.
    const bool bad_stream = (co.sym > kOFMax) | (br.bits() < 0) | (lp + ll > lsize);
    const bool bad_output = o.op + ll + ml > o.cap, bad_offset = (off == 0) | (off > o.op + ll - o.frame0);
    if (bad_stream | bad_output | bad_offset) return bad_stream ? kErrStream : bad_output ? kErrOutput : kErrOffset;
    if (LEAD && (ll | ml) >= kLongSequence) {
      if (tm.lane() == 0) {
        z.seq.op = o.op;
        z.seq.lp = (uint32_t)lp;
        z.seq.ll = ll;
        z.seq.ml = ml;
        z.seq.off = off;
        z.seq.more = 1;
      }
      tm.sync();
      run_sequence<Team::size>(tm.lane(), o.dst, o.op, lit + lp, ll, ml, off);
      tm.sync();
      visible = o.op + ll + ml;
    } else {
      // a match that reads output above `visible` waits for it first
      const uint64_t from = o.op + ll - off, reach = from + (off < ml ? off : ml);
      if ((reach < o.op ? reach : o.op) > visible) {
        if (LEAD) tm.lead_sync();
        else tm.sync();
        visible = o.op;
      }
      run_sequence<LEAD ? Team::lead_size : Team::size>(tm.lane(), o.dst, o.op, lit + lp, ll, ml, off);
    }
    o.op += ll + ml;
    lp += ll;
  }
  return br.bits() == 0 ? kOk : kErrStream;
}

// One compressed block b[0, n) (RFC 8878 3.1.1.3). rep: repeat offsets. Literals
// that are not read in place go to near[0, room) if they fit, else to lit_far.
template <class Team>
__host__ __device__ __forceinline__ int32_t zstd_block(const Team& tm, ZState& z, const uint8_t* b, uint64_t n,
                                                       Out& o, Rep& rep, uint8_t* near, uint32_t room,
                                                       uint8_t* lit_far) {
  if (n < 1) return kErrTruncated;
  const uint32_t ltype = b[0] & 3u, sf = (b[0] >> 2) & 3u;
  uint32_t lh, lsize, lcsize = 0;
  bool four = false;
  if (ltype < 2) {
    lh = (sf & 1u) ? (sf == 1 ? 2u : 3u) : 1u;
    if (n < lh) return kErrTruncated;
    const uint32_t v = (uint32_t)load_le(b, lh, 0);
    lsize = lh == 1 ? v >> 3 : v >> 4;
  } else {
    lh = sf < 2 ? 3u : sf == 2 ? 4u : 5u;
    if (n < lh) return kErrTruncated;
    const uint64_t v = load_le(b, lh, 0);
    four = sf != 0;
    if (sf < 2) {
      lsize = (uint32_t)(v >> 4) & 0x3FFu;
      lcsize = (uint32_t)(v >> 14) & 0x3FFu;
    } else if (sf == 2) {
      lsize = (uint32_t)(v >> 4) & 0x3FFFu;
      lcsize = (uint32_t)(v >> 18) & 0x3FFFu;
    } else {
      lsize = (uint32_t)(v >> 4) & 0x3FFFFu;
      lcsize = (uint32_t)(v >> 22) & 0x3FFFFu;
    }
  }
  if (lsize > kBlockMax) return kErrFormat;
  uint64_t pos = lh;
  uint8_t* lit_buf = lsize <= room ? near : lit_far;
  const uint8_t* lit = lit_buf;
  if (ltype == 0) {                     // raw literals: read in place
    if (pos + lsize > n) return kErrTruncated;
    lit = b + pos;
    pos += lsize;
  } else if (ltype == 1) {              // RLE literals
    if (pos + 1 > n) return kErrTruncated;
    team_fill(tm, lit_buf, b[pos], lsize);
    tm.sync();
    pos += 1;
  } else {                              // Huffman-coded (2: with a new tree, 3: the previous tree)
    if (pos + lcsize > n) return kErrTruncated;
    const uint8_t* q = b + pos;
    uint32_t tree = 0;
    if (ltype == 2) {
      if (lcsize < 1) return kErrTruncated;
      tree = huf_desc_bytes(q[0]);
      if (tree > lcsize) return kErrTruncated;
      const int32_t e = build_huffman(tm, z, q);
      if (e) return e;
    } else if (z.huf_log == 0) {
      return kErrTable;
    }
    const uint8_t* s = q + tree;
    const uint32_t sn = lcsize - tree;
    const uint32_t ns = four ? 4u : 1u, seg = four ? (lsize + 3) / 4 : lsize;
    uint32_t l1 = sn, l2 = 0, l3 = 0, l4 = 0, at = 0;
    if (four) {
      if (sn < 6) return kErrTruncated;
      l1 = (uint32_t)load_le(s, 2, 0);
      l2 = (uint32_t)load_le(s + 2, 2, 0);
      l3 = (uint32_t)load_le(s + 4, 2, 0);
      if (6ull + l1 + l2 + l3 > sn) return kErrTruncated;
      l4 = sn - 6 - l1 - l2 - l3;
      if (3 * seg > lsize) return kErrFormat;
      at = 6;
    }
    // a stream's last byte holds its end: the highest set bit
    if (tm.lane() == 0) z.err = kOk;
    tm.sync();
    for (uint32_t st = tm.lane(); st < ns; st += Team::size) {
      const uint32_t off = at + (st > 0 ? l1 : 0) + (st > 1 ? l2 : 0) + (st > 2 ? l3 : 0);
      const uint32_t len = st == 0 ? l1 : st == 1 ? l2 : st == 2 ? l3 : l4;
      const uint8_t end = len ? s[off + len - 1] : (uint8_t)0;
      if (end == 0) {
        z.err = kErrStream;
      } else {
        z.hs[st].bits = (len - 1) * 8 + highbit(end);
        z.hs[st].off = off;
        z.hs[st].count = st < ns - 1 ? seg : lsize - (ns - 1) * seg;
        z.hs[st].at = 0;
      }
    }
    tm.sync();
    if (z.err || !huf_streams(tm, z, s, ns, seg, lit_buf)) return kErrStream;
    pos += lcsize;
  }

  // sequences section header (RFC 8878 3.1.1.3.2.1)
  if (pos >= n) return kErrTruncated;
  uint32_t nseq = b[pos];
  if (nseq == 0) {
    pos += 1;
  } else if (nseq < 128) {
    pos += 1;
  } else if (nseq < 255) {
    if (pos + 2 > n) return kErrTruncated;
    nseq = ((nseq - 128) << 8) + b[pos + 1];
    pos += 2;
  } else {
    if (pos + 3 > n) return kErrTruncated;
    nseq = b[pos + 1] + ((uint32_t)b[pos + 2] << 8) + 0x7F00u;
    pos += 3;
  }
  uint64_t lp = 0;                      // literals consumed
  if (nseq > 0) {
    if (pos >= n) return kErrTruncated;
    const uint32_t modes = b[pos++];
    if (modes & 3u) return kErrFormat;
    tm.sync();                          // the scratch's earlier use is over
    for (uint32_t k = 0; k < 3; ++k) {  // LL, OF, ML
      const int32_t used = seq_table(tm, z, k, (modes >> (6 - 2 * k)) & 3u, b + pos, n - pos);
      tm.sync();
      if (used < 0) return kErrTable;
      pos += (uint32_t)used;
    }
    // Most sequences of a block of many are a few bytes long, and each waits for its
    // bits, its table entries and the output it copies from, so more wavefronts
    // add nothing but a barrier between them and their share of the issue slots:
    // the leading lanes run them, and the others wait for a long one or the end.
    // A few sequences among many bytes want every lane, and no hand-over. MI355X, a
    // frame of 168 KB of text by all lanes / the leading ones 17.3 / 16.5 ms, 768 side
    // by side 20.8 / 18.8; 65 vectors of 4,096 indices (three or four sequences
    // each) 46.1 / 48 us. A sequence is long from 128 bytes on, two rounds of the
    // leading lanes: 4 MB of repeats of 300 bytes 16.9 ms by all lanes alike, 18.3
    // handed over from 512 bytes, 14.7 from 256 or 128; runs of 200 bytes on average
    // 24.5, 23.8, 22.7 and 22.2 ms.
    if (Team::size == Team::lead_size || nseq < kFewSequences) {
      const int32_t e = run_sequences<false>(tm, z, b, n, pos, nseq, o, rep, lit, lsize, lp);
      if (e) return e;
    } else {
      if (tm.leads()) {
        const int32_t e = run_sequences<true>(tm, z, b, n, pos, nseq, o, rep, lit, lsize, lp);
        if (tm.lane() == 0) {
          z.seq.op = o.op;
          z.seq.lp = (uint32_t)lp;
          z.seq.err = e;
          z.seq.more = 0;
          z.seq.rep = rep;
        }
        tm.sync();
      } else {
        for (;;) {
          tm.sync();
          if (!z.seq.more) break;
          run_sequence<Team::size>(tm.lane(), o.dst, z.seq.op, lit + z.seq.lp, z.seq.ll, z.seq.ml, z.seq.off);
          tm.sync();
        }
      }
      if (z.seq.err) return z.seq.err;
      o.op = z.seq.op;
      lp = z.seq.lp;
      rep = z.seq.rep;                  // a later block may be run by all lanes
    }
  }
  if (o.op + (lsize - lp) > o.cap) return kErrOutput;
  team_copy(tm, o.dst + o.op, lit + lp, lsize - lp);
  o.op += lsize - lp;
  tm.sync();
  return kOk;
}

// All frames in src[0, len) (zstd frames and skippable frames, back to back)
// into dst; *out_bytes receives the total decoded size.
template <class Team>
__host__ __device__ int32_t zstd_frames(const Team& tm, ZState& z, const uint8_t* src, uint64_t len, uint8_t* dst,
                                        uint64_t cap, uint8_t* lit_buf, uint64_t& out_bytes) {
  load_length_codes(tm, z);
  tm.sync();
  Out o{dst, cap, 0, 0};
  uint64_t ip = 0;
  out_bytes = 0;
  if (len == 0) return kErrTruncated;
  while (ip < len) {
    if (len - ip < 4) return kErrTruncated;
    const uint32_t magic = (uint32_t)load_le(src + ip, 4, 0);
    if ((magic & 0xFFFFFFF0u) == 0x184D2A50u) {          // skippable frame
      if (len - ip < 8) return kErrTruncated;
      const uint64_t sz = (uint32_t)load_le(src + ip + 4, 4, 0);
      if (sz > len - ip - 8) return kErrTruncated;
      ip += 8 + sz;
      continue;
    }
    if (magic != 0xFD2FB528u) return kErrFormat;
    ip += 4;
    if (ip >= len) return kErrTruncated;
    const uint32_t fhd = src[ip++];
    const uint32_t fcs_flag = fhd >> 6, single = (fhd >> 5) & 1u, checksum = (fhd >> 2) & 1u, did = fhd & 3u;
    if (fhd & 8u) return kErrFormat;                     // reserved bit
    const uint32_t did_bytes = did == 3 ? 4u : did;
    const uint32_t fcs_bytes = fcs_flag == 0 ? single : fcs_flag == 1 ? 2u : fcs_flag == 2 ? 4u : 8u;
    const uint64_t hdr = (single ? 0u : 1u) + did_bytes + fcs_bytes;
    if (hdr > len - ip) return kErrTruncated;
    ip += single ? 0u : 1u;
    if (did_bytes && load_le(src + ip, did_bytes, 0) != 0) return kErrFormat;   // dictionaries: unsupported
    ip += did_bytes;
    uint64_t fcs = fcs_bytes ? load_le(src + ip, fcs_bytes, 0) : 0;
    if (fcs_bytes == 2) fcs += 256;
    ip += fcs_bytes;
    o.frame0 = o.op;
    if (tm.lane() == 0) z.huf_log = z.have_ll = z.have_ml = z.have_of = 0;
    tm.sync();
    Rep rep{1u, 4u, 8u};
    for (;;) {
      if (len - ip < 3) return kErrTruncated;
      const uint32_t bh = (uint32_t)load_le(src + ip, 3, 0);
      ip += 3;
      const uint32_t last = bh & 1u, type = (bh >> 1) & 3u, bsize = bh >> 3;
      if (type == 0) {                                   // raw block
        if (bsize > len - ip) return kErrTruncated;
        if (bsize > o.cap - o.op) return kErrOutput;
        team_copy(tm, o.dst + o.op, src + ip, bsize);
        o.op += bsize;
        ip += bsize;
      } else if (type == 1) {                            // RLE block
        if (ip >= len) return kErrTruncated;
        if (bsize > o.cap - o.op) return kErrOutput;
        team_fill(tm, o.dst + o.op, src[ip], bsize);
        o.op += bsize;
        ip += 1;
      } else if (type == 2) {
        if (bsize > len - ip) return kErrTruncated;
        if (bsize > kBlockMax) return kErrFormat;
        int32_t e;
        if (bsize <= kStageBytes) {     // bit reads then come from shared memory, not global memory
          team_copy(tm, z.stage, src + ip, bsize);
          tm.sync();
          e = zstd_block(tm, z, z.stage, bsize, o, rep, z.stage + bsize, kStageBytes - bsize, lit_buf);
        } else {
          e = zstd_block(tm, z, src + ip, bsize, o, rep, z.stage, kStageBytes, lit_buf);
        }
        if (e) return e;
        ip += bsize;
      } else {
        return kErrFormat;
      }
      tm.sync();
      if (last) break;
    }
    if (checksum) {
      if (len - ip < 4) return kErrTruncated;
      ip += 4;
    }
    if (fcs_bytes && o.op - o.frame0 != fcs) return kErrOutput;
  }
  out_bytes = o.op;
  return kOk;
}

}  // namespace bs_zstd
