// Fragment-file import on the device: the text of a fragment file (lines
// "chrom\tstart\tend\tbarcode[\tcount[\tstrand]]") becomes the per-cell fragment
// store (CSR: row = barcode, column = genome base index, value = length) plus
// the per-barcode QC counts.
//
// Reference:
//   import_fragments / make_arraydata / count_fragments
//     (snapatac2-core/src/preprocessing/import.rs:31-204);
//   Fragment::from_str (snapatac2-core/src/preprocessing/qc.rs:306-345);
//   FragmentQCBuilder (qc.rs:427-466);
//   import_fragments and shift_fragment (snapatac2-python/src/preprocessing.rs:87-183).
//
// Steps (all on one stream; the host reads three scalars back in between):
//   1. newline count per 64 KiB block, scan, newline positions -> line starts;
//   2. one lane per line parses its fields (tab separated; eight characters at
//      a time where the line is an ordinary one), looks the chromosome up in a
//      hashed name table and writes per-line records;
//   3. the records with end > start are compacted;
//   4. each record gets its barcode's group in file order: the run of equal
//      barcodes it stands in (input sorted by barcode), or its entry in a hash
//      table (unsorted input; equal 64-bit hashes of different barcodes are
//      reported);
//   5. one radix sort of (group, position, value) in one 64-bit key, or, where the
//      three need more bits, a sort by (position, value) and a stable one by group;
//   6. QC sums per group by segmented wave sums; whitelist and minimum-count
//      filters; the groups of unsorted input are ranked by their barcode bytes
//      (LSD sort of 8-byte big-endian words), which is the reference's
//      external-sort order;
//   7. fill: each fragment of a kept group goes to row offset + its rank.
#include <hipcub/hipcub.hpp>

#include <cstring>
#include <type_traits>

#include "common.h"

namespace snapgpu {
namespace frag {

constexpr int kThreads = 256;
constexpr int kRounds = 16;                                     // 16-byte words per thread
constexpr int64_t kByteBlock = (int64_t)kThreads * kRounds * 16;  // 64 KiB of text per block
constexpr int64_t kLineBlock = (int64_t)kThreads * kRounds;       // 4096 records per block

// per-line flags
constexpr uint8_t F_KEEP = 1;     // a record with end != start (import.rs:66)
constexpr uint8_t F_GENOME = 2;   // chromosome in the genome (import.rs:168)
constexpr uint8_t F_MITO = 4;     // chromosome in the mitochondrial list
constexpr uint8_t F_STRAND = 8;   // a strand field is present (single-end record)
constexpr uint8_t F_REV = 16;     // strand '-'
constexpr uint8_t F_RANGE = 32;   // stored coordinate >= chromosome length (genome.rs:387-406)
constexpr uint8_t F_HUGE = 64;    // end - start > 2^32 - 1
constexpr uint8_t F_BIG = 128;    // +-(end - start) outside int32

// error codes (low byte of the error word; the line index is above it)
enum : uint32_t {
  E_START_MISSING = 1,
  E_END_MISSING = 2,
  E_BARCODE_MISSING = 3,
  E_START_BAD = 4,
  E_END_BAD = 5,
  E_COUNT_BAD = 6,
  E_STRAND_BAD = 7,
  E_BARCODE_NONE = 8,
  E_END_BEFORE_START = 9,
  E_BARCODE_LONG = 10,
  E_REVERSE_PAIRED = 11,
  E_SIZE_I32 = 12,
  E_RANGE = 13,
  E_SIZE_U32 = 14,
};

// Host-packed hashed name table (chromosomes, or a barcode whitelist):
// header | slots[cap] | entries[n] | name bytes.
struct TableHeader {
  uint32_t n, cap;
  uint64_t total;  // sum of lengths (chromosome table)
};
struct TableSlot {
  uint64_t hash;
  int32_t idx;  // -1 = empty
  int32_t pad;
};
struct TableEntry {
  uint64_t base, length;
  uint32_t name_off, name_len, flags, pad;
};
static_assert(sizeof(TableHeader) == 16 && sizeof(TableSlot) == 16 && sizeof(TableEntry) == 32, "layout");

struct Counters {
  unsigned long long err;       // min (line << 8 | code) over parse errors
  unsigned long long first;     // min (line << 1 | has_strand) over records
  unsigned long long n_rec;     // records (not comments, not empty)
  unsigned long long n_strand;  // records with a strand field
  unsigned long long bad;       // min (line << 8 | code) over conversion errors in whitelisted groups
  unsigned long long dup;       // min group index of a barcode seen in two runs
  unsigned int max_bc;          // longest barcode (bytes) over kept records
  unsigned int collision;       // two barcodes with one hash next to each other
  unsigned int any_bad;         // a whitelisted group holds a record count_fragments cannot convert
  unsigned int max_size;        // largest end - start (low 32 bits) over kept records
  unsigned long long n_groups;  // distinct barcodes of unsorted input
  unsigned int recount;         // a block's newlines are not as many as were counted
};

// How the records were sorted, for the kernels that read the result: the key holds
// group << pv | position << (vb + mb) | value << mb | mitochondrial, with mb = 1 for
// unsorted input; `alt`: the sorted keys (and counts) are in the second buffers.
// one = 0: the records are in order of a permutation instead.
struct SortPlan {
  uint64_t total;  // genome length: the position of records outside the genome
  uint32_t max_size;
  int32_t one, alt, pv, vb, mb, paired;
};
__device__ __forceinline__ uint64_t key_group(uint64_t key, const SortPlan& p) { return p.pv < 64 ? key >> p.pv : 0; }
__device__ __forceinline__ uint64_t key_pv(uint64_t key, const SortPlan& p) {
  return p.pv < 64 ? key & ((1ull << p.pv) - 1) : key;
}

// Hash of a name, eight bytes at a time (little endian, zeros past the end): a
// multiply and a shift per word on top of the length, and one more at the end.
__host__ __device__ inline uint64_t hash_start(uint32_t len) { return 0x2545F4914F6CDD1Dull + len; }
__host__ __device__ inline uint64_t hash_step(uint64_t h, uint64_t w) {
  h = (h ^ w) * 0x9E3779B97F4A7C15ull;
  return h ^ (h >> 32);
}
__host__ __device__ inline uint64_t hash_end(uint64_t h) {
  h *= 0xD6E8FEB86659FD93ull;
  return h ^ (h >> 32);
}
constexpr int64_t kNamePad = 8;  // readable bytes after a table's names

__device__ __forceinline__ uint8_t load_byte(const uint8_t* t, int64_t p) { return t[p]; }

// 8 bytes at the aligned address a (little endian); bytes at or past n read as 0.
__device__ __forceinline__ uint64_t load_word(const uint8_t* t, int64_t a, int64_t n) {
  if (a + 8 <= n) return *reinterpret_cast<const uint64_t*>(t + a);
  uint64_t w = 0;
  for (int k = 0; k < 8 && a + k < n; ++k) w |= (uint64_t)t[a + k] << (8 * k);
  return w;
}

// 8 bytes at any address (all readable).
struct __attribute__((packed)) Bytes8 {
  uint64_t v;
};
__device__ __forceinline__ uint64_t load8(const uint8_t* p) { return reinterpret_cast<const Bytes8*>(p)->v; }

// The first n (1 to 8) bytes of a word.
__device__ __forceinline__ uint64_t first_bytes(uint64_t w, uint32_t n) { return w & (~0ull >> (64 - 8 * n)); }

// 8 bytes at any offset p; bytes at or past n read as 0.
__device__ __forceinline__ uint64_t load_u8x8(const uint8_t* t, int64_t p, int64_t n) {
  if (p + 8 <= n) return load8(t + p);
  uint64_t w = 0;
  for (int k = 0; k < 8 && p + k < n; ++k) w |= (uint64_t)t[p + k] << (8 * k);
  return w;
}

// The text where it lies, and the part of it that a block holds in LDS (from byte
// `first`, a multiple of 16): eight bytes at any offset.
struct FarText {
  const uint8_t* t;
  int64_t n;
  __device__ __forceinline__ uint64_t at(int64_t off) const { return load_u8x8(t, off, n); }
};
struct NearText {
  const uint32_t* w;
  int64_t first;
  __device__ __forceinline__ uint64_t at(int64_t off) const {
    const uint32_t r = (uint32_t)(off - first), k = r >> 2;
    const uint32_t a = w[k], b = w[k + 1], c = w[k + 2];
    return ((uint64_t)__builtin_amdgcn_alignbyte(c, b, r & 3) << 32) | __builtin_amdgcn_alignbyte(b, a, r & 3);
  }
};

template <typename Text>
__device__ __forceinline__ uint64_t hash_text(const Text& t, int64_t off, uint32_t len) {
  uint64_t h = hash_start(len);
  for (uint32_t k = 0; k < len; k += 8) {
    const uint64_t w = t.at(off + k);
    h = hash_step(h, len - k < 8 ? first_bytes(w, len - k) : w);
  }
  return hash_end(h);
}

// Index of the name at offset off of the text in a table, or -1.
template <typename Text>
__device__ int table_find(const uint8_t* tab, uint64_t h, const Text& t, int64_t off, uint32_t len) {
  const TableHeader* H = reinterpret_cast<const TableHeader*>(tab);
  const uint32_t cap = H->cap, n = H->n;
  const TableSlot* S = reinterpret_cast<const TableSlot*>(tab + sizeof(TableHeader));
  const TableEntry* E = reinterpret_cast<const TableEntry*>(S + cap);
  const uint8_t* names = reinterpret_cast<const uint8_t*>(E + n);
  uint32_t i = (uint32_t)h & (cap - 1);
  for (uint32_t probe = 0; probe < cap; ++probe, i = (i + 1) & (cap - 1)) {
    const TableSlot sl = S[i];
    if (sl.idx < 0) return -1;
    if (sl.hash == h) {
      const TableEntry e = E[sl.idx];
      bool same = e.name_len == len;
      for (uint32_t k = 0; same && k < len; k += 8) {
        const uint64_t x = load8(names + e.name_off + k) ^ t.at(off + k);
        same = (len - k < 8 ? first_bytes(x, len - k) : x) == 0;
      }
      if (same) return sl.idx;
    }
  }
  return -1;
}

__device__ __forceinline__ const TableEntry& table_entry(const uint8_t* tab, int idx) {
  const TableHeader* H = reinterpret_cast<const TableHeader*>(tab);
  const TableSlot* S = reinterpret_cast<const TableSlot*>(tab + sizeof(TableHeader));
  return reinterpret_cast<const TableEntry*>(S + H->cap)[idx];
}

// Number of bytes equal to c in x.
__device__ __forceinline__ int count_byte(uint32_t x, uint32_t pat) {
  const uint32_t v = x ^ pat;
  uint32_t y = (v & 0x7F7F7F7Fu) + 0x7F7F7F7Fu;
  y = ~(y | v | 0x7F7F7F7Fu);
  return __popc(y);
}

// 16-bit mask of the bytes equal to '\n' in a 16-byte word (bit k = byte k).
__device__ __forceinline__ uint32_t newline_mask(uint4 w) {
  uint32_t m = 0;
  const uint32_t x[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const uint32_t v = x[q] ^ 0x0A0A0A0Au;
    uint32_t y = (v & 0x7F7F7F7Fu) + 0x7F7F7F7Fu;
    y = ~(y | v | 0x7F7F7F7Fu);  // 0x80 in each byte equal to '\n'
    m |= (((y >> 7) & 1u) | ((y >> 14) & 2u) | ((y >> 21) & 4u) | ((y >> 28) & 8u)) << (4 * q);
  }
  return m;
}

// The 16 bytes of word index wi (bytes past n_bytes read as 0, not '\n').
__device__ __forceinline__ uint4 load16(const uint8_t* t, int64_t wi, int64_t n) {
  const int64_t off = wi * 16;
  if (off + 16 <= n) return *reinterpret_cast<const uint4*>(t + off);
  uint32_t x[4] = {0, 0, 0, 0};
  for (int k = 0; k < 16 && off + k < n; ++k) x[k >> 2] |= (uint32_t)t[off + k] << (8 * (k & 3));
  return make_uint4(x[0], x[1], x[2], x[3]);
}

template <typename T>
__device__ T block_sum(T v, T* lds) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d, 64);
  if (lane == 0) lds[wid] = v;
  __syncthreads();
  T s = 0;
  for (int k = 0; k < kThreads / 64; ++k) s += lds[k];
  __syncthreads();
  return s;
}

// ---------------------------------------------------------------------------
// 1. lines
// ---------------------------------------------------------------------------

__global__ void __launch_bounds__(kThreads) nl_count_kernel(const uint8_t* __restrict__ text, int64_t n,
                                                            int64_t* __restrict__ blk) {
  __shared__ int64_t red[kThreads / 64];
  const int64_t w0 = (int64_t)blockIdx.x * kThreads * kRounds;
  int64_t c = 0;
  for (int r = 0; r < kRounds; ++r) {
    const int64_t wi = w0 + (int64_t)r * kThreads + threadIdx.x;
    if (wi * 16 < n) {
      const uint4 w = load16(text, wi, n);
      c += count_byte(w.x, 0x0A0A0A0Au) + count_byte(w.y, 0x0A0A0A0Au) + count_byte(w.z, 0x0A0A0A0Au) +
           count_byte(w.w, 0x0A0A0A0Au);
    }
  }
  c = block_sum<int64_t>(c, red);
  if (threadIdx.x == 0) blk[blockIdx.x] = c;
}

// line_start[0] = 0 and line_start[k + 1] = (position of newline k) + 1.
// blk_incl: inclusive scan of the per-block newline counts. A block that finds another
// number (a text that has changed since it was counted, a workspace of another text)
// says so, and n_lines bounds the writes: where none does, every entry is written.
__global__ void __launch_bounds__(kThreads) nl_index_kernel(const uint8_t* __restrict__ text, int64_t n,
                                                            const int64_t* __restrict__ blk_incl, int64_t n_lines,
                                                            int64_t* __restrict__ line_start, Counters* cnt) {
  __shared__ int64_t wsum[kThreads / 64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int64_t w0 = (int64_t)blockIdx.x * kThreads * kRounds;
  int64_t base = blockIdx.x == 0 ? 0 : blk_incl[blockIdx.x - 1];
  if (blockIdx.x == 0 && threadIdx.x == 0) line_start[0] = 0;
  for (int r = 0; r < kRounds; ++r) {
    const int64_t wi = w0 + (int64_t)r * kThreads + threadIdx.x;
    uint32_t m = 0;
    if (wi * 16 < n) m = newline_mask(load16(text, wi, n));
    const uint64_t c = (uint64_t)__popc(m);
    const uint64_t incl = wave_incl_scan_u64(c, lane);
    if (lane == 63) wsum[wid] = (int64_t)incl;
    __syncthreads();
    int64_t before = 0, total = 0;
    for (int k = 0; k < kThreads / 64; ++k) {
      const int64_t s = wsum[k];
      before += k < wid ? s : 0;
      total += s;
    }
    int64_t o = base + before + (int64_t)(incl - c);
    while (m) {
      const int k = __ffs(m) - 1;
      m &= m - 1;
      if ((uint64_t)o < (uint64_t)n_lines) line_start[1 + o] = wi * 16 + k + 1;
      ++o;
    }
    base += total;
    __syncthreads();
  }
  if (threadIdx.x == 0 && base != blk_incl[blockIdx.x]) atomicOr(&cnt->recount, 1u);
}

// ---------------------------------------------------------------------------
// 2. parse
// ---------------------------------------------------------------------------

struct ParseOut {
  uint32_t* pos;
  uint32_t* size;
  uint32_t* cnt;
  uint8_t* flags;
  uint64_t* bc;   // barcode offset << 8 | length
  uint64_t* bch;  // hash of the barcode (unsorted input, else null)
};

__device__ __forceinline__ uint64_t sat_add(uint64_t a, int64_t d) {
  if (d >= 0) {
    const uint64_t r = a + (uint64_t)d;
    return r < a ? ~0ull : r;
  }
  const uint64_t m = (uint64_t)(-(d + 1)) + 1;  // |d| without overflow
  return a < m ? 0 : a - m;
}

struct LineStats {
  uint32_t n_rec, n_strand, n_keep, max_bc, max_size;
  unsigned long long first;  // min (line << 1 | has_strand) over records
};

// The fields of a record line.
struct Fields {
  uint64_t start, end;
  int64_t bc_off;
  uint32_t chrom_len, bc_len, count, strand;  // strand: 0 none, 1 '+', 2 '-'
};

// Eight characters whose first 8 - n stand before the field: their value as a
// decimal number, or false if one of the last n (1 to 8) is no digit.
__device__ __forceinline__ bool digits8(uint64_t w, uint32_t n, uint32_t* value) {
  const uint64_t pad = n == 8 ? 0 : ~0ull >> (8 * n);  // bytes before the field
  w = (w & ~pad) | (0x3030303030303030ull & pad);
  const uint32_t a = (uint32_t)w ^ 0x30303030u, b = (uint32_t)(w >> 32) ^ 0x30303030u;  // 0 to 9 each, if digits
  // a byte of 10 to 15 carries into its high half when 6 is added
  if (((a | (a + 0x06060606u) | b | (b + 0x06060606u)) & 0xF0F0F0F0u) != 0) return false;
  const uint32_t hi = __builtin_amdgcn_udot4(a, 0x0000010Au, 0u, false) * 100u + __builtin_amdgcn_udot4(a, 0x010A0000u, 0u, false);
  const uint32_t lo = __builtin_amdgcn_udot4(b, 0x0000010Au, 0u, false) * 100u + __builtin_amdgcn_udot4(b, 0x010A0000u, 0u, false);
  *value = hi * 10000u + lo;
  return true;
}

// The number in the n characters that end before offset p.
__device__ __forceinline__ bool digits(const NearText& t, int64_t p, uint32_t n, uint64_t* value) {
  if (n == 0 || n > 16) return false;
  uint32_t lo, hi = 0;
  if (!digits8(t.at(p - 8), n < 8 ? n : 8, &lo)) return false;
  if (n > 8 && !digits8(t.at(p - 16), n - 8, &hi)) return false;
  *value = (uint64_t)hi * 100000000ull + lo;
  return true;
}

// The fields of an ordinary record line [s, e) of staged text: at least four fields,
// at most 64 characters, numbers of digits. The tabs come as one 64-bit mask from
// the aligned words that hold the line, each number from the eight characters before
// its end. False: the line goes through parse_fields (comments, errors, '.' fields,
// long lines).
__device__ __forceinline__ bool quick_fields(const NearText& t, int64_t s, int64_t e, Fields& f) {
  const int len = (int)min<int64_t>(e - s, 65);
  if (len < 7 || len > 64) return false;
  const uint32_t r = (uint32_t)(s - t.first), skip = r & 3;
  const uint32_t* w = t.w + (r >> 2);
  if ((uint8_t)(w[0] >> (8 * skip)) == '#') return false;
  uint64_t tabs = 0;
  uint32_t over = 0;
#pragma unroll
  for (int k = 0; k < 17; k += 2) {
    if (4 * k < len + (int)skip) {
      uint32_t m[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint32_t x = (k + h < 17 ? w[k + h] : 0) ^ 0x09090909u;
        const uint32_t y = (x & 0x7F7F7F7Fu) + 0x7F7F7F7Fu;
        m[h] = (~(y | x) & 0x80808080u) >> 7;  // 1 in each byte that is a tab
      }
      const uint32_t bits = __builtin_amdgcn_udot4(m[1], 0x80402010u, __builtin_amdgcn_udot4(m[0], 0x08040201u, 0u, false), false);
      if (k < 16) tabs |= (uint64_t)bits << (4 * k);
      else over = bits;
    }
  }
  tabs >>= skip;
  if (skip) tabs |= (uint64_t)over << (64 - skip);
  tabs &= ~0ull >> (64 - len);
  if (popc64(tabs) < 3) return false;
  const int t1 = lowbit64(tabs);
  tabs &= tabs - 1;
  const int t2 = lowbit64(tabs);
  tabs &= tabs - 1;
  const int t3 = lowbit64(tabs);
  tabs &= tabs - 1;
  const int t4 = tabs ? lowbit64(tabs) : len;
  f.chrom_len = t1;
  f.bc_off = s + t3 + 1;
  f.bc_len = t4 - t3 - 1;
  if (t1 == 0 || f.bc_len < 2) return false;
  if (!digits(t, s + t2, t2 - t1 - 1, &f.start) || !digits(t, s + t3, t3 - t2 - 1, &f.end)) return false;
  f.count = 1;
  f.strand = 0;
  if (tabs) {
    tabs &= tabs - 1;
    const int t5 = tabs ? lowbit64(tabs) : len;
    uint64_t v;
    if (t5 - t4 - 1 > 8 || !digits(t, s + t5, t5 - t4 - 1, &v)) return false;
    f.count = (uint32_t)v;
    if (tabs) {
      tabs &= tabs - 1;
      const int t6 = tabs ? lowbit64(tabs) : len;
      const uint32_t c = (uint32_t)t.at(s + t5 + 1) & 255u;
      if (t6 - t5 - 1 != 1 || (c != '+' && c != '-')) return false;
      f.strand = c == '+' ? 1 : 2;
    }
  }
  return true;
}

// The fields of any record line, one character after the other; an E_ code or 0.
__device__ __forceinline__ uint32_t parse_fields(const uint8_t* __restrict__ text, int64_t n_bytes, int64_t s, int64_t e,
                                              Fields& f, uint32_t& bc_c0) {
  // current field
  uint32_t field = 0, flen = 0, c0 = 0;
  uint64_t num = 0;
  bool nondigit = false;
  int64_t fstart = s;
  bool start_bad = false, end_bad = false, count_bad = false, strand_bad = false;
  f = Fields{0, 0, s, 0, 0, 1, 0};
  bc_c0 = 0;
  int64_t a = s & ~(int64_t)7;
  uint64_t word = load_word(text, a, n_bytes);
  for (int64_t p = s; p <= e; ++p) {
    uint32_t c = '\t';
    if (p < e) {
      if ((p & ~(int64_t)7) != a) {
        a = p & ~(int64_t)7;
        word = load_word(text, a, n_bytes);
      }
      c = (uint32_t)(word >> (8 * (p & 7))) & 0xFFu;
    }
    if (c == '\t') {
      const bool bad = nondigit || flen == 0;
      switch (field) {
        case 0: f.chrom_len = flen; break;
        case 1: f.start = num; start_bad = bad; break;
        case 2: f.end = num; end_bad = bad; break;
        case 3: f.bc_off = fstart; f.bc_len = flen; bc_c0 = c0; break;
        case 4:
          if (flen == 1 && c0 == '.') f.count = 1;
          else { f.count = (uint32_t)num; count_bad = bad || num > 0xFFFFFFFFull; }
          break;
        case 5:
          if (flen == 1 && c0 == '.') f.strand = 0;
          else if (flen == 1 && c0 == '+') f.strand = 1;
          else if (flen == 1 && c0 == '-') f.strand = 2;
          else strand_bad = true;
          break;
        default: break;
      }
      ++field;
      flen = 0;
      num = 0;
      nondigit = false;
      fstart = p + 1;
    } else {
      const uint32_t d = c - '0';
      const bool dig = d < 10;
      const bool ovf = num > 1844674407370955161ull || (num == 1844674407370955161ull && d > 5);
      nondigit |= !dig || ovf;
      num = num * 10 + (dig ? d : 0);
      c0 = flen == 0 ? c : c0;
      ++flen;
    }
  }
  if (field < 2) return E_START_MISSING;
  if (start_bad) return E_START_BAD;
  if (field < 3) return E_END_MISSING;
  if (end_bad) return E_END_BAD;
  if (field < 4) return E_BARCODE_MISSING;
  if (count_bad) return E_COUNT_BAD;
  if (strand_bad) return E_STRAND_BAD;
  return 0;
}

// Parses line i and writes its record; accumulates the block statistics. Returns
// the barcode (as in ParseOut) of a record that is kept, or 0.
template <typename Text>
__device__ __forceinline__ uint64_t parse_line(const Text& t, const uint8_t* __restrict__ text, int64_t n_bytes,
                                           const int64_t* __restrict__ line_start, int64_t i,
                                           const uint8_t* __restrict__ chroms, int64_t shift_left,
                                           int64_t shift_right, const ParseOut& out, Counters* cnt,
                                           LineStats& ls) {
  bool is_rec = false, has_strand = false;
  uint32_t err = 0, bc_len_keep = 0;
  uint64_t kept = 0;
  {
    const int64_t s = line_start[i];
    int64_t e = line_start[i + 1] - 1;
    if (e > n_bytes) e = n_bytes;
    if (e > s && (t.at(e - 1) & 255) == '\r') --e;
    uint8_t fl = 0;
    uint32_t pos = 0, size = 0, count = 1;
    uint64_t bcw = 0, bch = 0;
    Fields f{0, 0, s, 0, 0, 1, 0};
    uint32_t bc_c0 = 0;
    bool rec = false;
    if constexpr (std::is_same_v<Text, NearText>) rec = quick_fields(t, s, e, f);
    if (!rec && e > s && load_byte(text, s) != '#') {
      rec = true;
      err = parse_fields(text, n_bytes, s, e, f, bc_c0);
    }
    if (rec) {
      is_rec = true;
      count = f.count;
      has_strand = f.strand != 0;  // a '.' strand field is no strand (qc.rs:338-344)
      if (err == 0) {
        // shift_fragment (preprocessing.rs:173-183)
        const uint64_t st = shift_left != 0 ? sat_add(f.start, shift_left) : f.start;
        uint64_t en = f.end;
        if (has_strand && shift_left != 0) en = sat_add(f.end, shift_left);
        if (!has_strand && shift_right != 0) en = sat_add(f.end, shift_right);
        if (en < st) {
          err = E_END_BEFORE_START;
        } else if (en > st) {
          fl |= F_KEEP;
          if (f.bc_len == 1 && bc_c0 == '.') err = E_BARCODE_NONE;
          else if (f.bc_len > 255) err = E_BARCODE_LONG;
          bc_len_keep = f.bc_len;
          if (has_strand) fl |= F_STRAND;
          if (f.strand == 2) fl |= F_REV;
          const uint64_t sz = en - st;
          size = (uint32_t)sz;
          if (sz > 0xFFFFFFFFull) fl |= F_HUGE;
          if (sz > (f.strand == 2 ? 2147483648ull : 2147483647ull)) fl |= F_BIG;
          const int ci = table_find(chroms, hash_text(t, s, f.chrom_len), t, s, f.chrom_len);
          if (ci >= 0) {
            const TableEntry& ce = table_entry(chroms, ci);
            fl |= F_GENOME;
            if (ce.flags & 1u) fl |= F_MITO;
            const uint64_t coord = f.strand == 2 ? en - 1 : st;
            if (coord >= ce.length) fl |= F_RANGE;
            else pos = (uint32_t)(ce.base + coord);
          }
          bcw = ((uint64_t)f.bc_off << 8) | (f.bc_len > 255 ? 255u : f.bc_len);
          if (err == 0 && out.bch) bch = hash_text(t, f.bc_off, f.bc_len);
        }
      }
    }
    out.pos[i] = pos;
    out.size[i] = size;
    out.cnt[i] = count;
    out.flags[i] = err ? 0 : fl;
    out.bc[i] = bcw;
    if (out.bch) out.bch[i] = bch;
    if (err) atomicMin(&cnt->err, ((unsigned long long)i << 8) | err);
    if (!err && (fl & F_KEEP)) {
      kept = bcw;
      ++ls.n_keep;
      ls.max_size = size > ls.max_size ? size : ls.max_size;
    }
  }
  if (is_rec) {
    ++ls.n_rec;
    ls.n_strand += has_strand ? 1 : 0;
    const unsigned long long f = ((unsigned long long)i << 1) | (has_strand ? 1ull : 0ull);
    ls.first = f < ls.first ? f : ls.first;
  }
  ls.max_bc = bc_len_keep > ls.max_bc ? bc_len_keep : ls.max_bc;
  return kept;
}

// The text of a round's 256 lines is read once, in order, into LDS (kStage bytes; 16
// below it and kStagePad above are read past a line's ends and masked away): a lane
// reads its line in some thirty pieces, and from global memory those went to L2 again
// and again (2.94 ms for 55 million lines of 41 characters that way, 1.93 ms staged;
// 4.13 ms one character after the other, 0.9 ms the copy of the bytes alone). Rounds of longer lines read
// the text where it lies, one character after the other.
constexpr int kStage = 16384, kStagePad = 96;

// same[i] (input sorted by barcode, else null): 1 if this line and the one before
// are kept and their barcodes are known to be equal (both were staged).
//
// kLineBlock lines per block (lane t of round r takes line b0 + r * 256 + t);
// blk[block] = records kept. The block statistics go to the counters with one
// atomic each, so the counters see a few tens of thousands of atomics.
__global__ void __launch_bounds__(kThreads) parse_kernel(const uint8_t* __restrict__ text, int64_t n_bytes,
                                                         const int64_t* __restrict__ line_start, int64_t n_lines,
                                                         const uint8_t* __restrict__ chroms, int64_t shift_left,
                                                         int64_t shift_right, ParseOut out, Counters* cnt,
                                                         int64_t* __restrict__ blk, uint8_t* __restrict__ same) {
  __shared__ unsigned long long red[6][kThreads / 64];
  __shared__ uint4 stage[1 + kStage / 16 + kStagePad / 16];
  __shared__ uint64_t barcode[kThreads];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int64_t b0 = (int64_t)blockIdx.x * kLineBlock;
  LineStats ls{0, 0, 0, 0, 0, ~0ull};
  for (int r = 0; r < kRounds; ++r) {
    const int64_t i0 = b0 + (int64_t)r * kThreads, i = i0 + threadIdx.x;
    if (i0 >= n_lines) break;
    const int64_t w0 = line_start[i0] / 16;
    const int64_t stop = min(n_bytes, line_start[min(i0 + kThreads, n_lines)]);
    if (stop - 16 * w0 <= kStage) {
      for (int64_t w = w0 + threadIdx.x; 16 * w < stop; w += kThreads) stage[1 + w - w0] = load16(text, w, n_bytes);
      __syncthreads();
      const NearText near{reinterpret_cast<const uint32_t*>(stage), 16 * w0 - 16};
      uint64_t b = 0;
      if (i < n_lines)
        b = parse_line(near, text, n_bytes, line_start, i, chroms, shift_left, shift_right, out, cnt, ls);
      if (same) {
        barcode[threadIdx.x] = b;
        __syncthreads();
        if (i < n_lines) {
          const uint64_t p = threadIdx.x > 0 ? barcode[threadIdx.x - 1] : 0;
          const uint32_t len = (uint32_t)(b & 255);
          bool eq = b && p && (uint32_t)(p & 255) == len;
          for (uint32_t k = 0; eq && k < len; k += 8) {
            const uint64_t x = near.at((int64_t)(b >> 8) + k) ^ near.at((int64_t)(p >> 8) + k);
            eq = (len - k < 8 ? first_bytes(x, len - k) : x) == 0;
          }
          same[i] = eq ? 1 : 0;
        }
      }
      __syncthreads();
    } else if (i < n_lines) {
      parse_line(FarText{text, n_bytes}, text, n_bytes, line_start, i, chroms, shift_left, shift_right, out, cnt, ls);
      if (same) same[i] = 0;
    }
  }
  unsigned long long v[6] = {ls.n_rec, ls.n_strand, ls.n_keep, ls.max_bc, ls.first, ls.max_size};
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
#pragma unroll
    for (int q = 0; q < 3; ++q) v[q] += __shfl_xor(v[q], d, 64);
    const unsigned long long m = __shfl_xor(v[3], d, 64), f = __shfl_xor(v[4], d, 64),
                             z = __shfl_xor(v[5], d, 64);
    v[3] = m > v[3] ? m : v[3];
    v[4] = f < v[4] ? f : v[4];
    v[5] = z > v[5] ? z : v[5];
  }
  if (lane == 0)
    for (int q = 0; q < 6; ++q) red[q][wid] = v[q];
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kThreads / 64; ++w) {
      for (int q = 0; q < 3; ++q) v[q] += red[q][w];
      v[3] = red[3][w] > v[3] ? red[3][w] : v[3];
      v[4] = red[4][w] < v[4] ? red[4][w] : v[4];
      v[5] = red[5][w] > v[5] ? red[5][w] : v[5];
    }
    blk[blockIdx.x] = (int64_t)v[2];
    if (v[0]) atomicAdd(&cnt->n_rec, v[0]);
    if (v[1]) atomicAdd(&cnt->n_strand, v[1]);
    if (v[3] && v[3] > *reinterpret_cast<volatile unsigned int*>(&cnt->max_bc))
      atomicMax(&cnt->max_bc, (unsigned int)v[3]);
    if (v[4] != ~0ull && v[4] < *reinterpret_cast<volatile unsigned long long*>(&cnt->first))
      atomicMin(&cnt->first, v[4]);
    if (v[5] && v[5] > *reinterpret_cast<volatile unsigned int*>(&cnt->max_size))
      atomicMax(&cnt->max_size, (unsigned int)v[5]);
  }
}

// ---------------------------------------------------------------------------
// 3. compaction of the kept records (file order)
// ---------------------------------------------------------------------------

__global__ void __launch_bounds__(kThreads) keep_write_kernel(const uint8_t* __restrict__ flags, int64_t n,
                                                              const int64_t* __restrict__ blk_incl,
                                                              uint32_t* __restrict__ kept) {
  __shared__ int64_t wsum[kThreads / 64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int64_t b0 = (int64_t)blockIdx.x * kLineBlock;
  int64_t base = blockIdx.x == 0 ? 0 : blk_incl[blockIdx.x - 1];
  for (int r = 0; r < kRounds; ++r) {
    const int64_t i = b0 + (int64_t)r * kThreads + threadIdx.x;
    const bool k = i < n && (flags[i] & F_KEEP);
    const uint64_t bal = ballot64(k);
    if (lane == 0) wsum[wid] = popc64(bal);
    __syncthreads();
    int64_t before = 0, total = 0;
    for (int q = 0; q < kThreads / 64; ++q) {
      const int64_t s = wsum[q];
      before += q < wid ? s : 0;
      total += s;
    }
    if (k) kept[base + before + popc64(bal & lanemask_lt(lane))] = (uint32_t)i;
    base += total;
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// 4. sort keys and barcode comparisons
// ---------------------------------------------------------------------------

// Equality of the len bytes at offsets a and b, eight at a time.
__device__ __forceinline__ bool text_equal(const uint8_t* t, int64_t n, int64_t a, int64_t b, uint32_t len) {
  for (uint32_t k = 0; k < len; k += 8) {
    const uint64_t x = load_u8x8(t, a + k, n) ^ load_u8x8(t, b + k, n);
    const uint32_t rem = len - k;
    const uint64_t mask = rem >= 8 ? ~0ull : ((1ull << (8 * rem)) - 1);
    if (x & mask) return false;
  }
  return true;
}

__global__ void iota_kernel(uint32_t* __restrict__ v, int64_t n) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j < n) v[j] = (uint32_t)j;
}

// (position, value) of a record: position above the value, the value offset by
// max_size for single-end records so that -size .. +size order as integers. Records
// outside the genome get the genome's length as position (above every genome key)
// and sort last inside their group.
__device__ __forceinline__ uint64_t pv_of(uint8_t f, uint32_t pos, uint32_t size, const SortPlan& p) {
  if (!(f & F_GENOME)) return p.total << (p.vb + p.mb);
  const uint64_t v = p.paired ? size : ((f & F_REV) ? (uint64_t)p.max_size - size : (uint64_t)p.max_size + size);
  return ((((uint64_t)pos << p.vb) | v) << p.mb) | (p.mb && (f & F_MITO) ? 1ull : 0ull);
}

// Boundaries of equal-barcode runs over kept records in file order (input
// sorted by barcode): run[v] = 1 where a new run starts. What the parser could not
// tell from staged text (the first line of its rounds, after a line that was not kept)
// is compared here. 55 million records: 0.91 ms with every barcode compared here (the
// text once more), 0.39 so, and 0.1 more in the parser.
__global__ void __launch_bounds__(kThreads) run_bound_kernel(const uint8_t* __restrict__ text, int64_t n_bytes,
                                                             const uint32_t* __restrict__ kept,
                                                             const uint64_t* __restrict__ bc,
                                                             const uint8_t* __restrict__ same, int64_t n,
                                                             int64_t* __restrict__ run) {
  const int64_t v = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  const uint32_t line = v < n ? kept[v] : 0;
  uint32_t before = (uint32_t)__shfl_up((int)line, 1, 64);
  if (v >= n) return;
  if ((threadIdx.x & 63) == 0) before = v > 0 ? kept[v - 1] : 0;
  bool eq = v > 0 && line == before + 1 && same[line];
  if (!eq && v > 0) {
    const uint64_t a = bc[line], b = bc[before];
    eq = (a & 255) == (b & 255) && text_equal(text, n_bytes, (int64_t)(a >> 8), (int64_t)(b >> 8), (uint32_t)(a & 255));
  }
  run[v] = eq ? 0 : 1;
}

// Groups of unsorted input: each record's barcode hash in a table of 2 n slots
// (empty: all ones), whose index is written down; the first to arrive is the slot's
// representative. A plain load that still sees an empty slot is settled by the atomics.
// (0.23 ms for 20.5 million records of 3,001 barcodes, and 0.75 for the comparison
// below, which reads the text again: 1.0 GB.)
constexpr uint64_t kEmpty = ~0ull;

__global__ void __launch_bounds__(kThreads) group_slot_kernel(const uint32_t* __restrict__ kept,
                                                              const uint64_t* __restrict__ bch, int64_t n,
                                                              unsigned long long* __restrict__ slots,
                                                              uint32_t* __restrict__ rep, uint32_t* __restrict__ slot) {
  const int64_t v = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (v >= n) return;
  uint64_t h = bch[kept[v]];
  if (h == kEmpty) --h;
  const uint64_t cap = 2 * (uint64_t)n;
  uint64_t s = __umul64hi(h, cap);
  for (uint64_t probe = 0; probe < cap; ++probe) {
    unsigned long long cur = slots[s];
    if (cur == kEmpty) cur = __hip_atomic_load(&slots[s], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (cur == kEmpty) {
      cur = atomicCAS(&slots[s], (unsigned long long)kEmpty, (unsigned long long)h);
      if (cur == kEmpty) {
        rep[s] = (uint32_t)v;
        break;
      }
    }
    if (cur == h) break;
    s = s + 1 < cap ? s + 1 : 0;
  }
  slot[v] = (uint32_t)s;
}

// Numbers the occupied slots (in any order: the groups are ranked later) and keeps
// each group's representative line and its barcode.
__global__ void __launch_bounds__(kThreads) group_number_kernel(const unsigned long long* __restrict__ slots,
                                                                const uint32_t* __restrict__ rep, int64_t cap,
                                                                const uint32_t* __restrict__ kept,
                                                                const uint64_t* __restrict__ bc,
                                                                uint32_t* __restrict__ id, uint32_t* __restrict__ gline,
                                                                uint64_t* __restrict__ gbc, Counters* cnt) {
  const int64_t s = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  const int lane = threadIdx.x & 63;
  const bool used = s < cap && slots[s] != kEmpty;
  const uint64_t bal = ballot64(used);
  if (!bal) return;
  const int lead = lowbit64(bal);
  uint64_t base = 0;
  if (lane == lead) base = atomicAdd(&cnt->n_groups, (unsigned long long)popc64(bal));
  base = shfl_u64(base, lead);
  if (!used) return;
  const uint64_t g = base + popc64(bal & lanemask_lt(lane));
  const uint32_t line = kept[rep[s]];
  id[s] = (uint32_t)g;
  gline[g] = line;
  gbc[g] = bc[line];
}

// run[v] = group + 1 of each record, whose barcode must be its representative's.
__global__ void __launch_bounds__(kThreads) group_of_kernel(const uint8_t* __restrict__ text, int64_t n_bytes,
                                                            const uint32_t* __restrict__ kept,
                                                            const uint64_t* __restrict__ bc,
                                                            const uint32_t* __restrict__ slot,
                                                            const uint32_t* __restrict__ id,
                                                            const uint64_t* __restrict__ gbc, int64_t n,
                                                            int64_t* __restrict__ run, Counters* cnt) {
  const int64_t v = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (v >= n) return;
  const uint32_t g = id[slot[v]];
  const uint64_t a = bc[kept[v]], b = gbc[g];
  run[v] = (int64_t)g + 1;
  if ((a & 255) != (b & 255) ||
      !text_equal(text, n_bytes, (int64_t)(a >> 8), (int64_t)(b >> 8), (uint32_t)(a & 255)))
    atomicOr(&cnt->collision, 1u);
}

// The sort key of each record in file order, with the group above (position, value)
// where one key holds both; its count beside it for unsorted input (else count =
// null). g_bad: the groups of records that count_fragments cannot convert.
__global__ void __launch_bounds__(kThreads) key_kernel(const uint32_t* __restrict__ kept,
                                                       const uint8_t* __restrict__ flags,
                                                       const uint32_t* __restrict__ pos,
                                                       const uint32_t* __restrict__ size,
                                                       const uint32_t* __restrict__ cnt_in,
                                                       const int64_t* __restrict__ run, int64_t n, SortPlan plan,
                                                       uint64_t* __restrict__ key, uint32_t* __restrict__ count,
                                                       unsigned int* __restrict__ g_bad) {
  const int64_t v = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (v >= n) return;
  const uint32_t line = kept[v];
  const uint8_t f = flags[line];
  const uint64_t g = (uint64_t)run[v] - 1;
  const uint64_t pv = pv_of(f, pos[line], size[line], plan);
  key[v] = plan.one && plan.pv < 64 ? (g << plan.pv) | pv : pv;
  if (count) count[v] = cnt_in[line];
  const uint32_t bad = f & (F_RANGE | F_HUGE | (plan.paired ? F_REV : F_BIG));
  if ((f & F_GENOME) && bad && (g_bad[g] & bad) != bad) atomicOr(&g_bad[g], bad);
}

// Second sort key of the two-sort order: the group.
__global__ void group_key_kernel(const uint32_t* __restrict__ perm, const int64_t* __restrict__ run, int64_t n,
                                 uint64_t* __restrict__ key) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  key[j] = (uint64_t)run[perm[j]];
}

// QC sums of the records of a wave (FragmentQCBuilder::update over the in-genome
// records, qc.rs:442-449), which goes through kSumRounds * 64 consecutive records
// and whose groups are contiguous: one atomic per sum and group. Atomics on one
// address go one after the other; with one per 64 records they were most of the
// time (55 million records, 8,000 groups: 545 us, 364 so; from the sorted keys of
// 20.5 million records 250 us and 81).
constexpr int kSumRounds = 8;
constexpr int kSumBlockRecords = kThreads * kSumRounds;

struct GroupSums {
  unsigned long long *total, *mito, *uniq;
  int64_t g = -1;  // the group whose records ended the last round; its sums (all lanes alike)
  uint64_t t = 0;
  uint32_t m = 0, u = 0;

  __device__ __forceinline__ void add(int64_t g_, uint64_t t_, uint32_t m_, uint32_t u_) {
    if (t_) atomicAdd(&total[g_], (unsigned long long)t_);
    if (m_) atomicAdd(&mito[g_], (unsigned long long)m_);
    if (u_) atomicAdd(&uniq[g_], (unsigned long long)u_);
  }

  // One record per lane (active lanes first). `first`: the record before is of another group.
  __device__ __forceinline__ void round(bool act, bool first, int64_t gr, bool genome, bool is_mito, uint64_t cnt) {
    const int lane = threadIdx.x & 63;
    const uint64_t on = ballot64(act);
    if (!on) return;
    const uint64_t heads = ballot64(act && (first || lane == 0));
    const uint64_t mitos = ballot64(act && genome && is_mito), uniqs = ballot64(act && genome && !is_mito);
    const uint64_t incl = wave_incl_scan_u64(act && genome ? cnt : 0, lane);
    const uint64_t upto = lanemask_lt(lane) | (1ull << lane);
    const uint64_t own = heads & upto;
    const int start = own ? 63 - __clzll((long long)own) : 0;
    const uint64_t before = shfl_u64(incl, start > 0 ? start - 1 : 0);
    const uint64_t piece = upto & ~lanemask_lt(start);
    const int last = 63 - __clzll((long long)on);
    uint64_t pt = incl - (start > 0 ? before : 0);
    uint32_t pm = popc64(mitos & piece), pu = popc64(uniqs & piece);
    const bool joins = (int64_t)shfl_u64((uint64_t)gr, 0) == g;
    if (joins && start == 0) {
      pt += t;
      pm += m;
      pu += u;
    }
    if (!joins && g >= 0 && lane == 0) add(g, t, m, u);
    // pieces that end before the last active lane are complete
    if (act && lane < last && (heads >> (lane + 1) & 1)) add(gr, pt, pm, pu);
    g = (int64_t)shfl_u64((uint64_t)gr, last);
    t = shfl_u64(pt, last);
    m = __shfl(pm, last, 64);
    u = __shfl(pu, last, 64);
  }

  __device__ __forceinline__ void finish() {
    if (g >= 0 && (threadIdx.x & 63) == 0) add(g, t, m, u);
  }
};

// First record of round r of this lane's wave.
__device__ __forceinline__ int64_t sum_record(int r) {
  return (int64_t)blockIdx.x * kSumBlockRecords + (int64_t)(threadIdx.x >> 6) * 64 * kSumRounds + r * 64 +
         (threadIdx.x & 63);
}

// Sums, start slot and (sorted input) first line of each group, with the records in
// file order (perm = null: input sorted by barcode, where the groups lie as they
// will when sorted) or in the order of a permutation.
__global__ void __launch_bounds__(kThreads) group_stats_kernel(
    const uint32_t* __restrict__ perm, const uint32_t* __restrict__ kept, const uint8_t* __restrict__ flags,
    const uint32_t* __restrict__ cnt_in, const int64_t* __restrict__ run, int64_t n, int64_t* __restrict__ gstart,
    uint32_t* __restrict__ gline, unsigned long long* __restrict__ g_total, unsigned long long* __restrict__ g_mito,
    unsigned long long* __restrict__ g_uniq) {
  GroupSums sums{g_total, g_mito, g_uniq};
  int64_t g[kSumRounds], prev[kSumRounds];
  uint32_t line[kSumRounds], cnt[kSumRounds];
  uint8_t f[kSumRounds];
#pragma unroll
  for (int r = 0; r < kSumRounds; ++r) {  // past the end: the last record, not used
    const int64_t j = min(sum_record(r), n - 1), v = perm ? perm[j] : j;
    line[r] = kept[v];
    g[r] = run[v] - 1;
    prev[r] = j > 0 ? run[perm ? perm[j - 1] : j - 1] - 1 : -1;
  }
#pragma unroll
  for (int r = 0; r < kSumRounds; ++r) {
    f[r] = flags[line[r]];
    cnt[r] = cnt_in[line[r]];
  }
#pragma unroll
  for (int r = 0; r < kSumRounds; ++r) {
    const int64_t j = sum_record(r);
    const bool act = j < n, first = act && prev[r] != g[r];
    if (first) {
      gstart[g[r]] = j;
      if (!perm) gline[g[r]] = line[r];
    }
    sums.round(act, first, g[r], (f[r] & F_GENOME) != 0, (f[r] & F_MITO) != 0, cnt[r]);
  }
  sums.finish();
}

// The same from the sorted keys of unsorted input and the counts beside them.
__global__ void __launch_bounds__(kThreads) key_stats_kernel(const uint64_t* __restrict__ key,
                                                             const uint32_t* __restrict__ count, int64_t n,
                                                             SortPlan plan, int64_t* __restrict__ gstart,
                                                             unsigned long long* __restrict__ g_total,
                                                             unsigned long long* __restrict__ g_mito,
                                                             unsigned long long* __restrict__ g_uniq) {
  GroupSums sums{g_total, g_mito, g_uniq};
  uint64_t k[kSumRounds], before[kSumRounds];
  uint32_t cnt[kSumRounds];
#pragma unroll
  for (int r = 0; r < kSumRounds; ++r) {  // past the end: the last record, not used
    const int64_t j = min(sum_record(r), n - 1);
    k[r] = key[j];
    before[r] = key[j > 0 ? j - 1 : 0];
    cnt[r] = count[j];
  }
#pragma unroll
  for (int r = 0; r < kSumRounds; ++r) {
    const int64_t j = sum_record(r), g = (int64_t)key_group(k[r], plan);
    const uint64_t pv = key_pv(k[r], plan);
    const bool act = j < n, first = act && (j == 0 || (int64_t)key_group(before[r], plan) != g);
    if (first) gstart[g] = j;
    sums.round(act, first, g, (pv >> (plan.vb + plan.mb)) < plan.total, (pv & 1) != 0, cnt[r]);
  }
  sums.finish();
}

// Whether a whitelisted group holds a record that count_fragments cannot
// convert (then bad_kernel names the first such line).
__global__ void bad_group_kernel(const unsigned int* __restrict__ g_bad, const uint8_t* __restrict__ wl,
                                 int64_t n_groups, int paired, Counters* cnt) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= n_groups) return;
  const uint32_t mask = F_RANGE | F_HUGE | (paired ? F_REV : F_BIG);
  if (wl[g] && (g_bad[g] & mask)) atomicOr(&cnt->any_bad, 1u);
}

// Whitelist membership of each group's barcode (import.rs:74).
__global__ void whitelist_kernel(const uint8_t* __restrict__ text, int64_t n_bytes,
                                 const uint32_t* __restrict__ gline,
                                 const uint64_t* __restrict__ bc, int64_t n_groups,
                                 const uint8_t* __restrict__ wl_table, uint8_t* __restrict__ wl) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= n_groups) return;
  uint8_t w = 1;
  if (wl_table) {
    const uint64_t b = bc[gline[g]];
    const FarText t{text, n_bytes};
    w = table_find(wl_table, hash_text(t, (int64_t)(b >> 8), (uint32_t)(b & 255)), t, (int64_t)(b >> 8),
                   (uint32_t)(b & 255)) >= 0 ? 1 : 0;
  }
  wl[g] = w;
}

__global__ void group_hash_kernel(const uint8_t* __restrict__ text, int64_t n_bytes,
                                  const uint32_t* __restrict__ gline, const uint64_t* __restrict__ bc,
                                  int64_t n_groups, uint64_t* __restrict__ key, uint32_t* __restrict__ idx) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= n_groups) return;
  const uint64_t b = bc[gline[g]];
  key[g] = hash_text(FarText{text, n_bytes}, (int64_t)(b >> 8), (uint32_t)(b & 255));
  idx[g] = (uint32_t)g;
}

// A barcode in two runs of sorted input (import.rs:139-141), among
// whitelisted groups: equal hashes next to each other after sorting by hash.
__global__ void dup_kernel(const uint8_t* __restrict__ text, int64_t n_bytes, const uint64_t* __restrict__ key,
                           const uint32_t* __restrict__ idx, const uint32_t* __restrict__ gline,
                           const uint64_t* __restrict__ bc, const uint8_t* __restrict__ wl, int64_t n_groups,
                           Counters* cnt) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r == 0 || r >= n_groups || key[r] != key[r - 1]) return;
  // scan back over the equal-hash run for the same barcode
  const uint32_t g = idx[r];
  if (!wl[g]) return;
  const uint64_t b = bc[gline[g]];
  for (int64_t q = r - 1; q >= 0 && key[q] == key[r]; --q) {
    const uint32_t h = idx[q];
    if (!wl[h]) continue;
    const uint64_t c = bc[gline[h]];
    if ((b & 255) == (c & 255) &&
        text_equal(text, n_bytes, (int64_t)(b >> 8), (int64_t)(c >> 8), (uint32_t)(b & 255))) {
      atomicMin(&cnt->dup, (unsigned long long)(g > h ? g : h));
      return;
    }
  }
}

// First record of a whitelisted group that count_fragments cannot convert
// (import.rs:173-198): coordinate outside the chromosome, or a size that does
// not fit the value type (u32 paired, i32 single-end).
__global__ void bad_kernel(const uint32_t* __restrict__ kept, const uint8_t* __restrict__ flags,
                           const int64_t* __restrict__ run, const uint8_t* __restrict__ wl, int64_t n, int paired,
                           Counters* cnt) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= n) return;
  const uint32_t line = kept[v];
  const uint8_t f = flags[line];
  if (!(f & F_GENOME) || !wl[run[v] - 1]) return;
  uint32_t code = 0;
  if (f & F_RANGE) code = E_RANGE;
  else if (f & F_HUGE) code = E_SIZE_U32;
  else if (paired && (f & F_REV)) code = E_REVERSE_PAIRED;
  else if (!paired && (f & F_BIG)) code = E_SIZE_I32;
  if (code) atomicMin(&cnt->bad, ((unsigned long long)line << 8) | code);
}

// Barcode length of each group, the least significant key of that order (a barcode
// before its own continuations by zero bytes), and the groups' numbers.
__global__ void length_key_kernel(const uint32_t* __restrict__ gline, const uint64_t* __restrict__ bc, int64_t n_groups,
                                  uint64_t* __restrict__ key, uint32_t* __restrict__ idx) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= n_groups) return;
  key[g] = bc[gline[g]] & 255;
  idx[g] = (uint32_t)g;
}

// Word w (8 bytes, big endian, zero padded) of each group's barcode, for the
// lexicographic LSD sort of the groups of unsorted input.
__global__ void word_key_kernel(const uint8_t* __restrict__ text, const uint32_t* __restrict__ order,
                                const uint32_t* __restrict__ gline, const uint64_t* __restrict__ bc,
                                int64_t n_groups, int w, uint64_t* __restrict__ key) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n_groups) return;
  const uint64_t b = bc[gline[order[r]]];
  const uint8_t* s = text + (b >> 8);
  const int len = (int)(b & 255);
  uint64_t k = 0;
  for (int q = 0; q < 8; ++q) {
    const int p = 8 * w + q;
    k = (k << 8) | (p < len ? s[p] : 0u);
  }
  key[r] = k;
}

// keep flag of the group at rank r (whitelisted and at least min unique
// fragments, import.rs:142-148), for the row scan.
__global__ void keep_rank_kernel(const uint32_t* __restrict__ order, const uint8_t* __restrict__ wl,
                                 const unsigned long long* __restrict__ g_uniq, int64_t n_groups, uint64_t min_frag,
                                 int64_t* __restrict__ kr) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n_groups) return;
  const uint32_t g = order ? order[r] : (uint32_t)r;
  kr[r] = (wl[g] && g_uniq[g] >= min_frag) ? 1 : 0;
}

// rowid[g] (-1 = dropped), rowgroup[row], row length (in-genome records).
__global__ void rows_kernel(const uint32_t* __restrict__ order, const int64_t* __restrict__ kr_incl,
                            const unsigned long long* __restrict__ g_uniq,
                            const unsigned long long* __restrict__ g_mito, int64_t n_groups,
                            int64_t* __restrict__ rowid, uint32_t* __restrict__ rowgroup,
                            int64_t* __restrict__ rowlen) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n_groups) return;
  const uint32_t g = order ? order[r] : (uint32_t)r;
  const int64_t inc = kr_incl[r], prev = r == 0 ? 0 : kr_incl[r - 1];
  if (inc != prev) {
    const int64_t row = inc - 1;
    rowid[g] = row;
    rowgroup[row] = g;
    rowlen[row] = (int64_t)(g_uniq[g] + g_mito[g]);
  } else {
    rowid[g] = -1;
  }
}

// ---------------------------------------------------------------------------
// 6. fill
// ---------------------------------------------------------------------------

// From the sorted keys, or record by record through the permutation.
__global__ void __launch_bounds__(kThreads) fill_kernel(
    const SortPlan* __restrict__ d_plan, const uint64_t* __restrict__ keyA, const uint64_t* __restrict__ keyB,
    const uint32_t* __restrict__ perm, const uint32_t* __restrict__ kept, const uint8_t* __restrict__ flags,
    const uint32_t* __restrict__ pos, const uint32_t* __restrict__ size, const int64_t* __restrict__ run,
    const int64_t* __restrict__ gstart, const int64_t* __restrict__ rowid, const int64_t* __restrict__ row_incl,
    int64_t n, uint32_t* __restrict__ out_pos, uint32_t* __restrict__ out_val) {
  const int64_t j = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (j >= n) return;
  const SortPlan plan = *d_plan;
  int64_t g;
  uint32_t p, val;
  if (plan.one) {
    const uint64_t key = (plan.alt ? keyB : keyA)[j];
    const uint64_t pv = key_pv(key, plan) >> plan.mb;
    if ((pv >> plan.vb) >= plan.total) return;
    g = (int64_t)key_group(key, plan);
    p = (uint32_t)(pv >> plan.vb);
    val = (uint32_t)(pv & ((1ull << plan.vb) - 1)) - (plan.paired ? 0u : plan.max_size);
  } else {
    const uint32_t v = perm[j], line = kept[v];
    const uint8_t f = flags[line];
    if (!(f & F_GENOME)) return;
    g = run[v] - 1;
    p = pos[line];
    const uint32_t sz = size[line];
    val = plan.paired ? sz : ((f & F_REV) ? (uint32_t)(0u - sz) : sz);
  }
  const int64_t row = rowid[g];
  if (row < 0) return;
  const int64_t o = (row == 0 ? 0 : row_incl[row - 1]) + (j - gstart[g]);
  out_pos[o] = p;
  out_val[o] = val;
}

__global__ void rows_out_kernel(const uint8_t* __restrict__ text, const uint32_t* __restrict__ rowgroup,
                                const uint32_t* __restrict__ gline, const uint64_t* __restrict__ bc,
                                const int64_t* __restrict__ row_incl, const unsigned long long* __restrict__ g_uniq,
                                const unsigned long long* __restrict__ g_total,
                                const unsigned long long* __restrict__ g_mito, int64_t n_rows,
                                int64_t* __restrict__ cell_ptr, unsigned long long* __restrict__ qc,
                                uint8_t* __restrict__ names, int width) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n_rows) return;
  const uint32_t g = rowgroup[r];
  if (r == 0) cell_ptr[0] = 0;
  cell_ptr[r + 1] = row_incl[r];
  if (qc) {
    qc[3 * r] = g_uniq[g];
    qc[3 * r + 1] = g_total[g];
    qc[3 * r + 2] = g_mito[g];
  }
  if (names) {
    const uint64_t b = bc[gline[g]];
    const uint8_t* s = text + (b >> 8);
    const int len = (int)(b & 255);
    uint8_t* o = names + r * (int64_t)width;
    for (int q = 0; q < width; ++q) o[q] = q < len ? s[q] : 0;
  }
}

// ---------------------------------------------------------------------------
// export: fragments -> text lines (Fragment's Display, qc.rs:286-303, as
// written by export_fragments, snapatac2-core/src/export.rs:90-106)
// ---------------------------------------------------------------------------

__device__ __forceinline__ int dec_digits(uint64_t x) {
  int d = 1;
  while (x >= 10) {
    x /= 10;
    ++d;
  }
  return d;
}

__device__ __forceinline__ void put_dec(uint8_t* o, uint64_t x, int d) {
  for (int k = d - 1; k >= 0; --k) {
    o[k] = (uint8_t)('0' + x % 10);
    x /= 10;
  }
}

struct FmtLine {
  uint32_t chrom;
  uint64_t start, end;
  uint32_t strand;  // 0 none, 1 '+', 2 '-'
  int64_t row;
};

__device__ FmtLine fmt_line(int64_t f, const int64_t* __restrict__ cell_ptr, int64_t n_cells,
                            const uint32_t* __restrict__ pos, const uint32_t* __restrict__ val, int paired,
                            const uint8_t* __restrict__ chroms) {
  FmtLine L{};
  int64_t lo = 0, hi = n_cells;  // last row with cell_ptr[row] <= f
  while (hi - lo > 1) {
    const int64_t mid = (lo + hi) / 2;
    if (cell_ptr[mid] <= f) lo = mid;
    else hi = mid;
  }
  L.row = lo;
  const TableHeader* H = reinterpret_cast<const TableHeader*>(chroms);
  const uint32_t n = H->n;
  const uint32_t p = pos[f];
  uint32_t a = 0, b = n;  // last chromosome with base <= p
  while (b - a > 1) {
    const uint32_t mid = (a + b) / 2;
    if (table_entry(chroms, mid).base <= p) a = mid;
    else b = mid;
  }
  L.chrom = a;
  const uint64_t coord = p - table_entry(chroms, a).base;
  if (paired) {
    L.start = coord;
    L.end = coord + val[f];
  } else {
    const int32_t v = (int32_t)val[f];
    if (v >= 0) {
      L.start = coord;
      L.end = coord + (uint64_t)v;
      L.strand = 1;
    } else {
      const uint64_t m = (uint64_t)(-(int64_t)v);
      L.end = coord + 1;
      L.start = L.end >= m ? L.end - m : 0;
      L.strand = 2;
    }
  }
  return L;
}

__device__ __forceinline__ int name_len(const uint8_t* nm, int width) {
  int l = 0;
  while (l < width && nm[l] != 0) ++l;
  return l;
}

__global__ void fmt_len_kernel(const int64_t* __restrict__ cell_ptr, int64_t n_cells, const uint32_t* __restrict__ pos,
                               const uint32_t* __restrict__ val, int paired, const uint8_t* __restrict__ chroms,
                               const uint8_t* __restrict__ names, int width, const int64_t* __restrict__ order,
                               int64_t n, int64_t* __restrict__ line_end) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  if (reinterpret_cast<const TableHeader*>(chroms)->n == 0) {
    line_end[k] = 0;
    return;
  }
  const int64_t f = order ? order[k] : k;
  const FmtLine L = fmt_line(f, cell_ptr, n_cells, pos, val, paired, chroms);
  const int64_t len = table_entry(chroms, L.chrom).name_len + 1 + dec_digits(L.start) + 1 + dec_digits(L.end) + 1 +
                      name_len(names + L.row * (int64_t)width, width) + 2 + (L.strand ? 2 : 0) + 1;
  line_end[k] = len;
}

__global__ void fmt_write_kernel(const int64_t* __restrict__ cell_ptr, int64_t n_cells,
                                 const uint32_t* __restrict__ pos, const uint32_t* __restrict__ val, int paired,
                                 const uint8_t* __restrict__ chroms, const uint8_t* __restrict__ names, int width,
                                 const int64_t* __restrict__ order, int64_t n, const int64_t* __restrict__ line_end,
                                 uint8_t* __restrict__ text) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const TableHeader* H = reinterpret_cast<const TableHeader*>(chroms);
  if (H->n == 0) return;
  const int64_t f = order ? order[k] : k;
  const FmtLine L = fmt_line(f, cell_ptr, n_cells, pos, val, paired, chroms);
  const int64_t begin = k == 0 ? 0 : line_end[k - 1];
  const TableEntry& ce = table_entry(chroms, L.chrom);
  const uint8_t* nm = names + L.row * (int64_t)width;
  const int nl = name_len(nm, width);
  const int64_t len = ce.name_len + 1 + dec_digits(L.start) + 1 + dec_digits(L.end) + 1 + nl + 2 +
                      (L.strand ? 2 : 0) + 1;
  if (begin + len != line_end[k]) return;  // line ends from another call: write nothing
  uint8_t* o = text + begin;
  const uint8_t* cn = reinterpret_cast<const uint8_t*>(
                          reinterpret_cast<const TableEntry*>(chroms + sizeof(TableHeader) + H->cap * sizeof(TableSlot)) +
                          H->n) +
                      ce.name_off;
  for (uint32_t q = 0; q < ce.name_len; ++q) *o++ = cn[q];
  *o++ = '\t';
  int d = dec_digits(L.start);
  put_dec(o, L.start, d);
  o += d;
  *o++ = '\t';
  d = dec_digits(L.end);
  put_dec(o, L.end, d);
  o += d;
  *o++ = '\t';
  for (int q = 0; q < nl; ++q) *o++ = nm[q];
  *o++ = '\t';
  *o++ = '1';
  if (L.strand) {
    *o++ = '\t';
    *o++ = L.strand == 1 ? '+' : '-';
  }
  *o++ = '\n';
}

// ---------------------------------------------------------------------------
// workspace layout
// ---------------------------------------------------------------------------

struct Layout {
  int64_t blk, scan, line_start, pos, size, cnt, flags, bc, bch, kept, permA, permB, keyA, keyB, run,
      gstart, gline, gtot, gmito, guniq, gbad, wl, ordA, ordB, gkA, gkB, kr, rowid, rowgroup, rowlen, counters, plan, tmp,
      total;
  size_t tmp_bytes;
};

inline int64_t align256(int64_t x) { return (x + 255) & ~(int64_t)255; }

Layout make_layout(int64_t n_bytes, int64_t L) {
  Layout o{};
  const int64_t nb = ceil_div(n_bytes > 0 ? n_bytes : 1, kByteBlock);
  const int64_t lb = ceil_div(L > 0 ? L : 1, kLineBlock);
  const int64_t Lc = L > 0 ? L : 1;
  int64_t p = 0;
  auto take = [&](int64_t bytes) {
    const int64_t at = p;
    p += align256(bytes);
    return at;
  };
  o.blk = take(8 * (nb > lb ? nb : lb));
  int64_t sw = snapgpu_scan_workspace_bytes(nb);
  const int64_t sw2 = snapgpu_scan_workspace_bytes(Lc + 1);
  if (sw2 > sw) sw = sw2;
  o.scan = take(sw);
  o.line_start = take(8 * (Lc + 1));
  o.pos = take(4 * Lc);
  o.size = take(4 * Lc);
  o.cnt = take(4 * Lc);
  o.flags = take(Lc);
  o.bc = take(8 * Lc);
  o.bch = take(8 * Lc);
  o.kept = take(4 * Lc);
  o.permA = take(4 * Lc);
  o.permB = take(4 * Lc);
  o.keyA = take(8 * Lc);
  o.keyB = take(8 * Lc);
  o.run = take(8 * Lc);
  o.gstart = take(8 * Lc);
  o.gline = take(4 * Lc);
  o.gtot = take(8 * Lc);
  o.gmito = take(8 * Lc);
  o.guniq = take(8 * Lc);
  o.gbad = take(4 * Lc);
  o.wl = take(Lc);
  o.ordA = take(4 * Lc);
  o.ordB = take(4 * Lc);
  o.gkA = take(8 * Lc);
  o.gkB = take(8 * Lc);
  o.kr = take(8 * Lc);
  o.rowid = take(8 * Lc);
  o.rowgroup = take(4 * Lc);
  o.rowlen = take(8 * Lc);
  o.counters = take(sizeof(Counters));
  o.plan = take(sizeof(SortPlan));
  size_t tmp = 0;
  hipcub::DoubleBuffer<uint64_t> kb(nullptr, nullptr);
  hipcub::DoubleBuffer<uint32_t> vb(nullptr, nullptr);
  (void)hipcub::DeviceRadixSort::SortPairs(nullptr, tmp, kb, vb, (int)(Lc < INT32_MAX ? Lc : INT32_MAX), 0, 64);
  size_t tmp2 = 0;
  (void)hipcub::DeviceRadixSort::SortKeys(nullptr, tmp2, kb, (int)(Lc < INT32_MAX ? Lc : INT32_MAX), 0, 64);
  if (tmp2 > tmp) tmp = tmp2;
  o.tmp_bytes = tmp;
  o.tmp = take((int64_t)tmp);
  o.total = p + 256;
  return o;
}

template <typename T>
inline T* at(void* ws, int64_t off) {
  char* base = (char*)(((uintptr_t)ws + 255) & ~(uintptr_t)255);
  return reinterpret_cast<T*>(base + off);
}

inline int grid(int64_t n, int t = kThreads) { return (int)ceil_div(n > 0 ? n : 1, t); }

const char* error_text(uint32_t code) {
  switch (code) {
    case E_START_MISSING: return "missing start position";
    case E_END_MISSING: return "missing end position";
    case E_BARCODE_MISSING: return "missing name (barcode)";
    case E_START_BAD: return "invalid start position";
    case E_END_BAD: return "invalid end position";
    case E_COUNT_BAD: return "invalid count (score) field";
    case E_STRAND_BAD: return "invalid strand";
    case E_BARCODE_NONE: return "the barcode field is '.'";
    case E_END_BEFORE_START: return "end position before start position";
    case E_BARCODE_LONG: return "barcode longer than 255 bytes";
    case E_REVERSE_PAIRED: return "a '-' strand record in a paired-end file: cannot convert its negative size to u32";
    case E_SIZE_I32: return "fragment size does not fit i32";
    case E_RANGE: return "position outside its chromosome";
    case E_SIZE_U32: return "fragment size does not fit u32";
    default: return "invalid record";
  }
}

int data_error(unsigned long long word) {
  const uint64_t line = word >> 8;
  set_error("line " + std::to_string(line + 1) + ": " + error_text((uint32_t)(word & 255)));
  return SNAPGPU_ERR_DATA;
}

uint64_t host_hash(const char* s, size_t len) {
  uint64_t h = hash_start((uint32_t)len);
  for (size_t k = 0; k < len; k += 8) {
    uint64_t w = 0;
    memcpy(&w, s + k, len - k < 8 ? len - k : 8);
    h = hash_step(h, w);
  }
  return hash_end(h);
}

}  // namespace frag
}  // namespace snapgpu

using namespace snapgpu;
using namespace snapgpu::frag;

extern "C" {

int64_t snapgpu_frag_table_bytes(const char* const* names, int32_t n) {
  if (n < 0 || (n > 0 && names == nullptr)) return -1;
  uint32_t cap = 16;
  while (cap < 2u * (uint32_t)n) cap <<= 1;
  int64_t bytes = (int64_t)sizeof(TableHeader) + (int64_t)cap * sizeof(TableSlot) + (int64_t)n * sizeof(TableEntry);
  for (int32_t k = 0; k < n; ++k) bytes += (int64_t)strlen(names[k]);
  return bytes + kNamePad;
}

int snapgpu_frag_table_pack(const char* const* names, const uint64_t* lengths, const uint8_t* mito, int32_t n,
                            int32_t genome, void* out, int64_t out_bytes) {
  clear_error();
  SG_ARG(n >= 0 && n < (1 << 24), "table size out of range");
  SG_ARG(n == 0 || names != nullptr, "null names");
  SG_ARG(!genome || n == 0 || lengths != nullptr, "null lengths");
  const int64_t need = snapgpu_frag_table_bytes(names, n);
  SG_ARG(out != nullptr && out_bytes >= need, "output buffer too small");
  uint32_t cap = 16;
  while (cap < 2u * (uint32_t)n) cap <<= 1;
  uint8_t* o = static_cast<uint8_t*>(out);
  memset(o, 0, (size_t)need);
  TableHeader* H = reinterpret_cast<TableHeader*>(o);
  TableSlot* S = reinterpret_cast<TableSlot*>(o + sizeof(TableHeader));
  TableEntry* E = reinterpret_cast<TableEntry*>(S + cap);
  char* blob = reinterpret_cast<char*>(E + n);
  for (uint32_t k = 0; k < cap; ++k) S[k].idx = -1;
  uint64_t base = 0, name_off = 0;
  for (int32_t k = 0; k < n; ++k) {
    const size_t len = strlen(names[k]);
    SG_ARG(len < (1u << 30), "name too long");
    E[k].base = base;
    E[k].length = genome ? lengths[k] : 0;
    E[k].name_off = (uint32_t)name_off;
    E[k].name_len = (uint32_t)len;
    E[k].flags = (mito && mito[k]) ? 1u : 0u;
    memcpy(blob + name_off, names[k], len);
    name_off += len;
    if (genome) {
      base += lengths[k];
      SG_ARG(base <= 0xFFFFFFFFull, "genome longer than 2^32 - 1 bases: positions are stored as uint32");
    }
    const uint64_t h = host_hash(names[k], len);
    uint32_t i = (uint32_t)h & (cap - 1);
    while (S[i].idx >= 0) {
      const TableEntry& e = E[S[i].idx];
      SG_ARG(!(S[i].hash == h && e.name_len == len && memcmp(blob + e.name_off, names[k], len) == 0),
             std::string("duplicate name: ") + names[k]);
      i = (i + 1) & (cap - 1);
    }
    S[i].hash = h;
    S[i].idx = k;
  }
  H->n = (uint32_t)n;
  H->cap = cap;
  H->total = base;
  return SNAPGPU_OK;
}

int64_t snapgpu_frag_count_workspace_bytes(int64_t n_bytes) {
  const int64_t nb = ceil_div(n_bytes > 0 ? n_bytes : 1, kByteBlock);
  return align256(8 * nb) + snapgpu_scan_workspace_bytes(nb) + 512;
}

int snapgpu_frag_count_lines(const uint8_t* d_text, int64_t n_bytes, void* d_ws, int64_t ws_bytes,
                             int64_t* h_n_lines, void* stream) {
  clear_error();
  SG_ARG(n_bytes >= 0 && h_n_lines != nullptr, "bad arguments");
  SG_ARG(n_bytes == 0 || ((uintptr_t)d_text & 15) == 0, "text must be 16-byte aligned");
  SG_ARG(ws_bytes >= snapgpu_frag_count_workspace_bytes(n_bytes), "workspace too small");
  *h_n_lines = 0;
  if (n_bytes == 0) return SNAPGPU_OK;
  hipStream_t st = as_stream(stream);
  const int64_t nb = ceil_div(n_bytes, kByteBlock);
  int64_t* blk = at<int64_t>(d_ws, 0);
  void* sws = at<char>(d_ws, align256(8 * nb));
  nl_count_kernel<<<(unsigned)nb, kThreads, 0, st>>>(d_text, n_bytes, blk);
  SG_LAUNCH_CHECK();
  int rc = snapgpu_scan_inclusive_i64(blk, nb, sws, snapgpu_scan_workspace_bytes(nb), stream);
  if (rc) return rc;
  int64_t n_nl = 0;
  uint8_t last = 0;
  SG_HIP(hipMemcpyAsync(&n_nl, blk + nb - 1, 8, hipMemcpyDeviceToHost, st));
  SG_HIP(hipMemcpyAsync(&last, d_text + n_bytes - 1, 1, hipMemcpyDeviceToHost, st));
  SG_HIP(hipStreamSynchronize(st));
  *h_n_lines = n_nl + (last != '\n' ? 1 : 0);
  return SNAPGPU_OK;
}

int64_t snapgpu_frag_workspace_bytes(int64_t n_bytes, int64_t n_lines) {
  if (n_bytes < 0 || n_lines < 0) return -1;
  return make_layout(n_bytes, n_lines).total;
}

int snapgpu_frag_index(const uint8_t* d_text, int64_t n_bytes, int64_t n_lines, const void* d_chroms,
                       const void* d_whitelist, const snapgpu_frag_options* opt, void* d_ws, int64_t ws_bytes,
                       snapgpu_frag_summary* h_sum, void* stream) {
  return snapgpu_frag_index_counted(d_text, n_bytes, n_lines, nullptr, 0, d_chroms, d_whitelist, opt, d_ws, ws_bytes,
                                    h_sum, stream);
}

int snapgpu_frag_index_counted(const uint8_t* d_text, int64_t n_bytes, int64_t n_lines, const void* d_count_ws,
                               int64_t count_ws_bytes, const void* d_chroms, const void* d_whitelist,
                               const snapgpu_frag_options* opt, void* d_ws, int64_t ws_bytes,
                               snapgpu_frag_summary* h_sum, void* stream) {
  clear_error();
  SG_ARG(d_count_ws == nullptr || count_ws_bytes >= snapgpu_frag_count_workspace_bytes(n_bytes),
         "count workspace too small");
  SG_ARG(n_bytes >= 0 && n_lines >= 0 && opt != nullptr && h_sum != nullptr && d_chroms != nullptr,
         "bad arguments");
  SG_ARG(n_bytes == 0 || ((uintptr_t)d_text & 15) == 0, "text must be 16-byte aligned");
  SG_ARG(n_lines <= n_bytes, "more lines than bytes");
  SG_ARG(n_lines < (int64_t)INT32_MAX, "at most 2^31 - 2 lines per call");
  const Layout Lo = make_layout(n_bytes, n_lines);
  SG_ARG(ws_bytes >= Lo.total, "workspace too small");
  *h_sum = snapgpu_frag_summary{};
  h_sum->n_lines = n_lines;
  h_sum->paired = 0;
  if (n_lines == 0) return SNAPGPU_OK;
  hipStream_t st = as_stream(stream);
  void* w = d_ws;
  int64_t* blk = at<int64_t>(w, Lo.blk);
  void* sws = at<char>(w, Lo.scan);
  const int64_t sws_bytes = Lo.line_start - Lo.scan;
  int64_t* line_start = at<int64_t>(w, Lo.line_start);
  Counters* C = at<Counters>(w, Lo.counters);
  const uint8_t* chroms = static_cast<const uint8_t*>(d_chroms);

  // 1. line starts (the sentinel after a last line without '\n' is n_bytes + 1)
  const int64_t nb = ceil_div(n_bytes, kByteBlock);
  int rc = SNAPGPU_OK;
  const int64_t* nl = at<int64_t>(const_cast<void*>(d_count_ws), 0);  // the counts' scan
  if (d_count_ws == nullptr) {
    nl_count_kernel<<<(unsigned)nb, kThreads, 0, st>>>(d_text, n_bytes, blk);
    SG_LAUNCH_CHECK();
    rc = snapgpu_scan_inclusive_i64(blk, nb, sws, sws_bytes, stream);
    if (rc) return rc;
    nl = blk;
  }
  Counters c0{};
  c0.err = ~0ull;
  c0.first = ~0ull;
  c0.bad = ~0ull;
  c0.dup = ~0ull;
  SG_HIP(hipMemcpyAsync(C, &c0, sizeof(Counters), hipMemcpyHostToDevice, st));
  nl_index_kernel<<<(unsigned)nb, kThreads, 0, st>>>(d_text, n_bytes, nl, n_lines, line_start, C);
  SG_LAUNCH_CHECK();
  // nothing reads line_start before the host knows that it is whole
  int64_t n_nl = 0;
  uint8_t last = 0;
  unsigned int recount = 0;
  SG_HIP(hipMemcpyAsync(&recount, &C->recount, 4, hipMemcpyDeviceToHost, st));
  SG_HIP(hipMemcpyAsync(&n_nl, nl + nb - 1, 8, hipMemcpyDeviceToHost, st));
  SG_HIP(hipMemcpyAsync(&last, d_text + n_bytes - 1, 1, hipMemcpyDeviceToHost, st));
  SG_HIP(hipStreamSynchronize(st));
  SG_ARG(n_lines == n_nl + (last != '\n' ? 1 : 0), "n_lines does not match the text");
  SG_ARG(recount == 0, "the count workspace is not this text's");
  const int64_t sentinel = n_bytes + 1;  // end of a last line without '\n'
  if (last != '\n') SG_HIP(hipMemcpyAsync(line_start + n_lines, &sentinel, 8, hipMemcpyHostToDevice, st));

  // 2. parse
  ParseOut po{at<uint32_t>(w, Lo.pos), at<uint32_t>(w, Lo.size), at<uint32_t>(w, Lo.cnt), at<uint8_t>(w, Lo.flags),
              at<uint64_t>(w, Lo.bc), opt->sorted_by_barcode ? nullptr : at<uint64_t>(w, Lo.bch)};
  const int64_t lb = ceil_div(n_lines, kLineBlock);
  const bool sorted = opt->sorted_by_barcode != 0;
  uint8_t* same = sorted ? at<uint8_t>(w, Lo.wl) : nullptr;  // wl is written after the runs are known
  parse_kernel<<<(unsigned)lb, kThreads, 0, st>>>(d_text, n_bytes, line_start, n_lines, chroms, opt->shift_left,
                                                  opt->shift_right, po, C, blk, same);
  SG_LAUNCH_CHECK();

  // 3. compaction
  rc = snapgpu_scan_inclusive_i64(blk, lb, sws, sws_bytes, stream);
  if (rc) return rc;
  uint32_t* kept = at<uint32_t>(w, Lo.kept);
  keep_write_kernel<<<(unsigned)lb, kThreads, 0, st>>>(po.flags, n_lines, blk, kept);
  SG_LAUNCH_CHECK();
  Counters ch{};
  TableHeader th{};
  int64_t K = 0;
  SG_HIP(hipMemcpyAsync(&ch, C, sizeof(Counters), hipMemcpyDeviceToHost, st));
  SG_HIP(hipMemcpyAsync(&K, blk + lb - 1, 8, hipMemcpyDeviceToHost, st));
  SG_HIP(hipMemcpyAsync(&th, d_chroms, sizeof(TableHeader), hipMemcpyDeviceToHost, st));
  SG_HIP(hipStreamSynchronize(st));
  if (ch.err != ~0ull) return data_error(ch.err);
  h_sum->n_records = (int64_t)ch.n_rec;
  h_sum->n_kept = K;
  h_sum->name_width = (int32_t)ch.max_bc;
  // paired-end unless the first record carries a strand (import.rs:46-55);
  // for unsorted input the first record is that of the smallest barcode, so
  // a file mixing both kinds is rejected there
  int paired = 0;
  if (ch.n_rec > 0) {
    if (opt->sorted_by_barcode) {
      paired = (ch.first & 1) ? 0 : 1;
    } else {
      if (ch.n_strand != 0 && ch.n_strand != ch.n_rec) {
        set_error("records with and without a strand field in one unsorted file");
        return SNAPGPU_ERR_DATA;
      }
      paired = ch.n_strand == 0 ? 1 : 0;
    }
  }
  h_sum->paired = paired;
  if (K == 0) return SNAPGPU_OK;

  // 4. groups in file order (run[v] = group + 1)
  uint32_t* permA = at<uint32_t>(w, Lo.permA);
  uint32_t* permB = at<uint32_t>(w, Lo.permB);
  uint64_t* keyA = at<uint64_t>(w, Lo.keyA);
  uint64_t* keyB = at<uint64_t>(w, Lo.keyB);
  void* tmp = at<char>(w, Lo.tmp);
  size_t tmp_bytes = Lo.tmp_bytes;
  int64_t* run = at<int64_t>(w, Lo.run);
  int64_t* gstart = at<int64_t>(w, Lo.gstart);
  uint32_t* gline = at<uint32_t>(w, Lo.gline);
  auto* gtot = at<unsigned long long>(w, Lo.gtot);
  auto* gmito = at<unsigned long long>(w, Lo.gmito);
  auto* guniq = at<unsigned long long>(w, Lo.guniq);
  auto* gbad = at<unsigned int>(w, Lo.gbad);
  // key widths: positions below the genome length, values up to the largest size
  auto bits_of = [](uint64_t x) {
    int b = 1;
    while (b < 64 && (x >> b) != 0) ++b;
    return b;
  };
  SortPlan plan{};
  plan.total = th.total;
  plan.max_size = ch.max_size;
  plan.paired = paired;
  plan.vb = bits_of(paired ? (uint64_t)ch.max_size : 2ull * ch.max_size);
  const int pos_bits = bits_of(th.total);
  SG_ARG(pos_bits + plan.vb <= 64, "position and value keys exceed 64 bits");
  int64_t G = 0;
  if (sorted) {
    run_bound_kernel<<<grid(K), kThreads, 0, st>>>(d_text, n_bytes, kept, po.bc, same, K, run);
    SG_LAUNCH_CHECK();
    rc = snapgpu_scan_inclusive_i64(run, K, sws, sws_bytes, stream);
    if (rc) return rc;
    SG_HIP(hipMemcpyAsync(&G, run + K - 1, 8, hipMemcpyDeviceToHost, st));
    SG_HIP(hipStreamSynchronize(st));
  } else {
    // the table takes gkA and gkB, which follow each other; its representatives,
    // numbers and barcodes arrays that are written after it has been read
    auto* slots = at<unsigned long long>(w, Lo.gkA);
    uint32_t* rep = at<uint32_t>(w, Lo.kr);
    uint32_t* slot = at<uint32_t>(w, Lo.ordA);
    uint32_t* id = at<uint32_t>(w, Lo.rowid);
    uint64_t* gbc = at<uint64_t>(w, Lo.gstart);
    SG_HIP(hipMemsetAsync(slots, 0xFF, 16 * K, st));
    group_slot_kernel<<<grid(K), kThreads, 0, st>>>(kept, po.bch, K, slots, rep, slot);
    SG_LAUNCH_CHECK();
    group_number_kernel<<<grid(2 * K), kThreads, 0, st>>>(slots, rep, 2 * K, kept, po.bc, id, gline, gbc, C);
    SG_LAUNCH_CHECK();
    group_of_kernel<<<grid(K), kThreads, 0, st>>>(d_text, n_bytes, kept, po.bc, slot, id, gbc, K, run, C);
    SG_LAUNCH_CHECK();
    SG_HIP(hipMemcpyAsync(&ch, C, sizeof(Counters), hipMemcpyDeviceToHost, st));
    SG_HIP(hipStreamSynchronize(st));
    if (ch.collision) {
      set_error("two different barcodes share a 64-bit hash; cannot group this unsorted file");
      return SNAPGPU_ERR_CAPACITY;
    }
    G = (int64_t)ch.n_groups;
  }
  h_sum->n_groups = G;

  // 5. sort, and 6. group sums. One sort where the key's bits suffice: 55 million
  // records of 8,000 barcodes take 2.3 ms of sorting and 0.95 ms of key, sums and fill
  // kernels; two sorts through a permutation and its gathers 3.8 and 2.4 ms. (20.5
  // million unsorted records: 1.4 and 0.3 ms; with a sort of 64-bit hashes 2.6 and 5.9.)
  const int gbits = G > 1 ? bits_of((uint64_t)(G - 1)) : 0;
  plan.mb = sorted ? 0 : 1;
  plan.pv = pos_bits + plan.vb + plan.mb;
  plan.one = plan.pv + gbits <= 64 ? 1 : 0;
  if (!plan.one) plan.mb = 0, plan.pv = pos_bits + plan.vb;
  SG_HIP(hipMemsetAsync(gtot, 0, 8 * G, st));
  SG_HIP(hipMemsetAsync(gmito, 0, 8 * G, st));
  SG_HIP(hipMemsetAsync(guniq, 0, 8 * G, st));
  SG_HIP(hipMemsetAsync(gbad, 0, 4 * G, st));
  key_kernel<<<grid(K), kThreads, 0, st>>>(kept, po.flags, po.pos, po.size, po.cnt, run, K, plan, keyA,
                                           plan.one && !sorted ? permA : nullptr, gbad);
  SG_LAUNCH_CHECK();
  hipcub::DoubleBuffer<uint64_t> kb(keyA, keyB);
  hipcub::DoubleBuffer<uint32_t> vb(permA, permB);
  const uint32_t* perm = nullptr;
  if (plan.one) {
    if (sorted)
      SG_HIP(hipcub::DeviceRadixSort::SortKeys(tmp, tmp_bytes, kb, (int)K, 0, plan.pv + gbits, st));
    else
      SG_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, tmp_bytes, kb, vb, (int)K, 0, plan.pv + gbits, st));
    plan.alt = kb.Current() != keyA;
  } else {
    iota_kernel<<<grid(K), kThreads, 0, st>>>(permA, K);
    SG_LAUNCH_CHECK();
    SG_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, tmp_bytes, kb, vb, (int)K, 0, plan.pv, st));
    group_key_kernel<<<grid(K), kThreads, 0, st>>>(vb.Current(), run, K, kb.Current());
    SG_LAUNCH_CHECK();
    SG_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, tmp_bytes, kb, vb, (int)K, 0, bits_of((uint64_t)G), st));
    if (vb.Current() != permA) SG_HIP(hipMemcpyAsync(permA, vb.Current(), 4 * K, hipMemcpyDeviceToDevice, st));
    perm = permA;
  }
  SG_HIP(hipMemcpyAsync(at<SortPlan>(w, Lo.plan), &plan, sizeof(SortPlan), hipMemcpyHostToDevice, st));
  if (plan.one && !sorted)
    key_stats_kernel<<<grid(K, kSumBlockRecords), kThreads, 0, st>>>(kb.Current(), vb.Current(), K, plan, gstart, gtot, gmito, guniq);
  else
    group_stats_kernel<<<grid(K, kSumBlockRecords), kThreads, 0, st>>>(sorted ? nullptr : perm, kept, po.flags, po.cnt, run, K, gstart,
                                                     gline, gtot, gmito, guniq);
  SG_LAUNCH_CHECK();
  uint8_t* wl = at<uint8_t>(w, Lo.wl);
  whitelist_kernel<<<grid(G), kThreads, 0, st>>>(d_text, n_bytes, gline, po.bc, G,
                                                 static_cast<const uint8_t*>(d_whitelist), wl);
  SG_LAUNCH_CHECK();
  uint32_t* ordA = at<uint32_t>(w, Lo.ordA);
  uint32_t* ordB = at<uint32_t>(w, Lo.ordB);
  uint64_t* gkA = at<uint64_t>(w, Lo.gkA);
  uint64_t* gkB = at<uint64_t>(w, Lo.gkB);
  if (sorted && G > 1) {
    group_hash_kernel<<<grid(G), kThreads, 0, st>>>(d_text, n_bytes, gline, po.bc, G, gkA, ordA);
    SG_LAUNCH_CHECK();
    hipcub::DoubleBuffer<uint64_t> gk(gkA, gkB);
    hipcub::DoubleBuffer<uint32_t> go(ordA, ordB);
    SG_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, tmp_bytes, gk, go, (int)G, 0, 64, st));
    dup_kernel<<<grid(G), kThreads, 0, st>>>(d_text, n_bytes, gk.Current(), go.Current(), gline, po.bc, wl, G, C);
    SG_LAUNCH_CHECK();
  }
  bad_group_kernel<<<grid(G), kThreads, 0, st>>>(gbad, wl, G, paired, C);
  SG_LAUNCH_CHECK();
  SG_HIP(hipMemcpyAsync(&ch, C, sizeof(Counters), hipMemcpyDeviceToHost, st));
  SG_HIP(hipStreamSynchronize(st));
  if (ch.any_bad) {
    bad_kernel<<<grid(K), kThreads, 0, st>>>(kept, po.flags, run, wl, K, paired, C);
    SG_LAUNCH_CHECK();
    SG_HIP(hipMemcpyAsync(&ch, C, sizeof(Counters), hipMemcpyDeviceToHost, st));
    SG_HIP(hipStreamSynchronize(st));
  }
  if (ch.dup != ~0ull) {
    set_error("a barcode appears in two separate runs: please sort the fragment file by barcodes (group " +
              std::to_string(ch.dup) + ")");
    return SNAPGPU_ERR_DATA;
  }
  if (ch.bad != ~0ull) return data_error(ch.bad);

  // group order: file order (sorted input) or barcode bytes (unsorted input)
  const uint32_t* order = nullptr;
  if (!sorted) {
    length_key_kernel<<<grid(G), kThreads, 0, st>>>(gline, po.bc, G, gkA, ordA);
    SG_LAUNCH_CHECK();
    hipcub::DoubleBuffer<uint64_t> gk(gkA, gkB);
    hipcub::DoubleBuffer<uint32_t> go(ordA, ordB);
    SG_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, tmp_bytes, gk, go, (int)G, 0, 8, st));
    const int words = (int)ceil_div(ch.max_bc > 0 ? ch.max_bc : 1, 8);
    for (int wd = words - 1; wd >= 0; --wd) {
      word_key_kernel<<<grid(G), kThreads, 0, st>>>(d_text, go.Current(), gline, po.bc, G, wd, gk.Current());
      SG_LAUNCH_CHECK();
      SG_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, tmp_bytes, gk, go, (int)G, 0, 64, st));
    }
    if (go.Current() != ordA) SG_HIP(hipMemcpyAsync(ordA, go.Current(), 4 * G, hipMemcpyDeviceToDevice, st));
    order = ordA;
  }
  int64_t* kr = at<int64_t>(w, Lo.kr);
  keep_rank_kernel<<<grid(G), kThreads, 0, st>>>(order, wl, guniq, G, opt->min_num_fragments, kr);
  SG_LAUNCH_CHECK();
  rc = snapgpu_scan_inclusive_i64(kr, G, sws, sws_bytes, stream);
  if (rc) return rc;
  int64_t* rowid = at<int64_t>(w, Lo.rowid);
  uint32_t* rowgroup = at<uint32_t>(w, Lo.rowgroup);
  int64_t* rowlen = at<int64_t>(w, Lo.rowlen);
  rows_kernel<<<grid(G), kThreads, 0, st>>>(order, kr, guniq, gmito, G, rowid, rowgroup, rowlen);
  SG_LAUNCH_CHECK();
  int64_t R = 0;
  SG_HIP(hipMemcpyAsync(&R, kr + G - 1, 8, hipMemcpyDeviceToHost, st));
  SG_HIP(hipStreamSynchronize(st));
  int64_t nnz = 0;
  if (R > 0) {
    rc = snapgpu_scan_inclusive_i64(rowlen, R, sws, sws_bytes, stream);
    if (rc) return rc;
    SG_HIP(hipMemcpyAsync(&nnz, rowlen + R - 1, 8, hipMemcpyDeviceToHost, st));
    SG_HIP(hipStreamSynchronize(st));
  }
  h_sum->n_rows = R;
  h_sum->nnz = nnz;
  return SNAPGPU_OK;
}

int snapgpu_frag_fill(const uint8_t* d_text, int64_t n_bytes, const void* d_ws, int64_t ws_bytes,
                      const snapgpu_frag_summary* h_sum, int64_t* d_cell_ptr, uint32_t* d_pos, uint32_t* d_val,
                      uint64_t* d_qc, uint8_t* d_names, int32_t name_width, void* stream) {
  clear_error();
  SG_ARG(h_sum != nullptr && d_cell_ptr != nullptr, "bad arguments");
  const Layout Lo = make_layout(n_bytes, h_sum->n_lines);
  SG_ARG(ws_bytes >= Lo.total, "workspace too small");
  SG_ARG(d_names == nullptr || name_width >= h_sum->name_width, "name_width below the longest barcode");
  SG_ARG(h_sum->nnz == 0 || (d_pos != nullptr && d_val != nullptr), "null outputs");
  hipStream_t st = as_stream(stream);
  const int64_t R = h_sum->n_rows, K = h_sum->n_kept;
  if (R == 0) {
    const int64_t zero = 0;
    SG_HIP(hipMemcpyAsync(d_cell_ptr, &zero, 8, hipMemcpyHostToDevice, st));
    SG_HIP(hipStreamSynchronize(st));
    return SNAPGPU_OK;
  }
  void* w = const_cast<void*>(d_ws);
  fill_kernel<<<grid(K), kThreads, 0, st>>>(
      at<SortPlan>(w, Lo.plan), at<uint64_t>(w, Lo.keyA), at<uint64_t>(w, Lo.keyB), at<uint32_t>(w, Lo.permA),
      at<uint32_t>(w, Lo.kept), at<uint8_t>(w, Lo.flags), at<uint32_t>(w, Lo.pos), at<uint32_t>(w, Lo.size),
      at<int64_t>(w, Lo.run), at<int64_t>(w, Lo.gstart), at<int64_t>(w, Lo.rowid), at<int64_t>(w, Lo.rowlen), K, d_pos,
      d_val);
  SG_LAUNCH_CHECK();
  rows_out_kernel<<<grid(R), kThreads, 0, st>>>(
      d_text, at<uint32_t>(w, Lo.rowgroup), at<uint32_t>(w, Lo.gline), at<uint64_t>(w, Lo.bc),
      at<int64_t>(w, Lo.rowlen), at<unsigned long long>(w, Lo.guniq), at<unsigned long long>(w, Lo.gtot),
      at<unsigned long long>(w, Lo.gmito), R, d_cell_ptr, reinterpret_cast<unsigned long long*>(d_qc), d_names,
      name_width);
  SG_LAUNCH_CHECK();
  return SNAPGPU_OK;
}

int64_t snapgpu_frag_format_workspace_bytes(int64_t n_fragments) {
  return snapgpu_scan_workspace_bytes(n_fragments > 0 ? n_fragments : 1);
}

int snapgpu_frag_format(const int64_t* d_cell_ptr, int64_t n_cells, const uint32_t* d_pos, const uint32_t* d_val,
                        int64_t n_fragments, int32_t paired, const void* d_chroms, const uint8_t* d_names,
                        int32_t name_width, const int64_t* d_order, int64_t* d_line_end, uint8_t* d_text,
                        int64_t text_bytes, void* d_ws, int64_t ws_bytes, int64_t* h_text_bytes, void* stream) {
  clear_error();
  SG_ARG(n_cells >= 0 && n_fragments >= 0 && d_chroms != nullptr && h_text_bytes != nullptr, "bad arguments");
  SG_ARG(name_width > 0 && d_names != nullptr, "names required");
  SG_ARG(ws_bytes >= snapgpu_frag_format_workspace_bytes(n_fragments), "workspace too small");
  *h_text_bytes = 0;
  if (n_fragments == 0) return SNAPGPU_OK;
  SG_ARG(n_cells > 0 && d_cell_ptr && d_pos && d_val && d_line_end, "null inputs");
  hipStream_t st = as_stream(stream);
  const uint8_t* chroms = static_cast<const uint8_t*>(d_chroms);
  if (d_text == nullptr) {
    fmt_len_kernel<<<grid(n_fragments), kThreads, 0, st>>>(d_cell_ptr, n_cells, d_pos, d_val, paired, chroms,
                                                           d_names, name_width, d_order, n_fragments, d_line_end);
    SG_LAUNCH_CHECK();
    int rc = snapgpu_scan_inclusive_i64(d_line_end, n_fragments, d_ws, ws_bytes, stream);
    if (rc) return rc;
  }
  int64_t total = 0;
  SG_HIP(hipMemcpyAsync(&total, d_line_end + n_fragments - 1, 8, hipMemcpyDeviceToHost, st));
  SG_HIP(hipStreamSynchronize(st));
  *h_text_bytes = total;
  if (d_text != nullptr) {
    SG_ARG(text_bytes >= total, "text buffer too small");
    fmt_write_kernel<<<grid(n_fragments), kThreads, 0, st>>>(d_cell_ptr, n_cells, d_pos, d_val, paired, chroms,
                                                             d_names, name_width, d_order, n_fragments, d_line_end,
                                                             d_text);
    SG_LAUNCH_CHECK();
  }
  return SNAPGPU_OK;
}

}  // extern "C"
