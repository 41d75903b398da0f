// Regions of the peak matrix: "chrom:start-end" strings to distinct regions (host),
// and the region index (regions of each chromosome by start, running maxima of their
// ends) that the peak kernels search (snapgpu_peak_index).
//
// Reference: GenomicRange::from_str of each peak and the index set of
// create_peak_matrix (snapatac2-core/src/feature_count/matrix.rs:113-124). In Python
// the two took eight times as long as the kernels: the peak matrix of 50,000 regions
// and 6,000 cells took 41.6 ms with them, 11.8 with both in native code on the host,
// and 9.6 with the index built on the device.
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cstring>
#include <string_view>
#include <unordered_map>
#include <vector>

#include "common.h"

namespace snapgpu {
namespace regions {

// The digits [a, b) as a number: no sign, no leading zero, below 10^18.
static bool number(const char* a, const char* b, int64_t* out) {
  if (b <= a || b - a > 18 || (*a == '0' && b - a > 1)) return false;
  int64_t v = 0;
  for (; a < b; ++a) {
    if (*a < '0' || *a > '9') return false;
    v = v * 10 + (*a - '0');
  }
  *out = v;
  return true;
}

// One region in the form that formats back to itself: printable ASCII without
// blanks, the range after the last colon.
static bool region(std::string_view s, std::string_view* chrom, int64_t* start, int64_t* end) {
  for (char c : s)
    if (c <= ' ' || c > '~') return false;
  const size_t colon = s.rfind(':');
  if (colon == std::string_view::npos) return false;
  const char *a = s.data() + colon + 1, *e = s.data() + s.size();
  const char* dash = static_cast<const char*>(memchr(a, '-', e - a));
  if (!dash || !number(a, dash, start) || !number(dash + 1, e, end)) return false;
  *chrom = s.substr(0, colon);
  return true;
}

// Fibonacci hashing (Knuth, The Art of Computer Programming 6.4): the product with the
// golden ratio's 64-bit fraction, its high half folded onto the low one.
static uint64_t mix(uint64_t x) {
  x *= 0x9e3779b97f4a7c15ull;
  return x ^ (x >> 32);
}

constexpr int kThreads = 256;

__global__ void start_key_kernel(const int64_t* __restrict__ start, int64_t n, uint64_t* __restrict__ key,
                                 uint32_t* __restrict__ idx) {
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  key[i] = (uint64_t)start[i];
  idx[i] = (uint32_t)i;
}

// regions of no chromosome of the genome go last
__global__ void chrom_key_kernel(const int32_t* __restrict__ chrom, const uint32_t* __restrict__ idx, int64_t n,
                                 int32_t n_chrom, uint64_t* __restrict__ key) {
  const int64_t j = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (j >= n) return;
  const int32_t c = chrom[idx[j]];
  key[j] = (uint64_t)(c >= 0 && c < n_chrom ? c : n_chrom);
}

__global__ void region_gather_kernel(const uint32_t* __restrict__ idx, const int64_t* __restrict__ start,
                                     const int64_t* __restrict__ end, const uint64_t* __restrict__ key, int64_t n,
                                     int32_t n_chrom, uint64_t* __restrict__ starts, uint64_t* __restrict__ ends,
                                     uint32_t* __restrict__ out_idx, int64_t* __restrict__ off) {
  const int64_t j = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (j <= n_chrom) {  // first region of chromosome j (n_chrom: the end of the last one)
    int64_t a = 0, b = n;
    while (a < b) {
      const int64_t mid = (a + b) / 2;
      if (key[mid] < (uint64_t)j) a = mid + 1;
      else b = mid;
    }
    off[j] = a;
  }
  if (j >= n) return;
  const uint32_t i = idx[j];
  out_idx[j] = i;
  starts[j] = (uint64_t)start[i];
  ends[j] = (uint64_t)end[i];
}

// Running maximum of each chromosome's ends: a block per chromosome, 256 at a time.
__global__ void __launch_bounds__(kThreads) region_max_kernel(const uint64_t* __restrict__ ends,
                                                              const int64_t* __restrict__ off,
                                                              uint64_t* __restrict__ pmax) {
  __shared__ uint64_t wave_top[kThreads / 64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int64_t lo = off[blockIdx.x], hi = off[blockIdx.x + 1];
  uint64_t top = 0;
  for (int64_t b = lo; b < hi; b += kThreads) {
    const int64_t i = b + threadIdx.x;
    uint64_t v = i < hi ? ends[i] : 0;
    for (int d = 1; d < 64; d <<= 1) {
      const uint64_t o = shfl_u64(v, lane >= d ? lane - d : lane);
      v = o > v ? o : v;
    }
    if (lane == 63) wave_top[wid] = v;
    __syncthreads();
    for (int w = 0; w < wid; ++w) v = wave_top[w] > v ? wave_top[w] : v;
    v = top > v ? top : v;
    if (i < hi) pmax[i] = v;
    for (int w = 0; w < kThreads / 64; ++w) top = wave_top[w] > top ? wave_top[w] : top;
    __syncthreads();
  }
}

static int64_t align256(int64_t x) { return (x + 255) & ~(int64_t)255; }

static size_t sort_bytes(int64_t n) {
  size_t tmp = 0;
  hipcub::DoubleBuffer<uint64_t> kb(nullptr, nullptr);
  hipcub::DoubleBuffer<uint32_t> vb(nullptr, nullptr);
  (void)hipcub::DeviceRadixSort::SortPairs(nullptr, tmp, kb, vb, (int)n, 0, 64);
  return tmp;
}

}  // namespace regions
}  // namespace snapgpu

using namespace snapgpu;
using namespace snapgpu::regions;

extern "C" {

int snapgpu_region_parse(const char* h_text, int64_t n_bytes, int64_t n, const char* const* h_chroms, int32_t n_chrom,
                         int32_t* h_chrom, int64_t* h_start, int64_t* h_end, int64_t* h_first, int64_t* n_distinct,
                         int32_t* plain) {
  clear_error();
  SG_ARG(n >= 0 && n_bytes >= 0 && n_chrom >= 0 && n_distinct && plain, "bad arguments");
  SG_ARG((n_bytes == 0 || h_text) && (n_chrom == 0 || h_chroms), "null pointer");
  SG_ARG(n == 0 || (h_chrom && h_start && h_end && h_first), "null output");
  *n_distinct = 0;
  *plain = 0;
  try {
    std::unordered_map<std::string_view, int32_t> ids;  // chromosomes outside the genome get ids past n_chrom
    for (int32_t c = 0; c < n_chrom; ++c) ids.emplace(h_chroms[c], c);
    int32_t next_id = n_chrom;
    size_t slots = 16;
    while (slots < (size_t)n * 2) slots *= 2;
    std::vector<int64_t> table(slots, -1);
    std::vector<int32_t> id(n);
    const char *p = h_text, *stop = h_text + n_bytes;
    std::string_view last;
    int32_t last_id = -1;
    int64_t kept = 0;
    for (int64_t i = 0; i < n; ++i) {
      if (i > 0) {
        if (p >= stop || *p != '\n') return SNAPGPU_OK;
        ++p;
      }
      const char* nl = p < stop ? static_cast<const char*>(memchr(p, '\n', stop - p)) : nullptr;
      const char* e = nl ? nl : stop;
      std::string_view chrom;
      int64_t a, b;
      if (!region(std::string_view(p, e - p), &chrom, &a, &b)) return SNAPGPU_OK;
      p = e;
      if (last_id < 0 || chrom != last) {
        last = chrom;
        const auto at = ids.emplace(chrom, next_id);
        next_id += at.second;
        last_id = at.first->second;
      }
      size_t s = mix((uint64_t)a + mix((uint64_t)b + ((uint64_t)last_id << 40))) & (slots - 1);
      bool seen = false;
      for (; table[s] >= 0; s = (s + 1) & (slots - 1)) {
        const int64_t k = table[s];
        if (h_start[k] == a && h_end[k] == b && id[k] == last_id) {
          seen = true;
          break;
        }
      }
      if (seen) continue;
      table[s] = kept;
      h_start[kept] = a;
      h_end[kept] = b;
      id[kept] = last_id;
      h_chrom[kept] = last_id < n_chrom ? last_id : -1;
      h_first[kept] = i;
      ++kept;
    }
    if (p != stop) return SNAPGPU_OK;  // more lines than items: an item holds a line break
    *n_distinct = kept;
    *plain = 1;
  } catch (const std::exception& ex) {
    set_error(std::string("region parse: ") + ex.what());
    return SNAPGPU_ERR_CAPACITY;
  }
  return SNAPGPU_OK;
}

int64_t snapgpu_region_index_workspace_bytes(int64_t n) {
  if (n < 0 || n >= INT32_MAX) return -1;
  return 2 * (align256(8 * n) + align256(4 * n)) + (int64_t)sort_bytes(std::max<int64_t>(n, 1)) + 512;
}

int snapgpu_region_index(const int32_t* d_chrom, const int64_t* d_start, const int64_t* d_end, int64_t n,
                         int32_t n_chrom, int64_t max_start, uint64_t* d_starts, uint64_t* d_ends, uint64_t* d_pmax,
                         uint32_t* d_idx, int64_t* d_off, void* d_ws, int64_t ws_bytes, void* stream) {
  clear_error();
  SG_ARG(n >= 0 && n < INT32_MAX && n_chrom >= 0 && max_start >= 0 && d_off, "bad arguments");
  SG_ARG(n == 0 || (d_chrom && d_start && d_end && d_starts && d_ends && d_pmax && d_idx && d_ws), "null pointer");
  SG_ARG(n == 0 || ws_bytes >= snapgpu_region_index_workspace_bytes(n), "workspace too small");
  hipStream_t st = as_stream(stream);
  const unsigned g = (unsigned)ceil_div(std::max<int64_t>(n, (int64_t)n_chrom + 1), kThreads);
  char* p = (char*)(((uintptr_t)d_ws + 255) & ~(uintptr_t)255);
  const auto take = [&](int64_t bytes) {
    char* at = p;
    p += align256(bytes);
    return at;
  };
  uint64_t* key = reinterpret_cast<uint64_t*>(n ? take(8 * n) : nullptr);
  uint64_t* key2 = reinterpret_cast<uint64_t*>(n ? take(8 * n) : nullptr);
  uint32_t* idx = reinterpret_cast<uint32_t*>(n ? take(4 * n) : nullptr);
  uint32_t* idx2 = reinterpret_cast<uint32_t*>(n ? take(4 * n) : nullptr);
  hipcub::DoubleBuffer<uint64_t> kb(key, key2);
  hipcub::DoubleBuffer<uint32_t> vb(idx, idx2);
  if (n > 0) {
    const auto bits_of = [](uint64_t x) {
      int b = 1;
      while (b < 64 && (x >> b) != 0) ++b;
      return b;
    };
    size_t tmp = sort_bytes(n);
    start_key_kernel<<<g, kThreads, 0, st>>>(d_start, n, key, idx);
    SG_LAUNCH_CHECK();
    SG_HIP(hipcub::DeviceRadixSort::SortPairs(p, tmp, kb, vb, (int)n, 0, bits_of((uint64_t)max_start), st));
    chrom_key_kernel<<<g, kThreads, 0, st>>>(d_chrom, vb.Current(), n, n_chrom, kb.Current());
    SG_LAUNCH_CHECK();
    SG_HIP(hipcub::DeviceRadixSort::SortPairs(p, tmp, kb, vb, (int)n, 0, bits_of((uint64_t)n_chrom), st));
  }
  region_gather_kernel<<<g, kThreads, 0, st>>>(vb.Current(), d_start, d_end, kb.Current(), n, n_chrom, d_starts,
                                               d_ends, d_idx, d_off);
  if (n > 0 && n_chrom > 0) region_max_kernel<<<(unsigned)n_chrom, kThreads, 0, st>>>(d_ends, d_off, d_pmax);
  SG_LAUNCH_CHECK();
  return SNAPGPU_OK;
}

}  // extern "C"
