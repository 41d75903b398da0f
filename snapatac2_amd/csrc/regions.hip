// Host side of the peak matrix: "chrom:start-end" strings to distinct regions, and
// the region index (regions of each chromosome by start, running maxima of their
// ends) that the peak kernels search (snapgpu_peak_index).
//
// Reference: GenomicRange::from_str of each peak and the index set of
// create_peak_matrix (snapatac2-core/src/feature_count/matrix.rs:113-124). In Python
// the two took eight times as long as the kernels: the peak matrix of 50,000 regions
// and 6,000 cells took 41.6 ms with them and takes 12.2 ms (4.5 ms of it kernels).
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

static uint64_t mix(uint64_t x) {
  x ^= x >> 33;
  x *= 0xff51afd7ed558ccdull;
  x ^= x >> 33;
  x *= 0xc4ceb9fe1a85ec53ull;
  return x ^ (x >> 33);
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
      size_t s = mix((uint64_t)a * 0x9e3779b97f4a7c15ull + mix((uint64_t)b + ((uint64_t)last_id << 40))) & (slots - 1);
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

int snapgpu_region_index(const int32_t* h_chrom, const int64_t* h_start, const int64_t* h_end, int64_t n,
                         int32_t n_chrom, uint64_t* h_starts, uint64_t* h_ends, uint64_t* h_pmax, uint32_t* h_idx,
                         int64_t* h_off) {
  clear_error();
  SG_ARG(n >= 0 && n < (1ll << 32) && n_chrom >= 0 && h_off, "bad arguments");
  SG_ARG(n == 0 || (h_chrom && h_start && h_end && h_starts && h_ends && h_pmax && h_idx), "null pointer");
  try {
    std::fill(h_off, h_off + n_chrom + 1, 0);
    for (int64_t i = 0; i < n; ++i) {
      SG_ARG(h_chrom[i] < n_chrom, "chromosome id out of range");
      if (h_chrom[i] >= 0) ++h_off[h_chrom[i] + 1];
    }
    for (int32_t c = 0; c < n_chrom; ++c) h_off[c + 1] += h_off[c];
    std::vector<int64_t> at(h_off, h_off + n_chrom);
    for (int64_t i = 0; i < n; ++i)
      if (h_chrom[i] >= 0) h_idx[at[h_chrom[i]]++] = (uint32_t)i;
    for (int32_t c = 0; c < n_chrom; ++c) {
      const auto less = [&](uint32_t x, uint32_t y) {
        return h_start[x] != h_start[y] ? h_start[x] < h_start[y] : x < y;
      };
      std::sort(h_idx + h_off[c], h_idx + h_off[c + 1], less);
      uint64_t top = 0;
      for (int64_t k = h_off[c]; k < h_off[c + 1]; ++k) {
        h_starts[k] = (uint64_t)h_start[h_idx[k]];
        h_ends[k] = (uint64_t)h_end[h_idx[k]];
        top = std::max(top, h_ends[k]);
        h_pmax[k] = top;
      }
    }
  } catch (const std::exception& ex) {
    set_error(std::string("region index: ") + ex.what());
    return SNAPGPU_ERR_CAPACITY;
  }
  return SNAPGPU_OK;
}

}  // extern "C"
