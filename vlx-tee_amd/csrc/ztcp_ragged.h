// ztcp_ragged.h -- which batches of pages without whole 64-byte units take the
// kernels that keep the payloads in LDS (ztcp_ragged.hip), and how many pages
// a workgroup of theirs holds.  Plain host code.
#pragma once
#include <cstddef>
#include <cstdint>

namespace ztcp {

constexpr int kRaggedMaxPages = 32;                          // two lanes of the hashing wave per page
constexpr size_t kRaggedFixed = 64;                          // LDS bytes of a workgroup beside its pages
constexpr size_t kRaggedRoom = 160 * 1024 - kRaggedFixed;    // ... and what is left for the pages

// LDS words of one page's payload: 64-byte blocks and a pad of 16 bytes, so
// that the hashing lanes' rows start at different banks.
constexpr uint32_t ragged_page_words(uint32_t payload) { return (payload + 63u) / 64u * 16u + 4u; }
// LDS bytes of one page: the payload, for ingress two copies of it and
// `layout_words` words of its own layout.
constexpr size_t ragged_page_bytes(uint32_t payload, bool ingress, int layout_words) {
    return (size_t)ragged_page_words(payload) * (ingress ? 8 : 4) + (ingress ? (size_t)layout_words * 4 : 0);
}

// Pages per workgroup of the LDS kernels, or 0 for the layout-agnostic kernels
// (ztcp_generic.hip).
// The LDS kernels run in rounds of the pages that fit the chip's LDS, `fit` on
// a CU, and a round lasts at least a page's hash chain; the layout-agnostic
// ones hash every page of the batch at once, 64 to a wave, at a higher price
// per byte.  So a page must fit, and where few do, the rounds must be few.
// Measured on 256 CUs (pages, rounds: us of the LDS kernels / of the others;
// the latter also depend on the blobs' stride, hence the spread at the lines):
//   ingress  fit 1: 50 KB  768, 3: 1,251 / 1,510; 1,024, 4: 1,652 / 1,618; 2,000, 8: 3,264 / 2,166
//                   78 KB  900, 4: 2,525 / 3,278; 67 KB  3,000, 12: 6,559 / 3,603
//            fit 2: 32 KB  2,560, 5: 1,391 / 1,512; 3,072, 6: 1,668 / 1,696; 8,000, 16: 4,417 / 3,168
//            fit 3: 24 KB  6,144, 8: 1,748 / 1,896; 8,000, 11: 2,391 / 2,304; 20,000, 27: 5,797 / 4,939
//            fit 4: 19 KB  20,000, 20: 3,866 / 4,152; fit 7: 11 KB  20,000, 12: 1,670 / 3,136
//   egress   fit 1: 119 KB  2,304, 9: 8,655 / 8,844; 2,560, 10: 9,609 / 9,446; 84 KB  4,000, 16: 10,931 / 9,261
//                   158 KB  2,560, 10: 12,755 / 13,345
//            fit 2: 78 KB  40,000, 79: 51,480 / 64,650
inline int ragged_pages(int64_t batch, size_t page_bytes, bool ingress, int cu_count) {
    if (page_bytes > kRaggedRoom || batch > ((int64_t)1 << 30)) return 0;
    const int64_t cus = cu_count > 0 ? cu_count : 1, fit = (int64_t)(kRaggedRoom / page_bytes);
    const int64_t rounds = (batch + cus * fit - 1) / (cus * fit);
    const int64_t most = ingress ? (fit == 1 ? 4 : (fit == 2 ? 6 : (fit == 3 ? 10 : rounds))) : (fit == 1 ? 10 : rounds);
    if (rounds > most) return 0;
    // one page a workgroup until every SIMD of the chip has one to hash, then more
    int64_t n = (batch + 4 * cus - 1) / (4 * cus);
    if (n > kRaggedMaxPages) n = kRaggedMaxPages;
    if (n > fit) n = fit;
    return n < 1 ? 1 : (int)n;
}

}  // namespace ztcp
