// CPU check of leaf_record: for leaves of every size and every candidate mask that a group of two to eight pre-tested
// primitives can leave, the record read lies in the leaf, and with candidates it is the lowest one's.
#include <cstdint>
#include <cstdio>

#include "../../blazert_amd/csrc/engine.h"

int main() {
  for (uint32_t begin : {0u, 1u, 327676u}) {
    for (uint32_t count = 1; count <= 64; count++) {
      for (uint32_t at = 0; at < count; at += 2) {  // where the group starts
        const uint32_t left = count - at;
        for (uint32_t cand = 0; cand < 256u && (left >= 8u || cand < (1u << left)); cand++) {
          const uint32_t p = brt::leaf_record(begin + at, cand);
          uint32_t want = begin + at;
          for (uint32_t k = 0; k < 8; k++)
            if ((cand >> k) & 1u) {
              want = begin + at + k;
              break;
            }
          if (p != want || p >= begin + count) {
            std::printf("leaf [%u, %u), group at %u, candidates %x: record %u\n", begin, begin + count, begin + at, cand, p);
            return 1;
          }
        }
      }
    }
  }
  std::printf("every record read lies in its leaf\n");
  return 0;
}
