// CPU check of the reference-order 4-wide records: walking the records collapse4 forms, slots in the order visit_order4
// gives for the ray's octant, meets the leaves of a binary tree in the order of the reference's depth-first traversal
// (near child = children[sign of the split axis], blazert/bvh/accel.h:95-104), for random trees and every octant.
#include <cstdint>
#include <cstdio>
#include <random>
#include <vector>

#include "../../blazert_amd/csrc/engine.h"

namespace {

std::mt19937 rng(5);

uint32_t grow(std::vector<brt_tree_node> &T, int depth) {
  const uint32_t id = (uint32_t)T.size();
  T.push_back(brt_tree_node{});
  std::uniform_real_distribution<double> u(0.0, 1.0);
  for (int k = 0; k < 3; k++) {
    T[id].min[k] = 0.0;
    T[id].max[k] = u(rng);
  }
  if (depth == 0 || u(rng) < 0.2) {
    T[id].leaf = 1;
    return id;
  }
  T[id].axis = rng() % 3u;
  const uint32_t a = grow(T, depth - 1), b = grow(T, depth - 1);
  T[id].children[0] = a;
  T[id].children[1] = b;
  return id;
}

void reference(const std::vector<brt_tree_node> &T, uint32_t v, uint32_t oct, std::vector<uint32_t> &out) {
  if (T[v].leaf) {
    out.push_back(v);
    return;
  }
  const uint32_t near = (oct >> T[v].axis) & 1u;
  reference(T, T[v].children[near], oct, out);
  reference(T, T[v].children[1 - near], oct, out);
}

void wide(const std::vector<brt_tree_node> &T, uint32_t v, uint32_t oct, std::vector<uint32_t> &out) {
  if (T[v].leaf) {
    out.push_back(v);
    return;
  }
  uint32_t slot[4], axis[16] = {}, ord[2];
  const int m = brt::collapse4(T.data(), v, slot, axis);
  brt::visit_order4(axis, m, ord);
  // the masks of octants 4..7 are the complements of those of the opposite octant
  const uint32_t c = (oct & 4u) ? (~oct & 3u) : oct;
  const uint32_t later = ((ord[c >> 1] >> (16 * (c & 1u))) ^ ((oct & 4u) ? 0xffffu : 0u));
  const uint32_t all = (1u << m) - 1u;
  uint32_t place[4];
  for (int s = 0; s < m; s++) {
    const uint32_t after = (later >> (4 * s)) & all & ~(1u << s);
    place[m - 1 - __builtin_popcount(after)] = slot[s];
  }
  for (int s = 0; s < m; s++) wide(T, place[s], oct, out);
}

}  // namespace

int main() {
  for (int trial = 0; trial < 2000; trial++) {
    std::vector<brt_tree_node> T;
    grow(T, 1 + trial % 9);
    for (uint32_t oct = 0; oct < 8; oct++) {
      std::vector<uint32_t> a, b;
      reference(T, 0, oct, a);
      wide(T, 0, oct, b);
      if (a != b) {
        std::printf("trial %d octant %u: orders differ\n", trial, oct);
        return 1;
      }
    }
  }
  std::printf("4-wide records visit the leaves in the reference's order\n");
  return 0;
}
