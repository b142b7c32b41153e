// periodic_check.cpp -- test helper, built by tests/test_periodic_host.py with
// g++.  For every axis of 2..9 nodes and ngg 3 and 4, fills the ghost layers
// of both periodic faces the way the reference does, layer after layer from
// whatever the array then holds, and from the node that periodic_source
// (openstc-mixinglayer_amd/csrc/ostc_faces.hpp) names, layers in any order;
// the two must agree and the source must be a node of the block.  The first
// and the last node carry different values, so that one taken for the other
// shows.
#include <cstdio>
#include <vector>

#include "ostc_faces.hpp"

int main() {
  for (int ngg = 3; ngg <= 4; ++ngg)
    for (int m = 2; m <= 9; ++m) {
      std::vector<int> a(m + 2 * ngg, -1), b;
      for (int i = 0; i < m; ++i) a[i + ngg] = i;
      b = a;
      for (int side = -1; side <= 1; side += 2) {
        const int face = side < 0 ? 0 : m - 1, from = side < 0 ? m - 1 : 0;
        for (int g = 1; g <= ngg; ++g) a[face + g * side + ngg] = a[from + g * side + ngg];
        for (int g = ngg; g >= 1; --g) {
          const int src = ostc::periodic_source(m, side, g);
          if (src < 0 || src > m - 1) {
            std::printf("m %d side %d layer %d: source %d is no node of the block\n", m, side, g, src);
            return 1;
          }
          b[face + g * side + ngg] = b[src + ngg];
        }
      }
      if (a != b) {
        std::printf("ngg %d m %d: the ghost layers differ\n", ngg, m);
        return 1;
      }
    }
  std::printf("ok\n");
}
