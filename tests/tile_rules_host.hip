// Host driver for tests/test_tile_rules.py: the kernels' tile rules
// (gki_common.cuh) on the CPU.
//
// stdin lines: n_q n_kv causal sink window q_lo q_hi k0 n_k
// stdout: tile_unseen, per line.
#include <cstdio>

#include "gki_common.cuh"

int main() {
  gki::Geom g{};
  int q_lo, q_hi, k0, n_k;
  while (std::scanf("%d %d %d %d %d %d %d %d %d", &g.n_q, &g.n_kv, &g.causal, &g.sink, &g.window, &q_lo, &q_hi,
                    &k0, &n_k) == 9) {
    g.q_off = g.n_kv - g.n_q;
    std::printf("%d\n", (int)gki::tile_unseen(g, q_lo, q_hi, k0, n_k));
  }
  return 0;
}
