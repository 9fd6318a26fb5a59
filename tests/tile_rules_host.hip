// Host driver for the CPU tests of the kernels' rules (gki_common.cuh).
//
// argv[1] "unseen": stdin lines n_q n_kv causal sink window q_lo q_hi k0 n_k,
//   stdout tile_unseen per line;
// "form": lines dtype scale, stdout bwd_form_of;
// "grid": lines head_dim tiles n_q n_kv causal sink window rows, stdout row_kv_tiles
//   of a tile of that many rows and the launch rules of a grid of that many tiles.
#include <cstdio>
#include <cstring>

#include "gki_common.cuh"

int main(int argc, char** argv) {
  const char* what = argc > 1 ? argv[1] : "";
  if (!std::strcmp(what, "unseen")) {
    gki::Geom g{};
    int q_lo, q_hi, k0, n_k;
    while (std::scanf("%d %d %d %d %d %d %d %d %d", &g.n_q, &g.n_kv, &g.causal, &g.sink, &g.window, &q_lo, &q_hi,
                      &k0, &n_k) == 9) {
      g.q_off = g.n_kv - g.n_q;
      std::printf("%d\n", (int)gki::tile_unseen(g, q_lo, q_hi, k0, n_k));
    }
  } else if (!std::strcmp(what, "form")) {
    int dtype;
    float scale;
    while (std::scanf("%d %f", &dtype, &scale) == 2) std::printf("%d\n", gki::bwd_form_of(dtype, scale));
  } else if (!std::strcmp(what, "grid")) {
    gki::Geom g{};
    int head_dim, tiles, rows;
    while (std::scanf("%d %d %d %d %d %d %d %d", &head_dim, &tiles, &g.n_q, &g.n_kv, &g.causal, &g.sink, &g.window,
                      &rows) == 8) {
      const int kv = gki::row_kv_tiles(g, rows);
      std::printf("%d %d %d %d\n", kv, (int)gki::fwd_shares_keys(head_dim, tiles, kv),
                  gki::f32_row_blocks(head_dim, tiles, kv), gki::f32_kv_blocks(head_dim, tiles));
    }
  } else {
    return 1;
  }
  return 0;
}
