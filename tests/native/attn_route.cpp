// Prints attn_route's choice (rusty_whisper_amd/csrc/rw_attn.hpp) for lines of
// "t_q t_kv n_head presplit" on stdin: tiles per k_attn_tile workgroup (0: k_attn)
// rows nsplit.
#include <cstdio>

#include "rw_attn.hpp"

int main() {
  size_t t_q, t_kv, n_head;
  int presplit;
  while (scanf("%zu %zu %zu %d", &t_q, &t_kv, &n_head, &presplit) == 4) {
    const rw::AttnRoute r = rw::attn_route(t_q, t_kv, n_head, presplit != 0, rw::ATT_MAX_SPLIT);
    printf("%d %d %d\n", r.qt, (int)r.rows, r.nsplit);
  }
  return 0;
}
