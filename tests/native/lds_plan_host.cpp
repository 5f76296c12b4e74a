// The LDS room of an operator's terms (lds_plan): what fits as a plain list beside
// the group's tables, with the row-pair table or without it, is accepted, whatever
// the parity tables take; entries are preferred, and the pair table kept, where they
// fit.
#include <cstdio>

#include "../../exactdiagonalization.jl_amd/csrc/host_logic.hpp"

using namespace edhip;

int main() {
  const uint32_t limit = 64 * 1024;
  auto up = [](uint32_t v) { return (v + 15u) & ~15u; };
  int one_by_one_without_pairs = 0;
  for (int bits : {16, 36, 63})
    for (uint32_t rank : {0u, (uint32_t)((bits + 1) * (bits + 1) * 8)})
      for (uint32_t pairs : {0u, 16384u})
        for (uint32_t group = 0; group <= 60 * 1024; group += 1000 / 16 * 16)
          for (int n_lin : {0, 1, 2, 65, 200})
            for (int single = 0; single <= 1700; single += 17) {  // terms matched by mask, in pairs of a mask
              const int n_rest = single + single % 2, n_off = 2 * n_lin + single;
              const uint32_t plain = up((uint32_t)n_off * 40), full = up(mv_layout(n_lin, mv_chunks(bits), n_rest, 1).total);
              const uint32_t with = group + pairs;
              const LdsPlan P = lds_plan(with, group, plain, full, rank);
              const uint32_t g = P.drop_pairs ? group : with;
              const uint32_t entries = P.one_by_one ? up(mv_layout(0, mv_chunks(bits), n_off, 0).total) : full;
              const bool accepted = g + std::max(plain, entries) + rank <= limit;
              if (accepted != (group + plain + rank <= limit)) return std::printf("accepts %d\n", accepted), 1;
              if (with + std::max(plain, full) + rank <= limit && (P.one_by_one || P.drop_pairs)) return std::printf("full\n"), 1;
              if (P.drop_pairs && (with + plain + rank <= limit || !pairs)) return std::printf("pairs\n"), 1;
              one_by_one_without_pairs += P.drop_pairs && P.one_by_one;
            }
  if (!one_by_one_without_pairs) return std::printf("not covered\n"), 1;
  std::printf("ok\n");
  return 0;
}
