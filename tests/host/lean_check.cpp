// Host-side check of the plans of less memory (PlanOptions::lean), built by
// tests/test_lean_plan.py with sanitizers (g++, host code only): prints, per
// slice of a file (the format of plan_check.cpp) and for the batched and the
// plain lowering, the arena of the default plan and of the lean one.
#include <cstdio>
#include <string>
#include <vector>

#include "tbh_plan.hpp"

int main(int argc, char** argv) {
  if (argc < 2) return 2;
  FILE* f = std::fopen(argv[1], "rb");
  if (!f) return 2;
  int n = 0;
  if (std::fread(&n, 4, 1, f) != 1) return 2;
  for (int i = 0; i < n; i++) {
    int h[5];
    if (std::fread(h, 4, 5, f) != 5) return 2;
    std::vector<int32_t> ixp(h[2]), ix(h[3]), tree(h[4]);
    if (std::fread(ixp.data(), 4, h[2], f) != (size_t)h[2] ||
        std::fread(ix.data(), 4, h[3], f) != (size_t)h[3] ||
        std::fread(tree.data(), 4, h[4], f) != (size_t)h[4])
      return 2;
    tbh::SliceIn in;
    in.nv = h[0];
    in.nleaves = h[1];
    in.ix_ptr = ixp.data();
    in.ix = ix.data();
    in.tree = tree.empty() ? nullptr : tree.data();
    in.unit_wbits = 0x3f800000u;  // Float32 1
    for (bool batched : {true, false}) {
      long arena[2];
      for (bool lean : {false, true}) {
        tbh::PlanOptions opt;
        opt.batched = batched;
        opt.lean = lean;
        tbh::SlicePlan P;
        std::string err;
        if (tbh::plan_slice(in, opt, &P, &err)) {
          std::fprintf(stderr, "slice %d: %s\n", i, err.c_str());
          return 1;
        }
        if (lean && (!P.units.empty() || (int)P.leaves.size() != in.nleaves)) {
          std::fprintf(stderr, "slice %d: a lean plan with units\n", i);
          return 1;
        }
        arena[lean] = (long)P.arena_bytes;
      }
      std::printf("%ld %ld\n", arena[0], arena[1]);
    }
  }
  std::fclose(f);
  return 0;
}
