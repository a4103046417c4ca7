// Host-side replay of the units of batched plans (csrc/tbh_plan.cpp), built by
// tests/test_unit_replay.py with sanitizers (g++, host code only).  The kernel
// runs a level's steps side by side with one barrier per level, each wave from
// a list of its own, and LDS blocks are used again once their tensor is read;
// so, level by level:
//  - a step reads only entries written before its level, all of them by one
//    step (or copied to LDS at the start) and as many as its operand has;
//  - a step writes no entry that any step of its level reads or writes;
//  - every chunk of every step's output is written once, and every tensor is
//    read by one step.
// Slices come from a file in the format of plan_check.cpp.  A second pass
// moves every item of some units a level earlier, which has to be noticed.
#include <cstdio>
#include <map>
#include <string>
#include <tuple>
#include <vector>

#include "tbh_plan.hpp"

using namespace tbh;

namespace {

struct Item {
  UnitItem it;
  int level;
};

// offsets of an operand's entries: bit k < n of the union, if set in m, at the
// place of m's lower bits; `fixed` bits are part of the item's offset
std::vector<uint32_t> places(uint32_t m, uint32_t free_bits) {
  std::vector<uint32_t> v{0};
  for (int k = 0; k < 16; k++) {
    if (!(m >> k & 1) || !(free_bits >> k & 1)) continue;
    const uint32_t stride = 1u << __builtin_popcount(m & ((1u << k) - 1));
    for (size_t i = 0, n = v.size(); i < n; i++) v.push_back(v[i] + stride);
  }
  return v;
}

std::string replay(const SlicePlan& P, const PUnit& u, bool early) {
  std::map<int, std::vector<UnitItem>> levels;
  for (int w = 0; w < kUnitWaves; w++) {
    int level = 0;
    for (int i = u.start[w]; i < u.start[w + 1]; i++) {
      UnitItem it = P.items[u.item0 + i];
      level += it.levels;
      levels[early && level > 0 ? level - 1 : level].push_back(it);
    }
  }
  // per LDS entry: the tensor it holds (-1: none), the last level that read it
  std::vector<int> owner(kUnitLds, -1), read_at(kUnitLds, -1), written_at(kUnitLds, -1);
  std::vector<int> entries, readers;  // per tensor
  auto tensor = [&](uint32_t off, uint32_t n) {
    const int t = (int)entries.size();
    entries.push_back((int)n);
    readers.push_back(0);
    for (uint32_t e = off; e < off + n; e++) {
      if (e >= (uint32_t)kUnitLds || owner[e] >= 0) return false;
      owner[e] = t;
    }
    return true;
  };
  bool ok = tensor(0, 4);  // the edge tensor
  for (int i = 0; ok && i < u.nvert; i++) ok = tensor(4 + 2 * i, 2);
  for (int q = 0; ok && q < u.next; q++)
    ok = tensor(P.ext[u.ext0 + q].off, 1u << P.tensors[P.ext[u.ext0 + q].tensor].rank);
  if (!ok) return "tensors at the start overlap";
  const int edge = 0;
  std::vector<int> root;
  for (auto& lv : levels) {
    const int L = lv.first;
    // a step: its items of one level, by its output and operands' labels
    std::map<std::tuple<int, int, int, int>, std::vector<UnitItem>> steps;
    for (const UnitItem& it : lv.second)
      steps[{it.f & 0x1ff, it.oC, it.mA, it.mB}].push_back(it);
    for (auto& s : steps) {
      int from[2] = {-1, -1};
      for (const UnitItem& it : s.second) {
        const int nP = it.f & 15, nR = (it.f >> 4) & 15, lc = it.f >> 12;
        uint32_t free_bits = ((1u << nR) - 1) << nP;
        for (int k = 0; k < nP; k++) free_bits |= (k < 6 + lc ? 1u : 0u) << k;
        for (int h = 0; h < 2; h++) {
          const uint32_t m = h ? it.mB : it.mA, at = h ? it.oB : it.oA;
          for (uint32_t p : places(m, free_bits)) {
            if (at + p >= (uint32_t)kUnitLds) return "operand out of LDS";
            const int t = owner[at + p];
            if (t < 0) return "operand never written";
            if (written_at[at + p] >= L) return "operand written at its own level";
            if (from[h] >= 0 && from[h] != t) return "operand of two tensors";
            from[h] = t;
            read_at[at + p] = L;
            if (entries[t] != 1 << __builtin_popcount(m)) return "operand of another size";
          }
        }
      }
      for (int h = 0; h < 2; h++)
        if (from[h] != edge && ++readers[from[h]] > 1) return "tensor read twice";
    }
    for (auto& s : steps) {
      const int nP = std::get<0>(s.first) & 15;
      const bool is_root = std::get<0>(s.first) & kItemRoot;
      const int chunks = nP > 6 ? 1 << (nP - 6) : 1;
      std::vector<int> seen(chunks, 0);
      const int t = (int)entries.size();
      entries.push_back(1 << nP);
      readers.push_back(0);
      if (is_root) root.push_back(t);
      for (const UnitItem& it : s.second)
        for (int c = it.c0; c < it.c0 + (1 << (it.f >> 12)); c++) {
          if (c >= chunks || seen[c]++) return "chunk written twice";
          if (is_root) continue;
          for (int e = 0; e < (nP > 6 ? 64 : 1 << nP); e++) {
            const uint32_t at = it.oC + 64 * c + e;
            if (at >= (uint32_t)kUnitLds) return "output out of LDS";
            if (read_at[at] == L) return "output over an operand of its level";
            if (written_at[at] == L) return "two outputs of a level";
            written_at[at] = L;
            owner[at] = t;
          }
        }
      for (int n : seen)
        if (n != 1) return "chunk not written";
    }
  }
  if (u.items() > 0 && root.size() != 1) return "roots";
  for (size_t t = 1; t < readers.size(); t++)
    if (readers[t] != (!root.empty() && (int)t == root[0] ? 0 : 1)) return "tensor not read";
  return "";
}

}  // namespace

int main(int argc, char** argv) {
  if (argc < 2) return 2;
  FILE* f = std::fopen(argv[1], "rb");
  if (!f) return 2;
  int n = 0;
  if (std::fread(&n, 4, 1, f) != 1) return 2;
  long plans = 0, units = 0, mixed = 0, deep = 0, noticed = 0;
  for (int i = 0; i < n; i++) {
    int h[5];
    if (std::fread(h, 4, 5, f) != 5) return 2;
    std::vector<int32_t> ixp(h[2]), ix(h[3]), tree(h[4]);
    if (std::fread(ixp.data(), 4, h[2], f) != (size_t)h[2] ||
        std::fread(ix.data(), 4, h[3], f) != (size_t)h[3] ||
        std::fread(tree.data(), 4, h[4], f) != (size_t)h[4])
      return 2;
    SliceIn in;
    in.nv = h[0];
    in.nleaves = h[1];
    in.ix_ptr = ixp.data();
    in.ix = ix.data();
    in.tree = tree.empty() ? nullptr : tree.data();
    in.unit_wbits = 0x3f800000u;  // Float32 1
    SlicePlan P;
    std::string err;
    // (tensors of more than 30 labels, of some random trees, are refused)
    if (plan_slice(in, PlanOptions(), &P, &err)) continue;
    plans++;
    for (const PUnit& u : P.units) {
      if (u.items() == 0) continue;
      units++;
      mixed += u.next > 0;
      const std::string bad = replay(P, u, false);
      if (!bad.empty()) {
        std::fprintf(stderr, "slice %d, unit of tensor %d: %s\n", i, u.tensor, bad.c_str());
        return 1;
      }
      if (u.items() >= 4) {
        deep++;
        noticed += !replay(P, u, true).empty();
      }
    }
  }
  std::fclose(f);
  std::printf("%ld plans %ld units %ld mixed %ld moved %ld noticed\n", plans, units, mixed, deep, noticed);
  return 0;
}
