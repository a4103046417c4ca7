// Host-side check of planning time, built by tests/test_long_chains.py (g++,
// host code only): batched plans of trees whose units do not fit in LDS at many
// nodes in a row.  Prints a line "name steps units" per tree and fails past
// the seconds of its argument for any of them.
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <string>
#include <vector>

#include "tbh_plan.hpp"

using namespace tbh;

namespace {

// The path of n vertices: vertex leaves 0 .. n-1, edge leaf n + v joins v, v+1.
struct Path {
  int n;
  std::vector<int32_t> ptr, ix, tree;
  int next;
  explicit Path(int n_) : n(n_), next(2 * n_ - 1) {
    ptr.push_back(0);
    for (int v = 0; v < n; v++) {
      ix.push_back(v);
      ptr.push_back((int32_t)ix.size());
    }
    for (int v = 0; v + 1 < n; v++) {
      ix.push_back(v);
      ix.push_back(v + 1);
      ptr.push_back((int32_t)ix.size());
    }
  }
  int join(int a, int b) {
    tree.push_back(a);
    tree.push_back(b);
    return next++;
  }
  // vertices a .. b - 1 halved over and over
  int halves(int a, int b) {
    if (b - a == 1) return a;
    const int m = (a + b) / 2;
    return join(join(halves(a, m), n + m - 1), halves(m, b));
  }
  // node x holds the vertices before a: one after another up to b - 1
  int chain(int x, int a, int b) {
    for (int v = a; v < b; v++) x = join(join(x, n + v - 1), v);
    return x;
  }
  SliceIn in() const {
    SliceIn s;
    s.nv = n;
    s.nleaves = 2 * n - 1;
    s.ix_ptr = ptr.data();
    s.ix = ix.data();
    s.tree = tree.data();
    s.unit_wbits = 0x3f800000u;
    return s;
  }
};

int plan(const char* name, const Path& p, double limit) {
  SlicePlan P;
  std::string err;
  const auto t0 = std::chrono::steady_clock::now();
  if (plan_slice(p.in(), PlanOptions(), &P, &err)) {
    std::fprintf(stderr, "%s: %s\n", name, err.c_str());
    return 1;
  }
  const double s = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  std::printf("%s %zu %zu\n", name, P.ops.size(), P.units.size());
  if (s <= limit) return 0;
  std::fprintf(stderr, "%s: planned in %.2f s\n", name, s);
  return 1;
}

}  // namespace

int main(int argc, char** argv) {
  const double limit = argc > 1 ? std::atof(argv[1]) : 1e9;
  Path chain(50000);
  chain.chain(0, 1, 50000);
  // a subtree whose widest level does not fit, below a long chain
  Path bush(4000);
  bush.chain(bush.halves(0, 2000), 2000, 4000);
  Path half(20000);
  half.halves(0, 20000);
  return plan("chain", chain, limit) || plan("bush", bush, limit) ||
         plan("halves", half, limit);
}
