// Host check of the one-workgroup V-cycle program's levels (small_levels and
// small_node of lattice.hip): programs that hold levels with compact stencils
// beside levels with per-node values, as the assembly leaves them.  A level
// whose classes are all uniform has no per-node values (null here: a read
// ends the program), one with a class that varies has them.  Every sweep and
// defect is compared with the level's CSR matrix.
// Built by tests/test_small_levels_host.py with hipcc (host code only runs).
#include "lattice.hip"
#include <cstdio>
#include <random>
using namespace cd3d;

template <int P, bool UNI>
static int sweeps(const SmallLevel<float> &L, const HostLevel &H, const std::vector<double> &val) {
  std::mt19937 g(11);
  std::uniform_real_distribution<double> u(-1, 1);
  const size_t n3 = (size_t)H.nn * H.nn * H.nn;
  std::vector<float> x(n3, 0.f), f(n3, 0.f), out(n3, 0.f);
  for (int d = 0; d < H.nact; d++) {
    x[H.dof_node[d]] = (float)u(g);
    f[H.dof_node[d]] = (float)u(g);
  }
  const float om = 0.5f;
  int bad = 0;
  for (int mode : {kLDefect, kLJacobi, kLJacobiZero}) {
    for (int c = 0; c < L.a.nclass; c++)
      for (int k = 0; k < (int)L.a.c[c].nodes; k++) {
        if (mode == kLDefect) small_node<P, kLDefect, UNI, float>(L, c, k, x.data(), f.data(), out.data(), om);
        else if (mode == kLJacobi) small_node<P, kLJacobi, UNI, float>(L, c, k, x.data(), f.data(), out.data(), om);
        else small_node<P, kLJacobiZero, UNI, float>(L, c, k, nullptr, f.data(), out.data(), om);
      }
    // FP32 products and sums of at most 125 terms: 127 2^-24 of the terms' magnitude
    for (int d = 0; d < H.nact; d++) {
      double s = 0, mag = 0, a = 0;
      for (int q = H.rowptr[d]; q < H.rowptr[d + 1]; q++) {
        if (H.kcol[q] == d) a = val[q];
        if (H.kcol[q] >= H.nact) continue;
        const double t = val[q] * x[H.dof_node[H.kcol[q]]];
        s += t;
        mag += fabs(t);
      }
      const int e = H.dof_node[d];
      const double r = f[e] - s, w = mode == kLDefect ? r : mode == kLJacobi ? x[e] + om * r / a : om * f[e] / a;
      mag += fabs(f[e]);
      const double scale = mode == kLDefect ? mag : mag / fabs(a) + fabs((double)x[e]);
      if (!(fabs(out[e] - w) <= 130.0 / (1 << 24) * scale)) bad++;
    }
  }
  return bad;
}

// levels[i].uniform: every row of a class has the same values
template <int P>
static int check(int m, int k0, const std::vector<bool> &uniform) {
  const int top = (int)uniform.size();
  std::vector<HostLevel> H(top + 1);
  std::vector<DevLevel> D(top + 1);
  std::vector<std::vector<double>> val(top + 1);
  std::vector<std::vector<float>> lval(top + 1), linv(top + 1), lcst(top + 1);
  std::mt19937 g(3);
  std::uniform_real_distribution<double> u(-1, 1);
  for (int i = 0; i <= top; i++) {
    build_host_level(H[i], P, m, k0 + i);
    D[i].nn = H[i].nn;
    D[i].nclass = (int)H[i].lat.size();
    for (int c = 0; c < D[i].nclass; c++) D[i].cls[c] = H[i].lat[c];
    D[i].lat_nval = H[i].lat_nval;
    if (i == 0) continue;
    // values by stencil id; a level that is not uniform: perturbed per row,
    // except in class 0, which stays uniform
    std::vector<double> st(8 * kCst);
    for (auto &v : st) v = u(g);
    val[i].assign(H[i].nnz, 0.0);
    lcst[i].assign(8 * kCst, 0.f);
    for (int64_t q = 0; q < H[i].rowptr[H[i].nact]; q++) val[i][q] = st[H[i].lat_sid[q]];
    for (int r = 0; r < H[i].nact; r++) {
      for (int q = H[i].rowptr[r]; q < H[i].rowptr[r + 1]; q++) {
        if (H[i].kcol[q] == r) val[i][q] += 8;
        if (!uniform[i - 1] && (P == 1 || H[i].lat_sid[q] >= 128)) val[i][q] *= 1.0 + 0.1 * u(g);
      }
    }
    bool all = true;
    for (int c = 0; c < D[i].nclass; c++) {
      const LatClass &C = D[i].cls[c];
      D[i].uni[c] = uniform[i - 1] || (P == 2 && c == 0);
      all = all && D[i].uni[c];
      for (int s = 0; s < C.nsten && C.nodes > 0; s++) lcst[i][c * kCst + s] = (float)val[i][H[i].lat_first[c * 128 + s]];
      if (C.nodes > 0) {
        const int r = H[i].lat_node2dof[C.first];
        for (int q = H[i].rowptr[r]; q < H[i].rowptr[r + 1]; q++)
          if (H[i].kcol[q] == r) lcst[i][c * kCst + kCst - 1] = (float)(1.0 / val[i][q]);
      }
    }
    D[i].lcst = lcst[i].data();
    if (all) continue;  // no per-node values
    lval[i].resize(H[i].lat_nval);
    linv[i].resize(H[i].lat_node2dof.size());
    for (int c = 0; c < D[i].nclass; c++) {
      const LatClass &C = D[i].cls[c];
      for (int64_t k = 0; k < C.nodes; k++) {
        const int r = H[i].lat_node2dof[C.first + k];
        for (int q = H[i].rowptr[r]; q < H[i].rowptr[r + 1]; q++) {
          lval[i][C.off + (int64_t)(H[i].lat_sid[q] & 127) * C.nodes + k] = (float)val[i][q];
          if (H[i].kcol[q] == r) linv[i][C.first + k] = (float)(1.0 / val[i][q]);
        }
      }
    }
    D[i].lval = lval[i].data();
    D[i].linv = linv[i].data();
  }
  SmallArgs<float> s{};
  const bool uni = small_levels<float>(D.data(), top, s);
  bool want = true;
  for (int i = 1; i <= top; i++) want = want && D[i].lval == nullptr;
  int bad = uni != want;
  for (int i = 1; i <= top; i++)
    bad += uni ? sweeps<P, true>(s.L[i], H[i], val[i]) : sweeps<P, false>(s.L[i], H[i], val[i]);
  printf("P%d m%d k0=%d top %d: compact %d, bad %d\n", P, m, k0, top, (int)uni, bad);
  fflush(stdout);
  return bad;
}

int main() {
  int bad = 0;
  bad += check<1>(1, 0, {true, true});    // one form for the whole program
  bad += check<1>(2, 0, {false, false});
  bad += check<1>(1, 0, {true, false});   // one unknown below a level that varies
  bad += check<1>(1, 0, {true, false, true});
  bad += check<1>(3, 0, {false, true});
  bad += check<2>(1, 0, {true, false});
  bad += check<2>(1, 0, {false, true});
  printf(bad ? "FAILED %d\n" : "OK\n", bad);
  return bad != 0;
}
