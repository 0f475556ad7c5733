// Host-side planning of the patch kernels (mfpatch.hip): the vertex orders of
// all element classes reduced to one reference class, and the elements cut into
// patches that share few dofs with each other.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <vector>

namespace ngsamd {

// The shape functions of class c expressed by those of class 0:
// phi_c,i(xi) = sign[i] phi_0,perm[i](A xi + b), so that with
// x'[perm[i]] = sign[i] x[i] and G' = A G A^T the class-0 operator applies.
struct ClassMap {
  std::vector<int> perm;
  std::vector<signed char> sign;
  double A[9] = {0};
};

// K(G) = sum_k g_k S_k over the packed symmetric components of G (2D xx, yy,
// xy; 3D xx, yy, zz, xy, xz, yz), S [ncomp][nd][nd].
inline void PackedForm(int dim, int nd, const double* S, const double* G, std::vector<double>& K) {
  const double g3[6] = {G[0], G[4], G[8], G[1], G[2], G[5]};
  const double g2[3] = {G[0], G[3], G[1]};
  const double* g = dim == 3 ? g3 : g2;
  const int nc = dim * (dim + 1) / 2;
  K.assign((size_t)nd * nd, 0.0);
  for (int k = 0; k < nc; k++)
    for (int i = 0; i < nd * nd; i++) K[i] += g[k] * S[(size_t)k * nd * nd + i];
}

// Numbers the rows of the symmetric matrix M by a signature that neither a
// reordering nor a change of signs of the rows and columns changes (the diagonal, then sums of
// squared entries weighted by the other rows' numbers, until all differ);
// false if some rows stay alike.
inline bool RowSignatures(int n, const std::vector<double>& M, std::vector<int>& col) {
  double mx = 0.0;
  for (double v : M) mx = std::max(mx, std::fabs(v));
  if (mx == 0.0) return false;
  std::vector<double> sig(n);
  std::vector<int> o(n);
  col.assign(n, 0);
  for (int i = 0; i < n; i++) sig[i] = M[(size_t)i * n + i] / mx;
  for (int it = 0; it < 6; it++) {
    for (int i = 0; i < n; i++) o[i] = i;
    std::sort(o.begin(), o.end(), [&](int a, int b) { return sig[a] < sig[b]; });
    int k = 0;
    col[o[0]] = 0;
    for (int i = 1; i < n; i++) {
      const double a = sig[o[i - 1]], b = sig[o[i]];
      if (b - a > 1e-9 * (std::fabs(a) + std::fabs(b) + 1e-3)) k++;
      col[o[i]] = k;
    }
    if (k == n - 1) return true;
    for (int i = 0; i < n; i++) {
      double s = std::sqrt(2.0 + col[i]);
      for (int j = 0; j < n; j++) {
        const double m = M[(size_t)i * n + j] / mx;
        s += 0.37 * m * m * std::cos(1.0 + col[j]);
      }
      sig[i] = s;
    }
  }
  return false;
}

// Class c against class 0: tries every relabelling of the reference
// element's dim + 1 vertices (barycentric coordinates xi, 1 - sum xi), finds
// the order and signs of the dofs from one generic metric and checks the
// result on every component to 1e-11 of the largest entry.
inline bool MapClass(int dim, int nd, const double* S0, const double* Sc, ClassMap& out) {
  const double G3[9] = {1.0, .31, -.23, .31, 1.7, .47, -.23, .47, 2.9}, G2[4] = {1.0, .31, .31, 1.7};
  const double* G = dim == 3 ? G3 : G2;
  std::vector<double> Mc, M0, Kc, K0;
  PackedForm(dim, nd, Sc, G, Mc);
  std::vector<int> cc, c0;
  if (!RowSignatures(nd, Mc, cc)) return false;
  double mx = 0.0;
  for (double v : Mc) mx = std::max(mx, std::fabs(v));
  auto turned = [&](const double* A, const double* H, double* R) {  // R = A H A^T
    for (int i = 0; i < dim; i++)
      for (int j = 0; j < dim; j++) {
        double s = 0.0;
        for (int k = 0; k < dim; k++)
          for (int l = 0; l < dim; l++) s += A[i * dim + k] * H[k * dim + l] * A[j * dim + l];
        R[i * dim + j] = s;
      }
  };
  std::vector<int> pi(dim + 1);
  for (int a = 0; a <= dim; a++) pi[a] = a;
  do {
    double A[9] = {0}, R[9];
    for (int a = 0; a <= dim; a++)
      if (pi[a] < dim)  // xi'_{pi(a)} = lambda_a
        for (int k = 0; k < dim; k++) A[pi[a] * dim + k] = a < dim ? (k == a ? 1.0 : 0.0) : -1.0;
    turned(A, G, R);
    PackedForm(dim, nd, S0, R, M0);
    if (!RowSignatures(nd, M0, c0)) return false;
    std::vector<int> inv(nd), s(nd);
    for (int i = 0; i < nd; i++) inv[c0[i]] = i;
    for (int i = 0; i < nd; i++) s[i] = inv[cc[i]];
    bool ok = true;
    for (int i = 0; ok && i < nd; i++)
      for (int j = 0; ok && j < nd; j++)
        ok = std::fabs(std::fabs(M0[(size_t)s[i] * nd + s[j]]) - std::fabs(Mc[(size_t)i * nd + j])) <= 1e-10 * mx;
    if (!ok) continue;
    std::vector<signed char> e(nd, 0);
    std::vector<int> todo;
    for (int r = 0; r < nd; r++) {
      if (e[r]) continue;
      e[r] = 1;
      todo.push_back(r);
      while (!todo.empty()) {
        const int i = todo.back();
        todo.pop_back();
        for (int j = 0; j < nd; j++) {
          const double a = Mc[(size_t)i * nd + j];
          if (e[j] || std::fabs(a) <= 1e-9 * mx) continue;
          e[j] = (signed char)(a * M0[(size_t)s[i] * nd + s[j]] > 0 ? e[i] : -e[i]);
          todo.push_back(j);
        }
      }
    }
    for (int a = 0; ok && a < dim; a++)
      for (int b = a; ok && b < dim; b++) {
        double E[9] = {0};
        E[a * dim + b] += 1.0;
        E[b * dim + a] += 1.0;
        turned(A, E, R);
        PackedForm(dim, nd, Sc, E, Kc);
        PackedForm(dim, nd, S0, R, K0);
        for (int i = 0; ok && i < nd; i++)
          for (int j = 0; ok && j < nd; j++)
            ok = std::fabs(Kc[(size_t)i * nd + j] - e[i] * e[j] * K0[(size_t)s[i] * nd + s[j]]) <= 1e-11 * mx;
      }
    if (!ok) continue;
    out.perm = s;
    out.sign = e;
    std::copy(A, A + 9, out.A);
    return true;
  } while (std::next_permutation(pi.begin(), pi.end()));
  return false;
}

// Elements around each of the first nv dofs of the elements (the vertices of an
// H1 element): adj[ptr[d] .. ptr[d + 1]).
inline void VertexElements(int64_t nel, int nd, int nv, int64_t ndof, const int* dofs, std::vector<int>& ptr,
                           std::vector<int>& adj) {
  ptr.assign(ndof + 1, 0);
  for (int64_t e = 0; e < nel; e++)
    for (int k = 0; k < nv; k++) ptr[dofs[e * nd + k] + 1]++;
  for (int64_t d = 0; d < ndof; d++) ptr[d + 1] += ptr[d];
  adj.resize(ptr[ndof]);
  std::vector<int> pos(ptr.begin(), ptr.end() - 1);
  for (int64_t e = 0; e < nel; e++)
    for (int k = 0; k < nv; k++) adj[pos[dofs[e * nd + k]]++] = (int)e;
}

// Cuts the elements e0 .. e1 - 1 into patches of `size` (the last one
// smaller), order[e0 .. e1): each grows from a seed beside the previous patch by
// the element sharing the most of its first nv dofs with the patch, the earliest
// found first.
inline void GrowPatches(int64_t e0, int64_t e1, int nd, int nv, int64_t ndof, const int* dofs,
                        const std::vector<int>& ptr, const std::vector<int>& adj, int size, int* order) {
  std::vector<int> stamp(ndof, -1), touched;
  std::vector<unsigned char> score(e1 - e0, 0), taken(e1 - e0, 0);
  std::vector<std::vector<int>> q(nv + 1);
  std::vector<size_t> head(nv + 1, 0);
  int64_t n = e0, next = e0;
  auto pop = [&]() -> int {
    for (int s = nv; s >= 1; s--)
      while (head[s] < q[s].size()) {
        const int e = q[s][head[s]++];
        if (!taken[e - e0] && score[e - e0] == s) return e;
      }
    return -1;
  };
  int seed = -1;
  for (int patch = 0; n < e1; patch++) {
    for (int e : touched) score[e - e0] = 0;
    touched.clear();
    for (int s = 0; s <= nv; s++) {
      q[s].clear();
      head[s] = 0;
    }
    for (int m = 0; m < size && n < e1; m++) {
      int e = m == 0 ? seed : pop();
      if (e < 0) {
        while (taken[next - e0]) next++;
        e = (int)next;
      }
      taken[e - e0] = 1;
      order[n++] = e;
      for (int k = 0; k < nv; k++) {
        const int d = dofs[(int64_t)e * nd + k];
        if (stamp[d] == patch) continue;
        stamp[d] = patch;
        for (int a = ptr[d]; a < ptr[d + 1]; a++) {
          const int f = adj[a];
          if (f < e0 || f >= e1 || taken[f - e0]) continue;
          if (score[f - e0]++ == 0) touched.push_back(f);
          q[std::min<int>(score[f - e0], nv)].push_back(f);
        }
      }
    }
    seed = pop();
  }
}

}  // namespace ngsamd
