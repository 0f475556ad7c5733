// Host-side planning of the patch kernels (mfpatch.hip): the vertex orders of
// all element classes reduced to one reference class, and the elements cut into
// patches that share few dofs with each other.
#pragma once
#include <algorithm>
#include <atomic>
#include <cmath>
#include <condition_variable>
#include <cstdint>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace ngsamd {

// A few threads for the loops of one plan, started once.  A sleeping processor
// takes 2 to 3 ms to run a new thread, as long as whole loops over a mesh of
// 30,000 triangles: the caller begins each loop at once and the threads join it
// when they are there.
class Workers {
 public:
  // the ranges of a loop, each given to one thread
  class Ranges {
   public:
    bool Next(int64_t& first, int64_t& last) {
      first = at_.fetch_add(grain_);
      last = std::min(n_, first + grain_);
      return first < n_;
    }
    // f(i) for the i of the calling thread's ranges
    template <class F>
    void Each(F f) {
      for (int64_t a, b; Next(a, b);)
        for (int64_t i = a; i < b; i++) f(i);
    }

   private:
    friend class Workers;
    Ranges(int64_t n, int64_t grain) : n_(n), grain_(grain) {}
    const int64_t n_, grain_;
    std::atomic<int64_t> at_{0};
  };

  explicit Workers(int most) {
    const int n = std::min(most, (int)std::thread::hardware_concurrency());
    try {
      th_.reserve(std::max(n - 1, 0));
      for (int i = 1; i < n; i++) th_.emplace_back([this] { Loop(); });
    } catch (...) {  // no memory or no thread to be had: those there are, at least the caller
    }
  }
  ~Workers() {
    {
      std::lock_guard<std::mutex> lock(mutex_);
      stop_ = true;
    }
    start_.notify_all();
    for (auto& t : th_) t.join();
  }
  Workers(const Workers&) = delete;
  Workers& operator=(const Workers&) = delete;

  // f(ranges), by the caller and by the threads that join it, each taking
  // ranges of `grain` of [0, n) from Next until none is left; an exception of
  // any of them ends the loop and is rethrown here
  template <class F>
  void Run(int64_t n, int64_t grain, F f) {
    Ranges ranges(n, grain);
    if (n <= grain || th_.empty()) return f(ranges);
    {
      std::lock_guard<std::mutex> lock(mutex_);
      call_ = [](void* p, Ranges& r) { (*static_cast<F*>(p))(r); };
      f_ = &f;
      ranges_ = &ranges;
      failed_ = nullptr;
      job_++;
    }
    start_.notify_all();
    Take(ranges);
    std::unique_lock<std::mutex> lock(mutex_);
    ranges_ = nullptr;  // too late to join
    done_.wait(lock, [this] { return running_ == 0; });
    if (failed_) std::rethrow_exception(failed_);
  }

 private:
  void Take(Ranges& r) {
    try {
      call_(f_, r);
    } catch (...) {
      r.at_ = r.n_;
      std::lock_guard<std::mutex> lock(mutex_);
      if (!failed_) failed_ = std::current_exception();
    }
  }
  void Loop() {
    long long seen = 0;
    std::unique_lock<std::mutex> lock(mutex_);
    while (true) {
      start_.wait(lock, [&] { return stop_ || (job_ != seen && ranges_); });
      if (stop_) return;
      seen = job_;
      running_++;
      Ranges& r = *ranges_;  // stays until running_ is 0
      lock.unlock();
      Take(r);
      lock.lock();
      if (--running_ == 0) done_.notify_one();
    }
  }
  std::vector<std::thread> th_;
  std::mutex mutex_;
  std::condition_variable start_, done_;
  void (*call_)(void*, Ranges&) = nullptr;
  void* f_ = nullptr;
  Ranges* ranges_ = nullptr;
  int running_ = 0;
  long long job_ = 0;
  bool stop_ = false;
  std::exception_ptr failed_;
};

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

// Factor of each class's reference matrices (see MfFacKernel): the rows
// Bw[(d,i)][q] = b_{q,i,d} sqrt(w_q) are orthonormalised by Gram-Schmidt with
// pivoting on the largest remaining row (each new vector orthogonalised twice
// against the basis), stopping when every remaining row is below 1e-10 of
// the largest row; D[(d,i)][k] = Bw[(d,i)] . phi_k.  Returns the largest rank
// over the classes (D has that many columns, zero beyond a class's own rank),
// or 0 if a weight is not positive or D Phi misses Bw by more than 1e-12
// relative.  D is [class][d][i][rank].
inline int FactorGradients(int dim, int nd, int nq, int nclass, const double* bmat, const double* w,
                           std::vector<double>& D) {
  for (int q = 0; q < nq; q++)
    if (!(w[q] > 0.0)) return 0;
  const int nr = dim * nd;
  const size_t bsz = (size_t)nq * nd * dim;
  std::vector<std::vector<double>> phis(nclass);
  std::vector<double> Bw((size_t)nr * nq);
  int rank = 0;
  auto dot = [&](const double* a, const double* b) {
    double t = 0.0;
    for (int q = 0; q < nq; q++) t += a[q] * b[q];
    return t;
  };
  for (int c = 0; c < nclass; c++) {
    for (int d = 0; d < dim; d++)
      for (int i = 0; i < nd; i++)
        for (int q = 0; q < nq; q++)
          Bw[((size_t)d * nd + i) * nq + q] = bmat[c * bsz + ((size_t)q * nd + i) * dim + d] * std::sqrt(w[q]);
    std::vector<double> res(Bw);
    std::vector<double>& phi = phis[c];
    double norm0 = 0.0;
    for (int r = 0; r < nr; r++) norm0 = std::max(norm0, std::sqrt(dot(&Bw[(size_t)r * nq], &Bw[(size_t)r * nq])));
    if (norm0 == 0.0) continue;
    for (int k = 0; k < std::min(nr, nq); k++) {
      int best = -1;
      double bn = 0.0;
      for (int r = 0; r < nr; r++) {
        const double t = std::sqrt(dot(&res[(size_t)r * nq], &res[(size_t)r * nq]));
        if (t > bn) bn = t, best = r;
      }
      if (best < 0 || bn <= 1e-10 * norm0) break;
      std::vector<double> v(res.begin() + (size_t)best * nq, res.begin() + (size_t)(best + 1) * nq);
      for (int pass = 0; pass < 2; pass++) {
        for (size_t j = 0; j < phi.size() / nq; j++) {
          const double t = dot(v.data(), &phi[j * nq]);
          for (int q = 0; q < nq; q++) v[q] -= t * phi[j * nq + q];
        }
        const double vn = std::sqrt(dot(v.data(), v.data()));
        for (int q = 0; q < nq; q++) v[q] /= vn;
      }
      phi.insert(phi.end(), v.begin(), v.end());
      for (int r = 0; r < nr; r++) {
        double* rr = &res[(size_t)r * nq];
        const double t = dot(rr, v.data());
        for (int q = 0; q < nq; q++) rr[q] -= t * v[q];
      }
    }
    rank = std::max(rank, (int)(phi.size() / nq));
  }
  if (rank == 0) return 0;
  D.assign((size_t)nclass * nr * rank, 0.0);
  for (int c = 0; c < nclass; c++) {
    const std::vector<double>& phi = phis[c];
    const int rc = (int)(phi.size() / nq);
    double norm0 = 0.0, err = 0.0;
    for (int d = 0; d < dim; d++)
      for (int i = 0; i < nd; i++) {
        std::vector<double> row(nq), rec(nq, 0.0);
        for (int q = 0; q < nq; q++) row[q] = bmat[c * bsz + ((size_t)q * nd + i) * dim + d] * std::sqrt(w[q]);
        double* Dr = &D[((size_t)c * nr + (size_t)d * nd + i) * rank];
        for (int k = 0; k < rc; k++) {
          Dr[k] = dot(row.data(), &phi[(size_t)k * nq]);
          for (int q = 0; q < nq; q++) rec[q] += Dr[k] * phi[(size_t)k * nq + q];
        }
        for (int q = 0; q < nq; q++) {
          norm0 = std::max(norm0, std::fabs(row[q]));
          err = std::max(err, std::fabs(row[q] - rec[q]));
        }
      }
    if (err > 1e-12 * norm0) return 0;
  }
  return rank;
}

// Whether the factor of class c is the one of class 0 relabelled, entry by entry
// in the operand format that `bits` rounds to: the directions permuted and
// turned by A, the dofs by the class map, the rank columns in some order
// and with some signs.  D0, Dc [d][i][rank] (FactorGradients).
template <class F>
inline bool SameRoundedFactor(int dim, int nd, int rank, const double* D0, const double* Dc, const ClassMap& m, F bits) {
  std::vector<int> pi(dim, -1), sd(dim, 0);
  for (int d = 0; d < dim; d++) {  // column d of A: one entry, +-1
    for (int r = 0; r < dim; r++)
      if (m.A[r * dim + d] != 0.0) {
        if (pi[d] >= 0) return false;
        pi[d] = r;
        sd[d] = m.A[r * dim + d] > 0 ? 1 : -1;
      }
    if (pi[d] < 0) return false;
  }
  std::vector<char> used(rank, 0);
  for (int k = 0; k < rank; k++) {
    auto same = [&](int q, int s) {
      for (int d = 0; d < dim; d++)
        for (int i = 0; i < nd; i++) {
          const double a = Dc[((size_t)d * nd + i) * rank + k];
          const double b = s * sd[d] * m.sign[i] * D0[((size_t)pi[d] * nd + m.perm[i]) * rank + q];
          if (bits(a) != bits(b) && !(std::fabs(a) + std::fabs(b) < 1e-12)) return false;
        }
      return true;
    };
    int found = -1;
    for (int q = 0; q < rank && found < 0; q++)
      if (!used[q] && (same(q, 1) || same(q, -1))) found = q;
    if (found < 0) return false;
    used[found] = 1;
  }
  return true;
}

// Elements around each of the first nv dofs of the elements (the vertices of an
// H1 element): adj[ptr[d] .. ptr[d + 1]), d up to the largest of these dofs.
inline void VertexElements(int64_t nel, int nd, int nv, const int* dofs, std::vector<int>& ptr,
                           std::vector<int>& adj) {
  int last = -1;
  for (int64_t e = 0; e < nel; e++)
    for (int k = 0; k < nv; k++) last = std::max(last, dofs[e * nd + k]);
  ptr.assign((size_t)last + 2, 0);
  for (int64_t e = 0; e < nel; e++)
    for (int k = 0; k < nv; k++) ptr[dofs[e * nd + k] + 1]++;
  for (int d = 0; d <= last; d++) ptr[d + 1] += ptr[d];
  adj.resize(ptr.back());
  std::vector<int> pos(ptr.begin(), ptr.end() - 1);
  for (int64_t e = 0; e < nel; e++)
    for (int k = 0; k < nv; k++) adj[pos[dofs[e * nd + k]]++] = (int)e;
}

// Cuts the elements e0 .. e1 - 1 into patches of `size` (the last one
// smaller), order[e0 .. e1): each grows from a seed beside the previous patch by
// the element sharing the most of its first nv dofs with the patch, the earliest
// found first.  stamp: the last patch of each vertex dof, 0 at first, and
// `patch` their number, kept from one call of a thread to the next (an array
// per call would take the whole mesh's size for each piece of it: 96^3 cubes
// p=4 39 s of set-up in place of 0.5).
inline void GrowPatches(int64_t e0, int64_t e1, int nd, int nv, const int* dofs, const std::vector<int>& ptr,
                        const std::vector<int>& adj, int size, std::vector<int>& stamp, int& patch, int* order) {
  std::vector<int> touched;
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
  while (n < e1) {
    patch++;
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

// Each range of `per` entries of the list by falling ptr[v + 1] - ptr[v], equal
// ones in their former order (a counting sort: the counts are small).
inline void SortRangesByCount(std::vector<int>& list, int64_t per, const std::vector<int>& ptr) {
  std::vector<int> at, part;
  const int64_t n = (int64_t)list.size();
  for (int64_t a = 0; a < n; a += per) {
    const int64_t b = std::min(n, a + per);
    int most = 0;
    for (int64_t i = a; i < b; i++) most = std::max(most, ptr[list[i] + 1] - ptr[list[i]]);
    at.assign(most + 2, 0);  // at[most - count + 1]: entries of that count
    for (int64_t i = a; i < b; i++) at[most - (ptr[list[i] + 1] - ptr[list[i]]) + 1]++;
    for (int c = 0; c <= most; c++) at[c + 1] += at[c];
    part.resize(b - a);
    for (int64_t i = a; i < b; i++) part[at[most - (ptr[list[i] + 1] - ptr[list[i]])]++] = list[i];
    std::copy(part.begin(), part.end(), list.begin() + a);
  }
}

// pos: the positions 0 .. n - 1 by rising key, equal ones in order.  Byte by
// byte, those in which the keys differ: 5 passes over the 370 dofs of a 2D patch
// take a third of a comparison sort's time, whose branches are random.
class KeySort {
 public:
  void operator()(const std::vector<uint64_t>& key, std::vector<int>& pos) {
    const int n = (int)key.size();
    pos.resize(n);
    to_.resize(n);
    uint64_t differ = 0;
    for (int i = 0; i < n; i++) {
      pos[i] = i;
      differ |= key[i] ^ key[0];
    }
    for (int s = 0; s < 64; s += 8) {
      if (!(differ >> s & 255)) continue;
      int at[256] = {0};
      for (int i = 0; i < n; i++) at[key[i] >> s & 255]++;
      for (int b = 0, sum = 0; b < 256; b++) {
        const int c = at[b];
        at[b] = sum;
        sum += c;
      }
      for (int i = 0; i < n; i++) to_[at[key[pos[i]] >> s & 255]++] = pos[i];
      pos.swap(to_);
    }
  }

 private:
  std::vector<int> to_;
};

// Numbers the distinct values of a list in the order they are added: a table
// of the list's size (the dofs of a patch), whatever the range of the values.
class Numbering {
 public:
  explicit Numbering(size_t most) {
    while (((size_t)1 << bits_) < 2 * most) bits_++;
    key_.assign((size_t)1 << bits_, 0);
    num_.resize(key_.size());
    round_.assign(key_.size(), 0);
  }
  void Clear() {
    n_ = 0;
    cur_++;
  }
  // the number of v, given to it now if it has none (then it equals the former Size())
  int Add(int v) {
    size_t h = Slot(v);
    if (round_[h] != cur_) {
      round_[h] = cur_;
      key_[h] = v;
      num_[h] = n_++;
    }
    return num_[h];
  }
  int Size() const { return n_; }

 private:
  size_t Slot(int v) const {
    const size_t mask = key_.size() - 1;
    size_t h = ((uint32_t)v * 2654435769u) >> (32 - bits_);
    while (round_[h] == cur_ && key_[h] != v) h = (h + 1) & mask;
    return h;
  }
  int bits_ = 4, n_ = 0;
  uint32_t cur_ = 1;
  std::vector<int> key_, num_;
  std::vector<uint32_t> round_;
};

}  // namespace ngsamd
