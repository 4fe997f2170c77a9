// The block-tridiagonal inverse factors of one system on the host, pivot by pivot, for tests/test_gpu_factor_edges.py: from both
// ends to the middle block; in each block, in-place Gauss-Jordan elimination with the largest unused entry of a column as its
// pivot (the first in the order of lanes), rows scaled at the end, one fused multiply-add for every update. A block's rows and
// columns are held in the order that the inverse before it in the chain left.
#include <cmath>
#include <vector>

namespace {

template <typename T>
struct Held {  // element (lane, slot) is row rowid[lane], column colid[slot]
  int n;
  std::vector<T> x;
  std::vector<int> rowid, colid;
  T &at(int lane, int slot) { return x[lane * n + slot]; }

  Held(int n, const double *v) : n(n), x(n * n), rowid(n), colid(n) {
    for (int r = 0; r < n; ++r) {
      rowid[r] = colid[r] = r;
      for (int c = 0; c < n; ++c) at(r, c) = (T)v[c * n + r];
    }
  }

  void invert() {
    std::vector<char> used(n, 0);
    std::vector<T> sig(n, T(1));
    std::vector<int> prow(n), row(rowid), col(colid);
    for (int k = 0; k < n; ++k) {
      int p = -1;
      for (int r = 0; r < n; ++r)
        if (!used[r] && (p < 0 || std::fabs(at(r, k)) > std::fabs(at(p, k)))) p = r;
      const T ip = T(1) / at(p, k);
      for (int r = 0; r < n; ++r) {
        if (r == p) continue;
        const T g = -(at(r, k) * ip);
        for (int c = 0; c < n; ++c)
          if (c != k) at(r, c) = std::fma(g, at(p, c), at(r, c));
        at(r, k) = g;
      }
      at(p, k) = T(1);
      used[p] = 1;
      sig[p] = ip;
      prow[k] = p;
    }
    for (int k = 0; k < n; ++k) {
      rowid[prow[k]] = col[k];
      colid[k] = row[prow[k]];
    }
    for (int r = 0; r < n; ++r)
      for (int c = 0; c < n; ++c) at(r, c) *= sig[r];
  }

  void next(const double *v, const double *rs, const double *cs) {  // the block after it in the chain
    for (int l = 0; l < n; ++l)
      for (int s = 0; s < n; ++s)
        at(l, s) = (T)std::fma(-(rs[rowid[l]] * cs[colid[s]]), (double)at(l, s), v[colid[s] * n + rowid[l]]);
  }

  void store(T *d) {
    for (int l = 0; l < n; ++l)
      for (int s = 0; s < n; ++s) d[colid[s] * n + rowid[l]] = at(l, s);
  }
};

template <typename T>
void factor(int nb, int n, const double *values, T *out) {
  const long n2 = (long)n * n;
  const double *sub = values + nb * n2, *sup = sub + (long)(nb - 1) * n;
  const int m = (nb - 1) / 2;
  Held<T> top(n, values), bottom(n, values + (nb - 1) * n2);
  for (int i = 0; i < m; ++i) {
    top.invert();
    top.store(out + i * n2);
    top.next(values + (i + 1) * n2, sub + i * n, sup + i * n);
  }
  for (int i = nb - 1; i > m; --i) {
    bottom.invert();
    bottom.store(out + i * n2);
    if (i - 1 > m) {
      bottom.next(values + (i - 1) * n2, sup + (i - 1) * n, sub + (i - 1) * n);
    } else {
      std::vector<double> term(n2);
      for (int l = 0; l < n; ++l)
        for (int s = 0; s < n; ++s) {
          const int r = bottom.rowid[l], c = bottom.colid[s];
          const double t = sup[(long)m * n + r] * (double)bottom.at(l, s);
          term[c * n + r] = t * sub[(long)m * n + c];
        }
      for (int l = 0; l < n; ++l)
        for (int s = 0; s < n; ++s) {
          const double t = term[top.colid[s] * n + top.rowid[l]];
          top.at(l, s) = (T)((double)top.at(l, s) - t);
        }
    }
  }
  top.invert();
  top.store(out + m * n2);
}

}  // namespace

extern "C" {
void inverse_factor_f64(int nb, int n, const double *values, double *out) { factor<double>(nb, n, values, out); }
void inverse_factor_f32(int nb, int n, const double *values, float *out) { factor<float>(nb, n, values, out); }
}
