// jja_rowparts.h -- tables of the tridiagonal systems of a lattice's modes cut into
// row parts (host code): what a part needs to solve its own block, and the end rows
// of all parts from those solutions (Wang, ACM TOMS 7 (1981) 170-183).
#ifndef JJA_ROWPARTS_H
#define JJA_ROWPARTS_H

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <vector>

namespace {

// the tables are formed in extended precision: their rounding is that of one value
using real = long double;

std::vector<real> thomas_inverse(real diag, real g, int32_t s) {
  std::vector<real> inv(s);
  real piv = diag;
  for (int32_t l = 0; l < s; ++l) {
    inv[l] = 1.0 / piv;
    piv = diag - g * g * inv[l];
  }
  return inv;
}

// g A^-1 e_0 for the block of s rows
std::vector<real> spike_of(const std::vector<real>& inv, real g, int32_t s) {
  std::vector<real> v(s);
  real d = 0.0;
  for (int32_t l = 0; l < s; ++l) v[l] = d = ((l == 0 ? g : 0.0) + g * d) * inv[l];
  for (int32_t l = s - 2; l >= 0; --l) v[l] += g * inv[l] * v[l + 1];
  return v;
}

// Inverse of the n x n matrix a in place (Gauss-Jordan, partial pivoting).
void invert(std::vector<real>& a, int32_t n) {
  std::vector<real> r(static_cast<size_t>(n) * n, 0.0);
  for (int32_t i = 0; i < n; ++i) r[static_cast<size_t>(i) * n + i] = 1.0;
  for (int32_t c = 0; c < n; ++c) {
    int32_t p = c;
    for (int32_t i = c + 1; i < n; ++i)
      if (std::fabs(a[static_cast<size_t>(i) * n + c]) > std::fabs(a[static_cast<size_t>(p) * n + c])) p = i;
    for (int32_t j = 0; j < n && p != c; ++j) {
      std::swap(a[static_cast<size_t>(p) * n + j], a[static_cast<size_t>(c) * n + j]);
      std::swap(r[static_cast<size_t>(p) * n + j], r[static_cast<size_t>(c) * n + j]);
    }
    const real d = 1.0 / a[static_cast<size_t>(c) * n + c];
    for (int32_t j = 0; j < n; ++j) {
      a[static_cast<size_t>(c) * n + j] *= d;
      r[static_cast<size_t>(c) * n + j] *= d;
    }
    for (int32_t i = 0; i < n; ++i) {
      const real f = a[static_cast<size_t>(i) * n + c];
      if (i == c || f == 0.0) continue;
      for (int32_t j = 0; j < n; ++j) {
        a[static_cast<size_t>(i) * n + j] -= f * a[static_cast<size_t>(c) * n + j];
        r[static_cast<size_t>(i) * n + j] -= f * r[static_cast<size_t>(c) * n + j];
      }
    }
  }
  a = r;
}

// R rows and C modes in G parts, the first R % G with a row more than R / G:
//   inv      [rows][C] inverse pivots of a part's own block (rows: the most a part has)
//   spike    [2][rows][C] response to the row below, parts of R / G and R / G + 1 rows
//   reduced  [2 G][2 G][C] first and last rows of the parts from their own blocks'
void row_part_tables(int32_t R, int32_t C, int32_t G, real g, real gc, std::vector<double>* inv_out,
                     std::vector<double>* spike_out, std::vector<double>* reduced_out) {
  const int32_t base = R / G, extra = R % G, rows = base + (extra ? 1 : 0);
  const real pi = 3.14159265358979323846264338328L;
  inv_out->assign(static_cast<size_t>(rows) * C, 0.0);
  spike_out->assign(2 * static_cast<size_t>(rows) * C, 0.0);
  reduced_out->assign(static_cast<size_t>(G) * 4 * G * C, 0.0);
  for (int32_t k = 0; k < C; ++k) {
    const real h = std::sin(pi * (k + 1) / (2 * static_cast<real>(C + 1))), diag = 2 * g + gc * 4 * h * h;
    const std::vector<real> inv = thomas_inverse(diag, g, rows);
    std::vector<real> v[2];
    for (int32_t i = 0; i < 2; ++i) {
      const int32_t s = std::min(base + i, rows);
      v[i] = spike_of(inv, g, s);
      for (int32_t l = 0; l < s; ++l) (*spike_out)[(static_cast<size_t>(i) * rows + l) * C + k] = static_cast<double>(v[i][l]);
    }
    for (int32_t l = 0; l < rows; ++l) (*inv_out)[static_cast<size_t>(l) * C + k] = static_cast<double>(inv[l]);
    // unknowns 2p, 2p + 1: the first and last row of part p
    const int32_t n = 2 * G;
    std::vector<real> m(static_cast<size_t>(n) * n, 0.0);
    for (int32_t p = 0; p < G; ++p) {
      const std::vector<real>& vp = v[p < extra ? 1 : 0];
      const int32_t s = base + (p < extra ? 1 : 0);
      for (int32_t e = 0; e < 2; ++e) {
        real* row = &m[static_cast<size_t>(2 * p + e) * n];
        const int32_t l = e ? s - 1 : 0;
        row[2 * p + e] = 1.0;
        if (p > 0) row[2 * p - 1] -= vp[l];
        if (p + 1 < G) row[2 * p + 2] -= vp[s - 1 - l];
      }
    }
    invert(m, n);
    for (size_t i = 0; i < m.size(); ++i) (*reduced_out)[i * C + k] = static_cast<double>(m[i]);
  }
}

}  // namespace

#endif  // JJA_ROWPARTS_H
