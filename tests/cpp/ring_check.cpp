// Host replay of the ring solve's LDS slots.
//
// The ring kernel keeps the value of the row at position p (all L rows of a
// block in storage order, then all U rows) in slot p % rows of its ring, rows =
// TrsvPack::window_needed.  Nothing orders the writes of one step: two waves
// take its rows, and the lanes of a wave write together.  So a step's writes
// are replayed in both row orders, each step's reads before its writes and
// (for a wave that is ahead) after the other rows' writes, and every replay must
// give the plain forward/backward substitution on the block's factors.
//
// usage: ring_check   (exit 0 when every level of every problem agrees)
#include <algorithm>
#include <cmath>
#include <complex>
#include <cstdio>
#include <string>
#include <vector>

#include "../../pargemslr_amd/csrc/host/gemslr_host.hpp"
#include "../../pargemslr_amd/csrc/host/gen.hpp"
#include "../../pargemslr_amd/csrc/host/trsv_pack.hpp"

using namespace pgs;

namespace {

constexpr int kStepRows = 32;
constexpr int kSlabWidth = 20;
constexpr int kMaxWindow = 8192;

template <typename T>
T value_of(double re, double im) {
  if constexpr (is_complex<T>::value) return T(re, im);
  else return re;
}

// y = L^{-1} b, x_i = dinv_i (y_i - U_i x)
template <typename T>
void block_solve(const IluFactor<T>& F, const T* b, T* x) {
  const int n = F.n;
  std::vector<T> y(n);
  for (int i = 0; i < n; ++i) {
    T s = b[i];
    for (int k = F.L.ia[i]; k < F.L.ia[i + 1]; ++k) s -= F.L.a[k] * y[F.L.ja[k]];
    y[i] = s;
  }
  for (int i = n - 1; i >= 0; --i) {
    T s = y[i];
    for (int k = F.U.ia[i]; k < F.U.ia[i + 1]; ++k) s -= F.U.a[k] * x[F.U.ja[k]];
    x[i] = F.Dinv[i] * s;
  }
}

// How a step's rows meet in the ring: in row order or against it, all reads
// before all writes or one row after the other.
struct Order {
  bool reversed, row_by_row;
};

template <typename T>
void ring_solve(const TrsvPack<T>& P, const std::vector<int>& desc, int sbeg, int sU, int send, int b, const T* rhs,
                T* x, int rows, Order o) {
  std::vector<T> ring(rows, T(0.0));
  const int64_t e0 = P.blk_ent0[b], q0 = P.blk_ri0[b];
  for (int s = sbeg; s < send; ++s) {
    const bool upper = s >= sU;
    const int ro = desc[4 * s], eo = desc[4 * s + 1], nr = desc[4 * s + 2], w = desc[4 * s + 3];
    const int end = ro + nr;
    std::vector<T> v(nr);
    auto solve = [&](int t) {
      const int row = P.rows[q0 + ro + t];
      T acc = T(0.0);
      for (int j = 0; j < w; ++j) {
        const int64_t e = e0 + eo + (int64_t)t * w + j;
        if (P.val[e] == T(0.0)) continue;  // padding
        const int p = end - 1 - ((end - 1 - P.col[e]) & (P.window - 1));
        acc += P.val[e] * ring[p % rows];
      }
      v[t] = (upper ? x[row] : rhs[row]) - acc;
      if (upper) v[t] *= P.dinv[q0 + ro + t];
    };
    auto write = [&](int t) {
      ring[(ro + t) % rows] = v[t];
      x[P.rows[q0 + ro + t]] = v[t];
    };
    auto each = [&](auto f) {
      for (int t = 0; t < nr; ++t) f(o.reversed ? nr - 1 - t : t);
    };
    if (o.row_by_row) {
      each([&](int t) {
        solve(t);
        write(t);
      });
    } else {
      each(solve);
      each(write);
    }
  }
}

// Replays every level; `shorter` takes rows off the ring (a control).
template <typename T>
bool check_op(const std::string& name, const HostOp<T>& op, int shorter) {
  bool ok = true;
  for (int l = 0; l < op.nlev; ++l) {
    const HostLevel<T>& L = op.levels[l];
    const int nl = op.nloc(l);
    TrsvPack<T> P = trsv_pack(L, op.lev_ptr[l], nl, kStepRows, kMaxWindow, kSlabWidth);
    std::vector<int> dh, sh, suh;
    half_steps(P.desc, P.blk_step, P.blk_stepU, dh, sh, suh);
    int longest = 0;
    for (size_t i = 2; i < P.desc.size(); i += 4) longest = std::max(longest, P.desc[i]);
    const int rows = std::max(1, P.window_needed - shorter);
    std::vector<double> g(2 * (size_t)nl);
    rng_normal(1000 + l, 2 * (int64_t)nl, g.data());
    std::vector<T> rhs(nl), ref(nl), x(nl);
    for (int i = 0; i < nl; ++i) rhs[i] = value_of<T>(g[2 * i], g[2 * i + 1]);
    double emax = 0.0, nmax = 0.0;
    for (int b = 0; b < L.ncomp; ++b) {
      const int r0 = P.blk_row0[b], nb = P.blk_row0[b + 1] - r0;
      block_solve(L.ilu[b], rhs.data() + r0, ref.data() + r0);
      for (int k = 0; k < 8; ++k) {
        const Order o = {(k & 1) != 0, (k & 2) != 0};
        if (k & 4)
          ring_solve(P, P.desc, P.blk_step[b], P.blk_stepU[b], P.blk_step[b + 1], b, rhs.data() + r0, x.data() + r0,
                     rows, o);
        else
          ring_solve(P, dh, sh[b], suh[b], sh[b + 1], b, rhs.data() + r0, x.data() + r0, rows, o);
        for (int i = r0; i < r0 + nb; ++i) {
          nmax = std::max(nmax, std::abs(ref[i]));
          const double e = std::abs(x[i] - ref[i]);
          emax = e <= emax ? emax : e;  // a NaN stays
        }
      }
    }
    const double rel = nmax > 0.0 ? emax / nmax : emax;
    const bool good = P.window > 0 && rel <= 1e-12;
    std::printf("%s level %d: %d blocks, longest step %d rows, ring %d rows%s, rel err %.2e %s\n", name.c_str(), l,
                L.ncomp, longest, rows, shorter ? " (shortened)" : "", rel, good ? "ok" : "MISMATCH");
    ok = ok && good;
  }
  return ok;
}

template <typename T>
bool run(const std::string& name, const Csr<T>& A, int nlev, int ncomp, double droptol, int rownnz, bool perm = true,
         int shorter = 0) {
  GemslrParams prm;
  prm.nlev = nlev;
  prm.ncomp = ncomp;
  prm.droptol_B = prm.droptol_C = droptol;
  prm.rownnz_B = prm.rownnz_C = rownnz;
  prm.lr_rank1 = prm.lr_rank2 = 0;
  prm.schur_enable = 0;
  if (!perm) prm.perm_option = 0;
  HostOp<T> op;
  std::string msg;
  if (gemslr_setup(A, prm, op, &msg)) {
    std::printf("%s: setup failed: %s\n", name.c_str(), msg.c_str());
    return false;
  }
  return check_op(name, op, shorter);
}

// n rows: the diagonal, and entries of the last row in the given columns (upper:
// of the first row, in the columns after them).
Csr<double> one_long_row(int n, const std::vector<int>& cols, bool upper) {
  Csr<double> A;
  A.nrows = A.ncols = n;
  A.ia.resize(n + 1, 0);
  for (int i = 0; i < n; ++i) {
    if (upper && i == 0) {
      A.ja.push_back(0);
      A.a.push_back(4.0);
      for (int c : cols) {
        A.ja.push_back(c + 1);
        A.a.push_back(-1.0 - 0.1 * c);
      }
    } else {
      if (!upper && i == n - 1)
        for (int c : cols) {
          A.ja.push_back(c);
          A.a.push_back(-1.0 - 0.1 * c);
        }
      A.ja.push_back(i);
      A.a.push_back(4.0);
    }
    A.ia[i + 1] = (int)A.ja.size();
  }
  return A;
}

}  // namespace

int main() {
  bool ok = true;
  // windows shorter than a step of 32 rows: the last row reads row 33 - w and row 31
  for (int w : {2, 5, 15, 16, 17, 20, 31})
    for (bool upper : {false, true}) {
      std::vector<int> cols = {33 - w};
      if (w > 2) cols.push_back(31);
      ok = run("one long row, window " + std::to_string(w) + (upper ? " (U)" : " (L)"), one_long_row(33, cols, upper), 1,
               1, 1e-6, 20, false) && ok;
    }
  ok = run("diagonal", one_long_row(70, {}, false), 1, 1, 1e-6, 20, false) && ok;
  // level sets of the coarser levels read the rows just before them
  ok = run("laplacian 100x100", laplacian<double>(100, 100, 1, 0.0, 0.0, 0.0, 0.0), 3, 4, 1e-3, 20) && ok;
  ok = run("laplacian 24^3", laplacian<double>(24, 24, 24, 0.0, 0.0, 0.0, 0.0), 3, 8, 1e-3, 20) && ok;
  ok = run("convdiff 20^3", convdiff_upwind(20, 20, 20, 0.3), 2, 4, 1e-2, 10) && ok;
  ok = run("complex laplacian 16^3", laplacian<zdouble>(16, 16, 16, zdouble(0.2, 0.02), 0.05, -0.02, 0.01), 3, 4, 1e-3,
           20) && ok;
  // controls: a ring one row too short must break the replay
  const bool c1 = run("control 24^3", laplacian<double>(24, 24, 24, 0.0, 0.0, 0.0, 0.0), 3, 8, 1e-3, 20, true, 1);
  const bool c2 = run("control one long row", one_long_row(33, {13, 31}, false), 1, 1, 1e-6, 20, false, 13);
  std::printf("%s\n", c1 || c2 ? "CONTROL NOT DETECTED" : "controls detected");
  ok = ok && !c1 && !c2;
  std::printf("%s\n", ok ? "all levels agree" : "MISMATCH");
  return ok ? 0 : 1;
}
