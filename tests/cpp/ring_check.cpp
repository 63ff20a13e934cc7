// Host replay of the ring solve from the arrays that the upload sends.
//
// Every level of a set-up operator is packed as the upload packs it (ring_pack)
// and solved from those arrays alone, as the ring kernel does: a group of 16
// rows' records copied to a stage piece by piece, lanes' entries and ring slots
// read from it, a row's own slot and id from its info pair, steps from their
// boundaries (whole and half steps), the value of the row at position p in slot
// p % rows of a ring that holds just the rows the packing asks for.  Nothing orders the
// writes of one step: two waves take its rows, and the lanes of a wave write
// together.  So a step's rows are replayed in both orders, with the reads
// before the writes and row by row, and every replay must give plain
// forward/backward substitution on the block's factors.
//
// usage: ring_check   (exit 0 when every level of every problem agrees)
#include <algorithm>
#include <cmath>
#include <complex>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "../../pargemslr_amd/csrc/host/gemslr_host.hpp"
#include "../../pargemslr_amd/csrc/host/gen.hpp"
#include "../../pargemslr_amd/csrc/host/ring_pack.hpp"
#include "../../pargemslr_amd/csrc/host/trsv_pack.hpp"

using namespace pgs;

namespace {

constexpr int kStepRows = 32;
constexpr int kMaxWindow = 8192;

template <typename V>
constexpr bool is_single = std::is_same<V, float>::value || std::is_same<V, std::complex<float>>::value;

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

// The lanes' view of a group's records: copied to a stage as the copying wave
// does (piece i of 4 n lanes from byte i * 64 n of the group to byte i * 1024 of
// the stage), read as a solving lane does.
template <typename V>
struct Stage {
  std::vector<unsigned char> bytes = std::vector<unsigned char>(16 * ring_row_bytes<V>(), 0);
  Stage(const unsigned char* group, int n) {
    constexpr int full = sizeof(V) == 4 ? 2 : sizeof(V) == 8 ? 3 : 6;  // pieces of 16 bytes a lane
    for (int i = 0; i < full; ++i) std::memcpy(&bytes[i * 1024], group + i * 64 * n, 64 * n);
    if (sizeof(V) == 8) std::memcpy(&bytes[3 * 1024], group + 3 * 64 * n, 16 * n);
  }
  template <typename X>
  X get(int at) const {
    X x;
    std::memcpy(&x, &bytes[at], sizeof(X));
    return x;
  }
  V value(int lane, int e) const {
    if (sizeof(V) == 4) return get<V>(e < 4 ? lane * 16 + 4 * e : 1024 + lane * 16);
    if (sizeof(V) == 8) return get<V>((e / 2) * 1024 + lane * 16 + (e % 2) * 8);
    return get<V>(e * 1024 + lane * 16);
  }
  int slot(int lane, int e) const {
    const int s01 = sizeof(V) == 4 ? 1024 + lane * 16 + 4 : sizeof(V) == 8 ? 2048 + lane * 16 + 8 : 5 * 1024 + lane * 16;
    const int s4 = sizeof(V) == 8 ? 3 * 1024 + lane * 4 : s01 + 8;
    return e < 4 ? get<uint16_t>(s01 + 2 * e) : (int)(get<uint32_t>(s4) & 0xffff);
  }
};

// One block: pos its step boundaries, nL of its nsteps steps in the L sweep, q0
// its first position.
template <typename V, typename T>
void ring_solve(const RingPack<V>& R, const int* pos, int nL, int nsteps, int64_t q0, const RingInfo* info,
                const T* dinv, const T* rhs, T* x, Order o) {
  std::vector<T> ring(R.rows, T(0.0));
  for (int s = 0; s < nsteps; ++s) {
    const bool upper = s >= nL;
    const int p0 = pos[s], n = pos[s + 1] - p0;
    std::vector<Stage<V>> st;
    for (int g = 0; g < n; g += 16)
      st.emplace_back(R.rec.data() + (q0 + p0 + g) * ring_row_bytes<V>(), std::min(16, n - g));
    std::vector<T> v(n);
    auto solve = [&](int t) {
      T acc = T(0.0);
      for (int q = 0; q < 4; ++q)
        for (int e = 0; e < 5; ++e) {
          const int lane = 4 * (t % 16) + q;
          acc += T(st[t / 16].value(lane, e)) * ring[st[t / 16].slot(lane, e)];
        }
      const int row = info[p0 + t].row;
      v[t] = (upper ? x[row] : rhs[row]) - acc;
      if (upper) v[t] *= dinv[q0 + p0 + t];
    };
    auto write = [&](int t) {
      const RingInfo i = info[p0 + t];
      ring.at(i.slot / sizeof(V)) = v[t];
      x[i.row] = v[t];
    };
    auto each = [&](auto f) {
      for (int t = 0; t < n; ++t) f(o.reversed ? n - 1 - t : t);
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

// Replays every level with the device's values in V; `shorter` takes rows off
// the ring (a control).
template <typename V, typename T>
bool check_op(const std::string& name, const HostOp<T>& op, int shorter) {
  bool ok = true;
  const double tol = is_single<V> ? 1e-5 : 1e-12;
  for (int l = 0; l < op.nlev; ++l) {
    const HostLevel<T>& L = op.levels[l];
    const int nl = op.nloc(l);
    TrsvPack<T> P = trsv_pack(L, op.lev_ptr[l], nl, kStepRows, kMaxWindow, kRingWidth);
    if (P.window == 0) {
      std::printf("%s level %d: not ring-packed MISMATCH\n", name.c_str(), l);
      ok = false;
      continue;
    }
    P.window_needed -= shorter;
    const RingPack<V> R = ring_pack<V>(P, [](const T& v) { return V(v); });
    int longest = 0;
    for (size_t i = 2; i < P.desc.size(); i += 4) longest = std::max(longest, P.desc[i]);
    std::vector<double> g(2 * (size_t)nl);
    rng_normal(1000 + l, 2 * (int64_t)nl, g.data());
    std::vector<T> rhs(nl), ref(nl), x(nl);
    for (int i = 0; i < nl; ++i) rhs[i] = value_of<T>(g[2 * i], g[2 * i + 1]);
    double emax = 0.0, nmax = 0.0;
    for (int b = 0; b < L.ncomp; ++b) {
      const int r0 = P.blk_row0[b], nb = P.blk_row0[b + 1] - r0;
      block_solve(L.ilu[b], rhs.data() + r0, ref.data() + r0);
      // lanes past a step's rows take the dummy row's pair, right after the block's own
      const int64_t np = P.blk_ri0[b + 1] - P.blk_ri0[b];
      const RingInfo* info = R.info.data() + ring_info0(P.blk_ri0[b], b);
      if (info[np].slot != R.rows * (int)sizeof(V) || info[np].row != kRingDummyRow || (info - R.info.data()) % 2) {
        std::printf("%s, level %d, block %d: no dummy pair, or pairs not aligned MISMATCH\n", name.c_str(), l, b);
        ok = false;
      }
      for (int k = 0; k < 8; ++k) {
        const Order o = {(k & 1) != 0, (k & 2) != 0};
        const bool half = (k & 4) != 0;
        const int s0 = half ? R.step_h[b] : P.blk_step[b], s1 = half ? R.step_h[b + 1] : P.blk_step[b + 1];
        const int sU = half ? R.stepU_h[b] : P.blk_stepU[b];
        ring_solve<V>(R, (half ? R.pos_h : R.pos).data() + s0 + b, sU - s0, s1 - s0, P.blk_ri0[b], info,
                      P.dinv.data(), rhs.data() + r0, x.data() + r0, o);
        for (int i = r0; i < r0 + nb; ++i) {
          nmax = std::max(nmax, std::abs(ref[i]));
          const double e = std::abs(x[i] - ref[i]);
          emax = e <= emax ? emax : e;  // a NaN stays
        }
      }
    }
    const double rel = nmax > 0.0 ? emax / nmax : emax;
    const bool good = rel <= tol;
    std::printf("%s, %d-byte values, level %d: %d blocks, longest step %d rows, ring %d rows%s, rel err %.2e %s\n",
                name.c_str(), (int)sizeof(V), l, L.ncomp, longest, R.rows, shorter ? " (shortened)" : "", rel,
                good ? "ok" : "MISMATCH");
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
  bool ok = check_op<T>(name, op, shorter);
  if constexpr (is_complex<T>::value) ok = check_op<std::complex<float>>(name, op, shorter) && ok;
  else ok = check_op<float>(name, op, shorter) && ok;
  return ok;
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
  // limits of the 32-bit offsets are a block's, whatever its level holds: the
  // largest blocks (FP32, FP64, complex128) and one row more, a block's vectors
  ok = ring_offsets_fit<float>(8388607, 64) && !ring_offsets_fit<float>(8388608, 1) && ok;
  ok = ring_offsets_fit<double>(5162220, 32) && !ring_offsets_fit<double>(5162221, 1) && ok;
  ok = ring_offsets_fit<zdouble>(2796202, 32) && !ring_offsets_fit<zdouble>(2796203, 1) && ok;
  ok = ring_offsets_fit<double>(4194303, 64) && !ring_offsets_fit<double>(4194304, 64) && ok;
  // controls: a ring one row too short must break the replay
  const bool c1 = run("control 24^3", laplacian<double>(24, 24, 24, 0.0, 0.0, 0.0, 0.0), 3, 8, 1e-3, 20, true, 1);
  const bool c2 = run("control one long row", one_long_row(33, {13, 31}, false), 1, 1, 1e-6, 20, false, 13);
  std::printf("%s\n", c1 || c2 ? "CONTROL NOT DETECTED" : "controls detected");
  ok = ok && !c1 && !c2;
  std::printf("%s\n", ok ? "all levels agree" : "MISMATCH");
  return ok ? 0 : 1;
}
