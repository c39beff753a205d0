// linear_op.hip -- host side of linear_block.h: the matrices of eight explicit
// conduction steps for one FTCS number, split and packed as the fragments the
// matrix instructions read.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>

#include "linear_block.h"
#include "runtime.h"

namespace btpm {
namespace {
constexpr int N = BTPM_NX - 1;       // interior nodes 1..55
constexpr int B = BTPM_BLK;
constexpr int L = N + B;             // inputs: nodes, then u0(0..7); outputs: nodes, base(1..8)

// entry of a slot: node - 1, or N + surface index, or -1 (node 56)
int slot_entry(int g, int q) {
  if (q < 2) return N + 2 * g + q;
  const int n = q < 4 ? 1 + 2 * g + (q - 2) : 9 + 16 * (q / 4 - 1) + 4 * g + (q & 3);
  return n <= N ? n - 1 : -1;
}

// u[node - 1][entry]: the nodes as functions of the entries
using Nodes = double[N][L];

// one FTCS step of the nodes, entry by entry, with surface value s[entry]
// (node 0) and the zero-flux bottom u[NX] = u[NX-1]
void ftcs(Nodes& u, double r, const double (&s)[L]) {
  double before[L], cur[L];
  std::memcpy(before, s, sizeof before);
  for (int i = 0; i < N; ++i) {
    std::memcpy(cur, u[i], sizeof cur);
    const double* next = i + 1 < N ? u[i + 1] : cur;
    for (int e = 0; e < L; ++e) u[i][e] = cur[e] + r * (next[e] - 2.0 * cur[e] + before[e]);
    std::memcpy(before, cur, sizeof before);
  }
}

// out[row][entry] of `steps` steps: nodes after them and, with `responses`,
// node 1 after 1..8 further steps without surface input
void respond(double r, int steps, bool responses, double (&out)[L][L]) {
  std::memset(out, 0, sizeof out);
  Nodes u = {};
  for (int i = 0; i < N; ++i) u[i][i] = 1.0;
  for (int k = 0; k < steps; ++k) {
    double s[L] = {0.0};
    s[N + k] = 1.0;
    ftcs(u, r, s);
  }
  std::memcpy(out, u, sizeof u);
  if (!responses) return;
  const double none[L] = {0.0};
  for (int s = 0; s < B; ++s) {
    ftcs(u, r, none);
    std::memcpy(out[N + s], u[0], sizeof u[0]);
  }
}

// takes the diagonal c of an interior row off the node rows; returns it
float take_own(double (&m)[L][L]) {
  const float c = (float)m[N / 2][N / 2];
  for (int i = 0; i < N; ++i) m[i][i] -= (double)c;
  return c;
}

// hi and lo of every entry times 2^15.  The hi halves of a row are whole
// multiples of 2^-15 of its largest power of two.  The error of a row's sum and
// of its first moment about the row's node (entries at their nodes, surface
// values at node 0), left by rounding the low halves, are then made up on two
// entries at a distance d to either side, d = 1..8: those of the far entries,
// which are small and so are their units, are exact enough.  What is left of
// the sum goes to the row's smallest entry.
void split_rows(const double (&m)[L][L], _Float16 (&hi)[L][L], _Float16 (&lo)[L][L]) {
  std::memset(hi, 0, sizeof hi);
  std::memset(lo, 0, sizeof lo);
  auto pos = [](int j) { return j < N ? j + 1 : 0; };
  for (int i = 0; i < L; ++i) {
    double top = 0.0;
    int least = -1;
    for (int j = 0; j < L; ++j) {
      const double a = std::fabs(m[i][j]);
      top = std::fmax(top, a);
      if (a > 0.0 && (least < 0 || a < std::fabs(m[i][least]))) least = j;
    }
    if (least < 0) continue;
    int e;
    std::frexp(top * btpm_lin::kScale, &e);
    const double unit = std::ldexp(1.0, e - 15);
    for (int j = 0; j < L; ++j) {
      if (m[i][j] == 0.0) continue;
      const double x = m[i][j] * btpm_lin::kScale;
      double h = (double)(_Float16)x;
      if (std::fabs(h) < 2048.0 * unit) h = (double)(_Float16)(std::rint(x / unit) * unit);
      hi[i][j] = (_Float16)h;
      lo[i][j] = (_Float16)(x - h);
    }
    const int at = i < N ? i + 1 : 1;
    double sum = 0.0, mom = 0.0;
    for (int j = 0; j < L; ++j) {
      if (m[i][j] == 0.0) continue;
      const double err = (double)hi[i][j] + (double)lo[i][j] - m[i][j] * btpm_lin::kScale;
      sum += err;
      mom += err * (pos(j) - at);
    }
    auto change = [&](int j, double by) {
      const double was = (double)lo[i][j];
      lo[i][j] = (_Float16)(was + by);
      const double d = (double)lo[i][j] - was;
      sum += d;
      mom += d * (pos(j) - at);
    };
    for (int d = 1; d <= B; ++d) {
      const int p = at > d ? at - d - 1 : N, q = std::min(at + d, N) - 1;
      if (m[i][p] == 0.0 || m[i][q] == 0.0 || pos(p) == pos(q)) continue;
      const double dp = pos(p) - at, dq = pos(q) - at;
      const double b = (sum * dp - mom) / (dq - dp), a = -sum - b;
      change(p, a);
      change(q, b);
    }
    change(least, -sum);
  }
}

// the fragment pair (hi, lo) of output tile t and input chunk h
void pack(const _Float16 (&hi)[L][L], const _Float16 (&lo)[L][L], int t, int h, _Float16* out) {
  for (int lane = 0; lane < 64; ++lane)
    for (int j = 0; j < 8; ++j) {
      const int m = lane & 15;
      const int row = slot_entry(m >> 2, 4 * t + (m & 3)), col = slot_entry(lane >> 4, 8 * h + j);
      const bool in = row >= 0 && col >= 0;
      out[lane * 8 + j] = in ? hi[row][col] : (_Float16)0.0f;
      out[btpm_lin::kFrag + lane * 8 + j] = in ? lo[row][col] : (_Float16)0.0f;
    }
}
}  // namespace

void linear_operator(float rf, int ntau, _Float16* op) {
  const double r = (double)rf;
  static thread_local double m[L][L];
  static thread_local _Float16 hi[L][L], lo[L][L];
  std::fill(op, op + BTPM_LIN_OP, (_Float16)0.0f);
  float own[2];
  respond(r, B, true, m);
  own[0] = take_own(m);
  split_rows(m, hi, lo);
  for (int b = 0; b < 6; ++b) pack(hi, lo, btpm_lin::kBlkTile[b], btpm_lin::kBlkChunk[b], op + 2 * b * btpm_lin::kFrag);
  // the last block's steps: nodes only
  respond(r, ntau - (nblocks(ntau) - 1) * B, false, m);
  own[1] = take_own(m);
  split_rows(m, hi, lo);
  for (int b = 0; b < 6; ++b)
    pack(hi, lo, btpm_lin::kBlkTile[b], btpm_lin::kBlkChunk[b], op + btpm_lin::kTail + 2 * b * btpm_lin::kFrag);
  // base(1..8) of the first block from the nodes (no steps before it)
  respond(r, 0, true, m);
  std::memset(m, 0, N * sizeof m[0]);
  split_rows(m, hi, lo);
  pack(hi, lo, 0, 0, op + btpm_lin::kInit);
  // g(k): node 1, k + 1 steps after a unit surface value
  float g[B];
  Nodes u = {};
  for (int k = 0; k < B; ++k) {
    double x[L] = {0.0};
    x[0] = k == 0 ? 1.0 : 0.0;
    ftcs(u, r, x);
    g[k] = (float)u[0][0];
  }
  std::memcpy(op + btpm_lin::kGain, g, sizeof g);
  std::memcpy(op + btpm_lin::kOwn, own, sizeof own);
}
}  // namespace btpm
