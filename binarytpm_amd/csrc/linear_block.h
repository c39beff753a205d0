// linear_block.h -- eight explicit conduction steps of a column as one matrix
// product on the matrix cores.
//
// Between two surface balances the explicit step is linear in the 55 interior
// nodes, so the nodes after the 8 steps of a time block are
//     nodes' = P^8 nodes + sum_j H_j u0(j),     j = 0..7,
// with u0(j) the surface offset before step j of the block, and node 1, the
// only node the surface balance of a step reads, is after s steps
//     u1(s) = base(s) + sum_{j < s} g(s-1-j) u0(j),
// base(s) being the part due to the nodes at the block's start.  base(1..8)
// of the NEXT block is again linear in (nodes, u0(0..7)), so one 64 x 64
// product per block gives both: 55 nodes + 8 surface values in, 55 nodes + 8
// responses out (one spare).  A step then costs the surface balance and at
// most 8 FMAs (36 a block) instead of 110 vector instructions.
//
// Layout.  The product runs on v_mfma_f32_16x16x32_f16: lane l supplies
// A[m = l%16][k = 8(l/16)+j] and B[k = 8(l/16)+j][n = l%16], j < 8, and
// receives D[m = 4(l/16)+i][n = l%16], i < 4.  A tile of 16 columns is held
// as u[16] per lane, lane (g = l/16, c = l%16) the 16 slots q of group g of
// column c.  Slot (g, q) is row 4(q/4).. of output tile t = q/4 and K entry of
// input chunk h = q/8, so the product's output is the next product's input
// without moving between lanes.  Which node a slot holds is free; with
//     tile 0: q = 0, 1: u0(2g + q) in, base(2g + q + 1) out;
//             q = 2, 3: node 1 + 2g + (q - 2)
//     tile t > 0:       node 9 + 16(t-1) + 4g + (q - 4t)
// the 17-wide band of P^8 leaves the blocks (tile 0, chunk 1) and (tile 3,
// chunk 0) empty: 6 of 8 blocks are stored and multiplied.
//
// Precision.  A node's own entry is nearly one when the FTCS number r is
// small; what the product forms is the rest of the row,
//     node' = c node + sum_j M_j entry_j,   M = P^8 - c I | H,
// c the diagonal of an interior row in FP32, added by one FMA, so that the
// product's rounding is that of the change over a block (about 16 r of the
// node) and the node itself is rounded once.  M and the columns are split
// x = hi + lo in fp16 and multiplied as hi hi + hi lo + lo hi with FP32
// accumulation.  The matrix instruction cuts each of 8 products toward zero at
// 2^-26 of the largest (by exponents) and its accumulator downward at 2^-26 of
// them: one-sided, and what is one-sided adds up over the blocks.  So the large
// products come first, and the hi halves of a row are whole multiples of 2^-15
// of its largest power of two: products of columns alike in size are then not
// cut at all.  M is scaled by 2^15 so that its low halves stay normal numbers.
// The rounding of the low halves is made up on entries far from the node, whose
// halves are finer: constants and linear profiles stay so (row sums to 4e-9,
// first moments to 5e-7).  Columns are held multiplied by 2^15 (as the product
// leaves them).  Errors against FP64 after 30 rotations, thermal inertias 20 to
// 1000, in 1e-6 K rms of the surface / of all nodes, eight FP32 steps in
// brackets:
//   r 0.474   6.9 /  6.9  (7.2 /  6.9)      r 0.015   7.4 / 12.2  (7.8 / 12.0)
//   r 0.126   7.1 /  7.7  (7.1 /  7.3)      r 0.0047  7.2 / 14.1  (7.7 / 14.8)
//   r 0.030   7.4 / 10.6  (7.5 / 10.5)      r 0.0005  7.7 / 12.3  (8.7 / 13.0)
// (P^8 whole in M, small products first: 40 to 60 for all nodes at r 0.03 to
// 0.005.)
#pragma once

#include <hip/hip_runtime.h>

#include "btpm_device.h"
#include "btpm_internal.h"

namespace btpm_lin {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr float kScale = 32768.0f;
constexpr int kFrags = 12;              // 6 blocks x (hi, lo), 64 lanes x 8 halves each
constexpr int kFrag = 64 * 8;           // halves per fragment
// an operator in memory (halves): main[12], tail[12] (the last block's steps),
// init[2] (base(1..8) of the first block from the nodes), then floats g[8] and
// the c of main and tail
constexpr int kTail = kFrags * kFrag;
constexpr int kInit = 2 * kFrags * kFrag;
constexpr int kGain = kInit + 2 * kFrag;
constexpr int kOwn = kGain + 2 * BTPM_BLK;
static_assert(kOwn + 4 <= BTPM_LIN_OP, "operator size");

// block b of the product: output tile and input chunk
constexpr int kBlkTile[6] = {0, 1, 1, 2, 2, 3};
constexpr int kBlkChunk[6] = {0, 0, 1, 0, 1, 1};

// node held by slot q of group g (0: a surface slot)
__device__ __forceinline__ int slot_node(int g, int q) {
  return q < 2 ? 0 : q < 4 ? 1 + 2 * g + (q - 2) : 9 + 16 * (q / 4 - 1) + 4 * g + (q & 3);
}

// fp16 hi / lo halves of 2^-15 x, two at a time: the empty asm keeps the hi
// pair packed, so that the low halves are taken from it in place
__device__ __forceinline__ void split2(float x, float y, h2& hi, h2& lo) {
  hi = h2{(_Float16)fmaf(x, 1.0f / kScale, 0.0f), (_Float16)fmaf(y, 1.0f / kScale, 0.0f)};
  asm("" : "+v"(hi));
  lo = h2{(_Float16)fmaf(x, 1.0f / kScale, -(float)hi.x),
          (_Float16)fmaf(y, 1.0f / kScale, -(float)hi.y)};
}
// the 8 slots of input chunk h
__device__ __forceinline__ void split_chunk(const float (&u)[16], int h, h8& hi, h8& lo) {
  h2 a[4], b[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) split2(u[8 * h + 2 * j], u[8 * h + 2 * j + 1], a[j], b[j]);
  hi = h8{a[0].x, a[0].y, a[1].x, a[1].y, a[2].x, a[2].y, a[3].x, a[3].y};
  lo = h8{b[0].x, b[0].y, b[1].x, b[1].y, b[2].x, b[2].y, b[3].x, b[3].y};
}

// u <- operator u for NT tiles of 16 columns; frag(i) gives fragment i (block
// i/2, hi then lo) of the lane, own is c
template <int NT, class Frag>
__device__ __forceinline__ void linear_block(float (&u)[NT][16], float own, Frag frag) {
  h8 bh[NT][2], bl[NT][2];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int h = 0; h < 2; ++h) split_chunk(u[t], h, bh[t][h], bl[t][h]);
#pragma unroll
  for (int ot = 0; ot < 4; ++ot) {
    f4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    h8 ahi[2], alo[2];
#pragma unroll
    for (int b = 0; b < 6; ++b)
      if (kBlkTile[b] == ot) {
        ahi[kBlkChunk[b]] = frag(2 * b);
        alo[kBlkChunk[b]] = frag(2 * b + 1);
      }
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
      for (int b = 0; b < 6; ++b)
        if (kBlkTile[b] == ot)
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            const int h = kBlkChunk[b];
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(p == 2 ? alo[h] : ahi[h],
                                                            p == 1 ? bl[t][h] : bh[t][h], acc[t],
                                                            0, 0, 0);
          }
    // (tile 0, i < 2: a surface slot)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        u[t][4 * ot + i] = ot == 0 && i < 2 ? acc[t][i] : fmaf(own, u[t][4 * ot + i], acc[t][i]);
  }
}

// four tiles, two at a time: half the registers for the split columns
template <class Frag>
__device__ __forceinline__ void linear_block_pairs(float (&u)[4][16], float own, Frag frag) {
  linear_block<2>(*reinterpret_cast<float (*)[2][16]>(&u[0]), own, frag);
  asm volatile("" ::: "memory");
  linear_block<2>(*reinterpret_cast<float (*)[2][16]>(&u[2]), own, frag);
}

// base(1..8) of a rotation's first block from the nodes (surface slots zero)
template <int NT>
__device__ __forceinline__ void linear_init(float (&u)[NT][16], h8 ahi, h8 alo) {
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    h8 bh, bl;
    split_chunk(u[t], 0, bh, bl);
    f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi, bh, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi, bl, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(alo, bh, acc, 0, 0, 0);
    u[t][0] = acc[0];
    u[t][1] = acc[1];
  }
}

__device__ __forceinline__ void swap32(float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false,
                                                  false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void swap16(float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false,
                                                  false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
// transposes (register i, lane group g) of four registers; its own inverse
__device__ __forceinline__ void transpose4(float& x0, float& x1, float& x2, float& x3) {
  swap32(x0, x2);
  swap32(x1, x3);
  swap16(x0, x1);
  swap16(x2, x3);
}

// Surface slots <-> one column per lane: lane group g takes the 8 surface
// values of its column of tile g % NT (with NT = 4 every lane its own column,
// with NT = 2 and 1 two and four lanes the same).
__device__ __forceinline__ void surface_out(const float (&u)[4][16], float (&w)[8]) {
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    float x0 = u[0][q], x1 = u[1][q], x2 = u[2][q], x3 = u[3][q];
    transpose4(x0, x1, x2, x3);
    w[q] = x0;
    w[2 + q] = x1;
    w[4 + q] = x2;
    w[6 + q] = x3;
  }
}
__device__ __forceinline__ void surface_in(float (&u)[4][16], const float (&w)[8]) {
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    float x0 = w[q], x1 = w[2 + q], x2 = w[4 + q], x3 = w[6 + q];
    transpose4(x0, x1, x2, x3);
    u[0][q] = x0;
    u[1][q] = x1;
    u[2][q] = x2;
    u[3][q] = x3;
  }
}
__device__ __forceinline__ void surface_out(const float (&u)[2][16], float (&w)[8]) {
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    float a = u[0][q], b = u[1][q];
    swap16(a, b);  // a: tiles 0, 1 from group 0, then from group 2; b: 1, then 3
    float a2 = a, b2 = b;
    swap32(a, a2);
    swap32(b, b2);
    w[q] = a;
    w[2 + q] = b;
    w[4 + q] = a2;
    w[6 + q] = b2;
  }
}
__device__ __forceinline__ void surface_in(float (&u)[2][16], const float (&w)[8]) {
  const bool hi = (threadIdx.x & 32) != 0;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    float a = hi ? w[4 + q] : w[q], b = hi ? w[6 + q] : w[2 + q];
    swap16(a, b);
    u[0][q] = a;
    u[1][q] = b;
  }
}
__device__ __forceinline__ void surface_out(const float (&u)[1][16], float (&w)[8]) {
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    float a = u[0][q], b = a;
    swap32(a, b);  // a: groups 0, 1 twice; b: groups 2, 3 twice
    float a2 = a, b2 = b;
    swap16(a, a2);
    swap16(b, b2);
    w[q] = a;
    w[2 + q] = a2;
    w[4 + q] = b;
    w[6 + q] = b2;
  }
}
__device__ __forceinline__ void surface_in(float (&u)[1][16], const float (&w)[8]) {
  const int g = (int)(threadIdx.x & 63) >> 4;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const float lo = (g & 1) ? w[2 + q] : w[q];
    const float hi = (g & 1) ? w[6 + q] : w[4 + q];
    u[0][q] = (g & 2) ? hi : lo;
  }
}

// The surface balances of a block's 8 steps for one column per lane (or copies
// of it).  In: w = base(1..8), tot = the absorbed flux of each step, tp = the
// previous rotation's surface temperatures; out: w = the surface offset before
// each step (x 2^15), tp = this rotation's temperatures.
//
// The Newton start of a step is the previous rotation's temperature at this
// step shifted by the difference between the two rotations, extrapolated
// linearly from the steps two and three back.  Taking it from there rather
// than from the step just solved leaves only
//   u0 -> node 1 -> first iterate
// (six dependent operations) between consecutive steps: the derivative, its
// reciprocal and the start's residual are formed during the step before.  The
// start only decides how many iterations a column takes, never where it stops.
struct Surface {
  float u0;           // surface offset x 2^15
  float d1, d2, d3;   // T - T_prev one, two and three steps back
  float dm;           // max |T - T_prev| of the rotation
};

// beside(k) is work of the caller's that does not depend on the steps, placed
// beside step k.
template <bool FULL, class Beside>
__device__ __forceinline__ void surface_steps(Surface& s, float (&w)[8], float (&tp)[8],
                                              const float (&tot)[8], const float (&gain)[8],
                                              double m1, double es, double Tref, double tol, int cap,
                                              int kend, Beside beside) {
  // constants held in registers: as literals they cost a move at every use
  double up = (double)kScale, down = 1.0 / (double)kScale;
  asm volatile("" : "+s"(up), "+s"(down));
  const double Trefs = -Tref * up;  // exact: a power of two
  auto start = [&](int k, float a, float b) {  // a, b: differences two and three steps back
    btpm_dev::FirstIterate f = btpm_dev::newton_first(
        (double)(tp[k] + (3.0f * a - 2.0f * b)), (double)tot[k], m1, es);
    return f;
  };
  btpm_dev::FirstIterate f = start(0, s.d2, s.d3);
#pragma unroll
  for (int k = 0; k < BTPM_BLK; ++k) {
    if (!FULL && k >= kend) {
      w[k] = 0.0f;
      continue;
    }
    beside(k);
#pragma unroll
    for (int kk = k; kk < BTPM_BLK; ++kk) w[kk] = fmaf(gain[kk - k], s.u0, w[kk]);
    const double t1 = fma((double)w[k], down, Tref);
    w[k] = s.u0;  // the surface value before this step, an input of the product
    double x = fma(f.b, t1, f.a);
    const double d0 = x - f.x0;
    btpm_dev::FirstIterate next = f;
    if (k + 1 < BTPM_BLK) {
      next = start(k + 1, s.d1, s.d2);
      // formed here, beside this step's chain, not behind the branch below
      asm volatile("" : "+v"(next.x0), "+v"(next.a), "+v"(next.b));
#pragma unroll
      for (int kk = k + 1; kk < BTPM_BLK; ++kk) asm volatile("" : "+v"(w[kk]));
    }
    if (__builtin_expect(__ballot(!(fabs(d0) < tol)) != 0, 0))  // a column needs another iteration
      x = btpm_dev::newton_finish(fma(m1, t1, (double)tot[k]), m1, es, x, d0, tol, cap);
    f = next;
    s.u0 = (float)fma(x, up, Trefs);
    const float t = (float)x;
    s.d3 = s.d2;
    s.d2 = s.d1;
    s.d1 = t - tp[k];
    s.dm = fmaxf(s.dm, fabsf(s.d1));
    tp[k] = t;
  }
}

// One tile's nodes from / to profile records (57 nodes, offsets from tref)
typedef float uf4 __attribute__((ext_vector_type(4), aligned(4)));
typedef float uf2 __attribute__((ext_vector_type(2), aligned(4)));
typedef __attribute__((address_space(1))) float gf;

__device__ __forceinline__ void load_nodes(const gf* rec, int g, float tref, float (&u)[16]) {
  const uf2 a = *reinterpret_cast<const __attribute__((address_space(1))) uf2*>(rec + 1 + 2 * g);
  u[0] = u[1] = 0.0f;
  u[2] = (a.x - tref) * kScale;
  u[3] = (a.y - tref) * kScale;
#pragma unroll
  for (int t = 1; t < 4; ++t) {
    const uf4 v = *reinterpret_cast<const __attribute__((address_space(1))) uf4*>(
        rec + 9 + 16 * (t - 1) + 4 * g);
#pragma unroll
    for (int i = 0; i < 4; ++i) u[4 * t + i] = (v[i] - tref) * kScale;
  }
}
// (node 56 is written as the copy of node 55, the zero-flux bottom)
__device__ __forceinline__ void store_nodes(gf* rec, int g, float tref, const float (&u)[16]) {
  auto node = [&](float x) { return fmaf(x, 1.0f / kScale, tref); };
  *reinterpret_cast<__attribute__((address_space(1))) uf2*>(rec + 1 + 2 * g) =
      uf2{node(u[2]), node(u[3])};
#pragma unroll
  for (int t = 1; t < 4; ++t) {
    uf4 v = {node(u[4 * t]), node(u[4 * t + 1]), node(u[4 * t + 2]), node(u[4 * t + 3])};
    if (t == 3 && g == 3) v[3] = v[2];
    *reinterpret_cast<__attribute__((address_space(1))) uf4*>(rec + 9 + 16 * (t - 1) + 4 * g) = v;
  }
}

}  // namespace btpm_lin
