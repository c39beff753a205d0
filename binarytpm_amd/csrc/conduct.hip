// conduct.hip -- persistent per-rotation conduction kernels for gfx950.
//
// One launch advances every listed tile by one full rotation (ntau steps):
// the 57-node depth profile of each column lives in VGPRs for the whole
// rotation, inputs/outputs stream through HBM in 8-step blocks (blocked SoA,
// see btpm_internal.h) with the next block prefetched while the current one
// is integrated, and the per-column rotation-to-rotation change is reduced
// in-kernel for the freeze test.
//
// Algorithm per column and step (the reference's inertiadifference,
// T175706/thermal.cpp:1895-1979, and the crater kernels finite_difference +
// boundary_condition, T175706/thermal_GPU.cu:430-574):
//   FTCS   T_i += r (T_{i+1} - 2 T_i + T_{i-1}),  i = 1..NX-1 (old values)
//   bottom T_NX = T_{NX-1}
//   SBC    Newton on (1-A)F + Q + m1 (T_1 - T_0) - es T_0^4 = 0 from the old
//          T_0 until |dT| < tol, in FP64
// where Q (self-heating) always uses the PREVIOUS rotation's surface
// temperatures at the same step.
//
// Precision: the profile is held as offsets u_i = T_i - T_ref with a
// per-column reference T_ref (the bottom node at rotation start).  The FTCS
// operator is exact on constants, so the offsets integrate the same
// recurrence while their FP32 rounding is set by the size of the offsets
// (K) rather than of the absolute temperature (hundreds of K).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "btpm_internal.h"
#include "btpm_kernels.h"
#include "btpm_device.h"
#include "linear_block.h"

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
// Pointers read from the set descriptor are generic; casting them to the
// global address space lets the compiler emit global (not flat) memory ops,
// whose completion is tracked by vmcnt alone so prefetches stay in flight.
#define GLOBAL_AS __attribute__((address_space(1)))
typedef GLOBAL_AS float gfloat;
typedef float float4_t __attribute__((ext_vector_type(4)));

namespace {

// FTCS in scaled form.  With c = 1 - 2r the step is u_i' = c u_i + r (u_{i-1}
// + u_{i+1}); holding U = u / s with s = c^k after k steps turns it into
//     U_i' = U_i + kr (U_{i-1} + U_{i+1}),   kr = r / c,
// one add and one FMA accumulated in place per node instead of three
// operations.  The per-step factor is made consistent with the rounded kr as
// sig = 1 / (1 + 2 kr) (so constants stay exactly constant), tracked in FP64
// with its inverse, and folded back into U once per 8-step block (U grows by
// at most c^-8 < 1e32 in between for r <= BTPM_R_MAX); the crater kernel
// folds every 1 to 3 blocks, as rarely as the FP32 range allows for its r.
// The zero-flux bottom is the reference's copy node u[NX] = u[NX-1]: node
// NX-1 sees its own old value in its place, and u[NX] itself is not carried
// (a profile enters with u[NX] = u[NX-1], which every FD step leaves so, and
// leaves through store_profile with the copy).
template <int NX>
__device__ __forceinline__ void ftcs_scaled(float (&u)[NX + 1], float kr) {
  float before = u[0];
#pragma unroll
  for (int i = 1; i < NX - 1; ++i) {
    const float cur = u[i];
    u[i] = fmaf(kr, u[i + 1] + before, cur);
    before = cur;
  }
  const float cur = u[NX - 1];
  u[NX - 1] = fmaf(kr, cur + before, cur);
}

// Per-column scale state of the scaled recurrence: real offset = sd * U.
struct Scale {
  float kr;         // r / (1 - 2r), FP32
  double sig, isig; // per-step factor 1 / (1 + 2 kr) and its inverse (exact)
  double sd, isd;   // current scale and its inverse
};

__device__ __forceinline__ float scaled_kr(float r) { return r / (1.0f - 2.0f * r); }

__device__ __forceinline__ Scale make_scale(float r) {
  Scale sc;
  sc.kr = scaled_kr(r);
  sc.isig = fma(2.0, (double)sc.kr, 1.0);
  sc.sig = 1.0 / sc.isig;
  sc.sd = 1.0;
  sc.isd = 1.0;
  return sc;
}

// Scale of the n steps between two rescales for one r, shared by all columns
// with that r: sk[k] = (sig^(k+1), sig^-(k+1)) in FP32 for the per-step
// conversions and pk[k] = sig^(k+1) in FP64 for the rescale.
__device__ __forceinline__ void scale_table(float r, float2* sk, double* pk, int n) {
  const double isig = fma(2.0, (double)scaled_kr(r), 1.0);
  const double sig = 1.0 / isig;
  double p = 1.0, ip = 1.0;
  for (int k = 0; k < n; ++k) {
    p *= sig;
    ip *= isig;
    sk[k] = make_float2((float)p, (float)ip);
    pk[k] = p;
  }
}

// The crater kernel folds the scale back into the profile every 1 to
// kRescaleMax blocks: as rarely as U <= 1e4 K x sig^-(8 blocks) stays inside
// the FP32 range for every crater of the workgroup (sig = 1 - 2r).
constexpr int kRescaleMax = 3;
__device__ __forceinline__ int rescale_blocks(float r) {
  const double c = 1.0 - 2.0 * (double)r;
  const double c2 = c * c, c4 = c2 * c2, c8 = c4 * c4;
  const double lim = 1e4 / 3.4e38;  // 1e4 K / FLT_MAX
  return c8 * c8 * c8 > lim ? 3 : c8 * c8 > lim ? 2 : 1;
}

// Per-crater constants of the crater kernel, shared by the crater's 100 lanes.
struct CraterConst {
  float2 sk[kRescaleMax * BTPM_BLK];  // scale_table
  double pk[kRescaleMax * BTPM_BLK];
  double r0[2];         // residual of the scale carried from the last rescale
  double m1;            // Gamma sqrt(2 pi n / P) / dz
  double es, tol;       // emissivity x sigma and the Newton tolerance, read from
                        // LDS at each step (held in VGPRs they would cost 4)
};

// Fold the accumulated scale into the profile: U *= f with f = fp32(sd); the
// residual sd / f (within 6e-8 of 1) is carried, so the block-to-block gain
// has no systematic rounding bias.  sd = 1 / isd to second order.
template <int NX>
__device__ __forceinline__ void rescale(float (&u)[NX + 1], Scale& sc) {
  const float f = (float)sc.sd;
#pragma unroll
  for (int i = 0; i < NX; ++i) u[i] *= f;
  sc.isd *= (double)f;
  sc.sd = 2.0 - sc.isd;
}

__device__ __forceinline__ void load8(const gfloat* p, float (&v)[BTPM_BLK]) {
  const GLOBAL_AS float4_t* q = reinterpret_cast<const GLOBAL_AS float4_t*>(p);
  const float4_t a = q[0], b = q[1];
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
  v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}

__device__ __forceinline__ void load4(const gfloat* p, float (&v)[BTPM_BLK], int k0) {
  const float4_t a = *reinterpret_cast<const GLOBAL_AS float4_t*>(p + k0);
  v[k0] = a.x; v[k0 + 1] = a.y; v[k0 + 2] = a.z; v[k0 + 3] = a.w;
}

// FTCS + bottom boundary + FP64 Newton SBC for one step; returns T_0.
// (s, is) is the scale after this step and its inverse (FP32 or FP64): the
// Newton solve sees the real T_1 = Tref + s U_1 and the root goes back into
// the scaled profile as U_0 = (T_0 - Tref) / s.
// The Newton start x0 is a predictor: the previous rotation's surface
// temperature at this step shifted by the difference between the two
// rotations, extrapolated linearly from the two previous steps (the caller's
// dl = t - t_prev at step k-1, dl2 at step k-2: x0 = t_prev + 2 dl - dl2).
template <int NX, typename SC>
__device__ __forceinline__ double conduct_step(float (&u)[NX + 1], float kr, SC s, SC is,
                                               double src, double m1, double es, double Tref,
                                               double tol, int cap, double x0) {
  ftcs_scaled<NX>(u, kr);
  double t1;
  if constexpr (std::is_same<SC, double>::value)
    t1 = fma(s, (double)u[1], Tref);
  else
    t1 = Tref + (double)(s * u[1]);
  // the first Newton iteration is straight-line code next to the FTCS of
  // nodes 2..NX, which do not depend on it: the empty asm statements keep
  // those nodes' updates ahead of the (rarely taken) iteration loop, so the
  // scheduler fills the FP64 chain's latency with them
  const double K = fma(m1, t1, src);
  double x = fmax(x0, 1.0);
  const double d0 = btpm_dev::newton_step(K, m1, es, x);
#pragma unroll
  for (int i = 2; i < NX; ++i) asm volatile("" : "+v"(u[i]));
  x = btpm_dev::newton_finish(K, m1, es, x, d0, tol, cap);
  if constexpr (std::is_same<SC, double>::value)
    u[0] = (float)((x - Tref) * is);
  else
    u[0] = (float)(x - Tref) * is;
  return x;
}

// profile of one column: 57 nodes in a 64-float record (one base address,
// immediate offsets), held as offsets from its bottom node
template <int NX>
__device__ __forceinline__ float load_profile(const gfloat* rec, float (&u)[NX + 1]) {
#pragma unroll
  for (int i = 0; i + 3 <= NX; i += 4) {
    const float4_t a = *reinterpret_cast<const GLOBAL_AS float4_t*>(rec + i);
    u[i] = a.x; u[i + 1] = a.y; u[i + 2] = a.z; u[i + 3] = a.w;
  }
#pragma unroll
  for (int i = (NX + 1) & ~3; i <= NX; ++i) u[i] = rec[i];
  const float tref = u[NX];
#pragma unroll
  for (int i = 0; i <= NX; ++i) u[i] -= tref;
  return tref;
}

// (node NX is written as the copy of node NX-1)
template <int NX>
__device__ __forceinline__ void store_profile(gfloat* rec, const float (&u)[NX + 1], float tref) {
  auto node = [&](int i) { return tref + u[i < NX ? i : NX - 1]; };
#pragma unroll
  for (int i = 0; i + 3 <= NX; i += 4)
    *reinterpret_cast<GLOBAL_AS float4_t*>(rec + i) =
        float4_t{node(i), node(i + 1), node(i + 2), node(i + 3)};
#pragma unroll
  for (int i = (NX + 1) & ~3; i <= NX; ++i) rec[i] = node(i);
}

__device__ __forceinline__ void store8(gfloat* p, const float (&v)[BTPM_BLK]) {
  GLOBAL_AS float4_t* q = reinterpret_cast<GLOBAL_AS float4_t*>(p);
  q[0] = float4_t{v[0], v[1], v[2], v[3]};
  q[1] = float4_t{v[4], v[5], v[6], v[7]};
}

}  // namespace

// ---------------------------------------------------------------------------
// Smooth facets: one lane per column, W columns per workgroup (W = 256, 128
// or 64, instantiated below; the set's tile_cols is W).  The width changes
// only which lanes share a workgroup, never a column's arithmetic.
// ---------------------------------------------------------------------------
template <int W>
__global__ __launch_bounds__(W, 4) void btpm_conduct_smooth(const btpm_tile* __restrict__ tiles,
                                                           const btpm_set_dev* __restrict__ sets,
                                                           const btpm_status_dev* __restrict__ status) {
  // previous-rotation T of the block, parked in LDS (lane-private slots)
  __shared__ float lds_p[BTPM_BLK][W];
  constexpr int NX = BTPM_NX;
  const btpm_tile tl = tiles[blockIdx.x];
  const btpm_set_dev& S = sets[tl.set];
  const btpm_status_dev st = status[tl.set];
  if (st.done || st.rev >= S.max_rev) return;
  const bool check = st.rev > S.check_after;

  const int ncols = S.ncols;
  // lane -> column through the compacted order of unfrozen columns; lanes
  // past its end take a valid column for their (unused) loads
  const int idx = tl.tile * W + (int)threadIdx.x;
  const int norder = st.norder;
  const bool valid = idx < norder;
  const int c = S.order[valid ? idx : (norder > 0 ? norder - 1 : 0)];
  const int cc = c;
  const bool active = valid && (S.inst || !S.frozen[cc]);
  const int nwork = __syncthreads_count(active);
  if (nwork == 0) {
    if (threadIdx.x == 0) {
      S.tile_active[tl.tile] = 0;
      S.tile_work[tl.tile] = 0;
    }
    return;
  }

  Scale sc = make_scale(S.r[cc]);
  const double m1 = (double)S.m1[cc];
  const double es = (double)S.es;
  const double tol = (double)S.newton_tol;
  const int cap = S.newton_cap;
  // with facet self-heating the SpMM has written src + Q into qext
  const gfloat* __restrict__ srcp = (const gfloat*)(S.qext != nullptr ? S.qext : S.src);
  const gfloat* __restrict__ Tin = (const gfloat*)S.T;
  gfloat* __restrict__ Tout = (gfloat*)S.T;
  gfloat* __restrict__ Eout = (gfloat*)S.emis;
  const bool has_e = S.emis != nullptr;
  const float esia = S.esia;

  float u[NX + 1];
  const float Tref = load_profile<NX>((const gfloat*)S.prof + (size_t)cc * BTPM_PSTRIDE, u);
  const double Trefd = (double)Tref;

  const int nb = S.nb;
  const int ntau = S.ntau;
  const size_t bstride = (size_t)ncols * BTPM_BLK;
  const size_t coff = (size_t)cc * BTPM_BLK;

  const int tid = (int)threadIdx.x;
  float nsrc[BTPM_BLK], nprev[BTPM_BLK];
  load8(srcp + coff, nsrc);
  load8(Tin + coff, nprev);

  float dm = 0.0f;
  float dl = 0.0f;   // T - T_prev at the previous step (predictor shift)
  float dl2 = 0.0f;  // and at the step before
  // the TI = 0 loop is a separate instantiation so the main loop stays lean
  auto rotation = [&](auto inst_tag) {
    constexpr bool INST = decltype(inst_tag)::value;
    for (int b = 0; b < nb; ++b) {
#pragma unroll
      for (int k = 0; k < BTPM_BLK; ++k) lds_p[k][tid] = nprev[k];
      // compiler barrier: keep the parked values in LDS, not in VGPRs
      asm volatile("" ::: "memory");
      const bool more = b + 1 < nb;
      const size_t o = (size_t)b * bstride + coff;
      const size_t on = (size_t)(b + 1) * bstride + coff;
      if (more) load8(Tin + on, nprev);
      const int kend = min(BTPM_BLK, ntau - b * BTPM_BLK);
#pragma unroll
      for (int k = 0; k < BTPM_BLK; ++k) {
        const float tp = lds_p[k][tid];
        float t = tp;
        if (k < kend) {
          if constexpr (INST) {  // instantaneous equilibrium (TI = 0), thermal.cpp:1985-2033
            t = (float)sqrt(sqrt((double)nsrc[k] / es));
          } else {
            sc.sd *= sc.sig;
            sc.isd *= sc.isig;
            t = (float)conduct_step<NX>(u, sc.kr, sc.sd, sc.isd, (double)nsrc[k], m1, es, Trefd,
                                        tol, cap, (double)(tp + (2.0f * dl - dl2)));
          }
          dl2 = dl;
          dl = t - tp;
          dm = fmaxf(dm, fabsf(dl));
        }
        lds_p[k][tid] = t;  // the slot now holds this rotation's T
        if (k == BTPM_BLK / 2 - 1 && more) load4(srcp + on, nsrc, 0);
        if (k == BTPM_BLK - 1 && more) load4(srcp + on, nsrc, 4);
      }
      asm volatile("" ::: "memory");
      if constexpr (!INST) rescale<NX>(u, sc);
      if (active) {
        float out[BTPM_BLK];
#pragma unroll
        for (int k = 0; k < BTPM_BLK; ++k) out[k] = lds_p[k][tid];
        store8(Tout + o, out);
        if (has_e) {
#pragma unroll
          for (int k = 0; k < BTPM_BLK; ++k) {
            const float t = out[k];
            out[k] = esia * (t * t) * (t * t);
          }
          store8(Eout + (size_t)cc * nb * BTPM_BLK + (size_t)b * BTPM_BLK, out);  // facet-major
        }
      }
    }
  };
  if (S.inst) rotation(std::true_type{});
  else rotation(std::false_type{});

  bool still = active;
  if (active) {
    if (!S.inst) {
      int cw = c;
      asm volatile("" : "+v"(cw));  // keep the record address out of the step loop
      store_profile<NX>((gfloat*)S.prof + (size_t)cw * BTPM_PSTRIDE, u, Tref);
    }
    S.dmax[c] = dm;
    if (check && dm < S.tacc) {
      still = false;
      if (!S.inst) S.frozen[c] = 1;
    }
  }
  const int nact = __syncthreads_count(still);
  if (threadIdx.x == 0) {
    S.tile_active[tl.tile] = nact;
    S.tile_work[tl.tile] = S.inst ? 0 : nwork;
  }
}

// every width with the same register budget (4 waves per SIMD, 128 VGPRs)
template __global__ void btpm_conduct_smooth<256>(const btpm_tile*, const btpm_set_dev*,
                                                  const btpm_status_dev*);
template __global__ void btpm_conduct_smooth<128>(const btpm_tile*, const btpm_set_dev*,
                                                  const btpm_status_dev*);
template __global__ void btpm_conduct_smooth<64>(const btpm_tile*, const btpm_set_dev*,
                                                 const btpm_status_dev*);

// ---------------------------------------------------------------------------
// Smooth facets with at most BTPM_LIN_CLASSES FTCS numbers, on the matrix cores
// (linear_block.h): one wave per workgroup, 16 NT columns.  NT = 1, 2: four
// or two lanes solve the surface balances of the same column (the balance is a
// chain of dependent FP64 operations, so the copies cost no time where a SIMD
// holds one or two waves, and the set spreads over that many more SIMDs);
// NT = 4: one column per lane.  A column's arithmetic is the same for each.
// The operator's 12 fragments stay in registers for the whole rotation.
// ---------------------------------------------------------------------------
template <int NT>
__global__ __launch_bounds__(64, 2) void btpm_conduct_smooth_lin(
    const btpm_tile* __restrict__ tiles, const btpm_set_dev* __restrict__ sets,
    const btpm_status_dev* __restrict__ status) {
  using namespace btpm_lin;
  constexpr int NX = BTPM_NX;
  constexpr int W = 16 * NT;
  const btpm_tile tl = tiles[blockIdx.x];
  const btpm_set_dev& S = sets[tl.set];
  const btpm_status_dev st = status[tl.set];
  if (st.done || st.rev >= S.max_rev) return;
  const bool check = st.rev > S.check_after;
  const int lane = (int)threadIdx.x, g = lane >> 4;
  const int ncols = S.ncols, norder = st.norder;
  // lane -> column through the compacted order; a tile holds columns of one
  // class, lanes past its columns mirror the first
  const int first = tl.tile * W < norder ? S.order[tl.tile * W] : -1;
  auto tile_col = [&](int l) {
    const int i = tl.tile * W + l;
    return i < norder ? S.order[i] : -1;
  };
  const int own = tile_col(lane % W);
  const bool valid = own >= 0;
  const int c = max(valid ? own : first, 0);
  const bool active = valid && (S.inst || !S.frozen[c]);
  const bool mine = active && lane < W;  // the lane that stores the column
  const int nwork = __popcll(__ballot(mine));
  if (nwork == 0) {
    if (lane == 0) {
      S.tile_active[tl.tile] = 0;
      S.tile_work[tl.tile] = 0;
    }
    return;
  }
  const double m1 = (double)S.m1[c];
  const double es = (double)S.es;
  const double tol = (double)S.newton_tol;
  const int cap = S.newton_cap;
  const gfloat* __restrict__ srcp = (const gfloat*)(S.qext != nullptr ? S.qext : S.src);
  const gfloat* __restrict__ Tin = (const gfloat*)S.T;
  gfloat* __restrict__ Tout = (gfloat*)S.T;
  gfloat* __restrict__ Eout = (gfloat*)S.emis;
  const bool has_e = S.emis != nullptr;
  const float esia = S.esia;
  const int nb = S.nb, ntau = S.ntau;
  const size_t bstride = (size_t)ncols * BTPM_BLK;
  const size_t coff = (size_t)c * BTPM_BLK;

  float nsrc[BTPM_BLK], nprev[BTPM_BLK];
  load8(srcp + coff, nsrc);
  load8(Tin + coff, nprev);
  Surface sf = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  auto store_block = [&](int b, const float (&out)[BTPM_BLK]) {
    if (!mine) return;
    store8(Tout + (size_t)b * bstride + coff, out);
    if (has_e) {
      float e[BTPM_BLK];
#pragma unroll
      for (int k = 0; k < BTPM_BLK; ++k) e[k] = esia * (out[k] * out[k]) * (out[k] * out[k]);
      store8(Eout + (size_t)c * nb * BTPM_BLK + (size_t)b * BTPM_BLK, e);  // facet-major
    }
  };

  if (S.inst) {  // instantaneous equilibrium (TI = 0), thermal.cpp:1985-2033
    for (int b = 0; b < nb; ++b) {
      load8(srcp + (size_t)b * bstride + coff, nsrc);
      load8(Tin + (size_t)b * bstride + coff, nprev);
      const int kend = min(BTPM_BLK, ntau - b * BTPM_BLK);
      float out[BTPM_BLK];
#pragma unroll
      for (int k = 0; k < BTPM_BLK; ++k) {
        out[k] = nprev[k];
        if (k < kend) {
          out[k] = (float)sqrt(sqrt((double)nsrc[k] / es));
          sf.dm = fmaxf(sf.dm, fabsf(out[k] - nprev[k]));
        }
      }
      store_block(b, out);
    }
  } else {
    const _Float16* opk = static_cast<const _Float16*>(S.op) +
                          (S.cls != nullptr ? (size_t)S.cls[first] * BTPM_LIN_OP : 0);
    const GLOBAL_AS h8* __restrict__ op = (const GLOBAL_AS h8*)opk + lane;
    h8 A[kFrags];
#pragma unroll
    for (int i = 0; i < kFrags; ++i) A[i] = op[i * 64];
    float gain[BTPM_BLK];
#pragma unroll
    for (int k = 0; k < BTPM_BLK; ++k)
      gain[k] = reinterpret_cast<const float*>(opk + kGain)[k];
    const float own_main = reinterpret_cast<const float*>(opk + kOwn)[0];
    const float own_tail = reinterpret_cast<const float*>(opk + kOwn)[1];
    const gfloat* prof = (const gfloat*)S.prof;
    float u[NT][16];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int ct = tile_col(16 * t + (lane & 15));
      const gfloat* rec = prof + (size_t)(ct >= 0 ? ct : first) * BTPM_PSTRIDE;
      load_nodes(rec, g, rec[NX], u[t]);
    }
    const gfloat* rec = prof + (size_t)c * BTPM_PSTRIDE;
    const float Tref = rec[NX];
    sf.u0 = (rec[0] - Tref) * kScale;
    const double Trefd = (double)Tref;
    linear_init<NT>(u, op[2 * kFrags * 64], op[(2 * kFrags + 1) * 64]);
    float w[BTPM_BLK];
    surface_out(u, w);

    auto block = [&](int b, auto full_tag) {
      constexpr bool FULL = decltype(full_tag)::value;
      const int kend = FULL ? BTPM_BLK : ntau - b * BTPM_BLK;
      float src[BTPM_BLK], out[BTPM_BLK];
#pragma unroll
      for (int k = 0; k < BTPM_BLK; ++k) {
        src[k] = nsrc[k];
        out[k] = nprev[k];
      }
      if (FULL) {
        load8(srcp + (size_t)(b + 1) * bstride + coff, nsrc);
        load8(Tin + (size_t)(b + 1) * bstride + coff, nprev);
      }
      surface_steps<FULL>(sf, w, out, src, gain, m1, es, Trefd, tol, cap, kend, [](int) {});
      store_block(b, out);
      surface_in(u, w);
      if constexpr (FULL) {
        if constexpr (NT == 4) linear_block_pairs(u, own_main, [&](int i) { return A[i]; });
        else linear_block<NT>(u, own_main, [&](int i) { return A[i]; });
        surface_out(u, w);
      } else {
        linear_block<NT>(u, own_tail, [&](int i) { return (h8)op[(kFrags + i) * 64]; });
      }
    };
    for (int b = 0; b + 1 < nb; ++b) block(b, std::true_type{});
    block(nb - 1, std::false_type{});

#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int ct = tile_col(16 * t + (lane & 15));
      if (ct < 0 || S.frozen[ct]) continue;
      gfloat* r = (gfloat*)S.prof + (size_t)ct * BTPM_PSTRIDE;
      store_nodes(r, g, r[NX], u[t]);
    }
    if (mine)
      ((gfloat*)S.prof)[(size_t)c * BTPM_PSTRIDE] = fmaf(sf.u0, 1.0f / kScale, Tref);
  }

  bool still = mine;
  if (mine) {
    S.dmax[c] = sf.dm;
    if (check && sf.dm < S.tacc) {
      still = false;
      if (!S.inst) S.frozen[c] = 1;
    }
  }
  const int nact = __popcll(__ballot(still));
  if (lane == 0) {
    S.tile_active[tl.tile] = nact;
    S.tile_work[tl.tile] = S.inst ? 0 : nwork;
  }
}

template __global__ void btpm_conduct_smooth_lin<1>(const btpm_tile*, const btpm_set_dev*,
                                                    const btpm_status_dev*);
template __global__ void btpm_conduct_smooth_lin<2>(const btpm_tile*, const btpm_set_dev*,
                                                    const btpm_status_dev*);
template __global__ void btpm_conduct_smooth_lin<4>(const btpm_tile*, const btpm_set_dev*,
                                                    const btpm_status_dev*);

// ---------------------------------------------------------------------------
// Crater columns: BTPM_CRATERS_WG craters x 100 sub-facets per workgroup of
// 1024 lanes (lane -> sub-facet column, 24 idle lanes).  Every 8-step block
// the workgroup evaluates the crater self-heating of all its craters for the
// 8 steps at once as one MFMA product
//     Q[j][n] = sum_i VF(j->i) E[i][n],   n = (crater, step in block)
// with M = 100 (padded 112), K = 100 (padded 128), N = 80, using
// v_mfma_f32_16x16x32_f16 and the three-product split
//     VF E ~ VFhi Ehi + VFhi Elo + VFlo Ehi   (FP32 accumulation),
// where x_hi = fp16(x) and x_lo = fp16(x - x_hi).  VF is stored pre-scaled by
// 2^s (max entry in [0.5, 1)) so its low halves stay normal fp16 numbers;
// the FP32 accumulator is multiplied by 2^-s, which is exact.
// ---------------------------------------------------------------------------
namespace {
constexpr int kMP = 112;           // padded M (receiving sub-facet j)
constexpr int kKP = 112;           // padded K (emitting sub-facet i)
// LDS row stride in halves: 52 dwords, so the 8 rows of one 16-byte fragment
// read (8 lanes) start at multiples of 4 banks, all different, and cover all
// 32 banks; k runs to 99 only (three chunks of 32 and the tail 96..99)
constexpr int kLdsK = 104;
constexpr int kNP = BTPM_CRATERS_WG * BTPM_BLK;  // 80 columns of the product
// Q row stride: 1000 columns + 24 idle lanes + 4 floats of padding, so the
// 8 step rows start in different LDS banks and the product's float4 stores
// for steps 0..7 of one column (8 lanes) do not collide on one bank
constexpr int kQCols = 1028;
constexpr int kMT = kMP / 16;      // 7 M tiles
constexpr int kNT = kNP / 16;      // 5 N tiles

// Q[n][m] = sum_k A[m][k] B[n][k] over the padded 112 x 112 x 80 tile held in
// LDS (A = VF^T hi/lo, B = E hi/lo).  Q is written column-major for the
// conduction lanes: product column n = crater * 8 + step goes to
// lds_q[step][crater * 100 + m], m < 100.  Output layout of the 16 x 16 MFMAs:
// lane l receives D[m = 4(l/16) + i][n = l%16], i = 0..3.
//
// The phase is bound by the latency of its LDS fragment reads, so a wave
// computes a strip of one m tile and 3 (or 2) n tiles, reading each A fragment
// once per K chunk for the whole strip; K runs as 4 chunks of 32
// (v_mfma_f32_16x16x32_f16, 16-byte fragment reads), the last with the tail
// k = 96..99 in its first slots and zeros in the others.  One instruction
// shape throughout: a 16x16x16 instruction that adds to what a 16x16x32 has
// just left there was seen to give wrong rows 4g, 4g + 1, and what keeps the
// two far enough apart is then up to the schedule.
// The 14 strips (7 m tiles x {n 0-2, n 3-4}) sit on the waves so that each
// SIMD (waves s, s+4, s+8, s+12) carries at most 9 of the 35 output tiles;
// waves 12 and 13 have none.  Within a lane, fragment slot j of A and of B
// hold the same k, which is all the product needs of the K layout.
//
// One K chunk of 32 (v_mfma_f32_16x16x32_f16): lane l supplies
// A[m = l%16][k = 8(l/16) .. +7] and B[k = 8(l/16) .. +7][n = l%16].
// The low halves lie AH (of A) and BH (of B) halves behind the high ones; A
// counts as zero in lanes without `use`.
template <int NNT, int AH, int BH>
__device__ __forceinline__ void strip_chunk32(const _Float16* lds_a, const _Float16* lds_b, int am,
                                              int k0, int nt0, int r, bool use,
                                              float4_t (&acc)[NNT]) {
  const half8_t zero = {0, 0, 0, 0, 0, 0, 0, 0};
  half8_t ahi = *reinterpret_cast<const half8_t*>(&lds_a[am * kLdsK + k0]);
  half8_t alo = *reinterpret_cast<const half8_t*>(&lds_a[AH + am * kLdsK + k0]);
  ahi = use ? ahi : zero;
  alo = use ? alo : zero;
#pragma unroll
  for (int t = 0; t < NNT; ++t) {
    const int bn = (nt0 + t) * 16 + r;
    const half8_t bhi = *reinterpret_cast<const half8_t*>(&lds_b[bn * kLdsK + k0]);
    const half8_t blo = *reinterpret_cast<const half8_t*>(&lds_b[BH + bn * kLdsK + k0]);
    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(alo, bhi, acc[t], 0, 0, 0);
    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi, blo, acc[t], 0, 0, 0);
    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi, bhi, acc[t], 0, 0, 0);
  }
}

// (QC: Q row stride; NV: product columns that exist, the rest of the last tile
// is padding and not stored)
template <int NNT, int AH, int BH, int QC, int NV>
__device__ __forceinline__ void product_strip(const _Float16* lds_a, const _Float16* lds_b,
                                              float* lds_q, int mt, int nt0, int lane,
                                              float unscale) {
  constexpr int kFull = BTPM_NS / 32 * 32;  // 96: sub-facets in full chunks of 32
  static_assert(BTPM_NS - kFull == 4 && kLdsK == kFull + 8, "one partial K chunk of 4");
  float4_t acc[NNT];
#pragma unroll
  for (int t = 0; t < NNT; ++t) acc[t] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
  const int r = lane & 15;
  const int g = lane >> 4;
  const int am = mt * 16 + r;
  // the tail k = 96..99 as a fourth chunk of 32 whose other slots are zero: A
  // in the lanes past the first 16 (B is read by all, so a NaN there is one of
  // the column's own), and k = 100..103 are zero in both
#pragma unroll 1
  for (int kt = 0; kt <= kFull / 32; ++kt) {
    const bool tail = kt == kFull / 32;
    strip_chunk32<NNT, AH, BH>(lds_a, lds_b, am, tail ? kFull : kt * 32 + 8 * g, nt0, r,
                               !tail || g == 0, acc);
  }
  const int m0 = mt * 16 + 4 * g;  // 4 receiving sub-facets m0 .. m0 + 3
  if (m0 < BTPM_NS) {
#pragma unroll
    for (int t = 0; t < NNT; ++t) {
      const int bn = (nt0 + t) * 16 + r;
      if (NV % 16 != 0 && bn >= NV) continue;
      float* q = &lds_q[(bn & (BTPM_BLK - 1)) * QC + (bn / BTPM_BLK) * BTPM_NS + m0];
      *reinterpret_cast<float4*>(q) = make_float4(acc[t][0] * unscale, acc[t][1] * unscale,
                                                  acc[t][2] * unscale, acc[t][3] * unscale);
    }
  }
}

// wave -> strip, one nibble per wave: 0..6 = m tile with n tiles 0-2,
// 7..13 = m tile (value - 7) with n tiles 3-4, 15 = none
constexpr unsigned long long kStripOfWave = 0xD9FFC852B741A630ull;

template <int AH, int BH, int QC>
__device__ __forceinline__ void crater_product(const _Float16* lds_a, const _Float16* lds_b,
                                               float* lds_q, int wave, int lane, float unscale) {
  static_assert(kMT == 7 && kNT == 5 && BTPM_CRATER_THREADS == 1024, "strip table shape");
  const int s = (int)((kStripOfWave >> (4 * wave)) & 15ull);
  if (s < kMT)
    product_strip<3, AH, BH, QC, kNP>(lds_a, lds_b, lds_q, s, 0, lane, unscale);
  else if (s < 2 * kMT)
    product_strip<2, AH, BH, QC, kNP>(lds_a, lds_b, lds_q, s - kMT, 3, lane, unscale);
}

// Stage VF^T hi/lo ([2][112][112] fp16 in global memory) into LDS, k < 104.
__device__ __forceinline__ void stage_vf(const _Float16* src, _Float16 (*lds_a)[kMP * kLdsK],
                                         int tid) {
  for (int e = tid; e < 2 * kMP * kLdsK; e += BTPM_CRATER_THREADS) {
    const int h = e / (kMP * kLdsK);
    const int rem = e - h * kMP * kLdsK;
    const int m = rem / kLdsK, k = rem - m * kLdsK;
    lds_a[h][rem] = src[(h * kMP + m) * kKP + k];
  }
}
}  // namespace

extern "C" __global__ __launch_bounds__(BTPM_CRATER_THREADS) void btpm_conduct_crater(
    const btpm_tile* __restrict__ tiles, const btpm_set_dev* __restrict__ sets,
    const btpm_status_dev* __restrict__ status) {
  constexpr int NX = BTPM_NX;
  constexpr int NS = BTPM_NS;
  constexpr int P = BTPM_CRATERS_WG;
  __shared__ _Float16 lds_a[2][kMP * kLdsK];   // VF^T hi / lo  (52 KB)
  __shared__ _Float16 lds_b[2][kNP * kLdsK];   // E hi / lo     (37 KB)
  __shared__ float lds_q[BTPM_BLK * kQCols];   // product [step][column] (32 KB)
  __shared__ float lds_p[BTPM_BLK][BTPM_CRATER_THREADS];  // T_prev, then T (32 KB)
  __shared__ CraterConst lds_cc[P];            // per-crater constants
  __shared__ unsigned lds_cmax[P];
  __shared__ int lds_cnt;
  __shared__ int lds_nres[P];                  // blocks per rescale per crater

  const btpm_tile tl = tiles[blockIdx.x];
  const btpm_set_dev& S = sets[tl.set];
  const btpm_status_dev st = status[tl.set];
  if (st.done || st.rev >= S.max_rev) return;
  const bool check = st.rev > S.check_after;

  const int tid = (int)threadIdx.x;
  const int lc = tid < P * NS ? tid : P * NS - 1;  // local column (clamped)
  const int lcr = lc / NS;                         // local crater
  const int j = lc - lcr * NS;                     // sub-facet
  // local crater -> crater through the compacted order of unfrozen craters;
  // slots past its end and the idle lanes (tid >= 1000) mirror a valid
  // crater's column, so they stay well-behaved
  const int norder = st.norder;
  const int slot = tl.tile * P + lcr;
  const bool valid = tid < P * NS && slot < norder;
  const int last = norder > 0 ? norder - 1 : 0;
  const int g = S.order[slot < norder ? slot : last];
  const int gg = g;
  const int c = gg * NS + j;                       // global column
  const bool active = valid && !S.frozen[gg];
  const int nwork = __syncthreads_count(active);
  if (nwork == 0) {
    if (tid == 0) {
      S.tile_active[tl.tile] = 0;
      S.tile_work[tl.tile] = 0;
    }
    return;
  }

  // stage VF^T (hi, lo) once per launch; zero the padded E rows
  {
    stage_vf(reinterpret_cast<const _Float16*>(S.vfA), lds_a, tid);
    for (int e = tid; e < 2 * kNP * kLdsK; e += BTPM_CRATER_THREADS)
      (&lds_b[0][0])[e] = (_Float16)0.0f;
    if (tid < P) {
      lds_cmax[tid] = 0u;
      const int gt = S.order[tl.tile * P + tid < norder ? tl.tile * P + tid : last];
      scale_table(S.r[gt], lds_cc[tid].sk, lds_cc[tid].pk, kRescaleMax * BTPM_BLK);
      lds_nres[tid] = rescale_blocks(S.r[gt]);
      lds_cc[tid].r0[0] = 1.0;
      lds_cc[tid].m1 = (double)S.m1[gt];
      lds_cc[tid].es = (double)S.es;
      lds_cc[tid].tol = (double)S.newton_tol;
    }
  }
  __syncthreads();
  // the idle lanes' Q slots are never written by the product
  if (tid >= P * NS)
    for (int k = 0; k < BTPM_BLK; ++k) lds_q[k * kQCols + tid] = 0.0f;

  const float kr = scaled_kr(S.r[gg]);
  CraterConst& cc = lds_cc[lcr];
  const int cap = S.newton_cap;
  int nres = kRescaleMax;  // blocks per rescale: the workgroup's smallest
  for (int i = 0; i < P; ++i) nres = min(nres, lds_nres[i]);
  nres = __builtin_amdgcn_readfirstlane(nres);
  int bph = 0;   // blocks since the last rescale
  int rpar = 0;  // rescales so far, mod 2
  const float esia = S.esia;
  const int ncols = S.ncols;
  // held in a register, so the block loop has no scalar load (read through S
  // there, it is reloaded after every barrier, and a pending scalar load
  // makes the product's first LDS wait a full drain of the shared counter)
  const float vf_unscale = S.vf_unscale;

  float u[NX + 1];
  const float Tref = load_profile<NX>((const gfloat*)S.prof + (size_t)c * BTPM_PSTRIDE, u);
  const double Trefd = (double)Tref;

  const int nb = S.nb;
  const int ntau = S.ntau;
  const size_t bstride = (size_t)ncols * BTPM_BLK;
  const unsigned coff = (unsigned)c * BTPM_BLK;   // < 2^32 / 4: lane part of an address
  const int wave = tid >> 6;
  const int lane = tid & 63;

  const gfloat* __restrict__ srcp = (const gfloat*)S.src;
  const gfloat* __restrict__ Tin = (const gfloat*)S.T;
  gfloat* __restrict__ Tout = (gfloat*)S.T;
  float nsrc[BTPM_BLK], nprev[BTPM_BLK];
  load8(srcp + coff, nsrc);
  load8(Tin + coff, nprev);

  float dm = 0.0f;
  float dl = 0.0f;   // T - T_prev at the previous step (predictor shift)
  float dl2 = 0.0f;  // and at the step before
  // the lane's part of a block address, 32 bits, added to the uniform block
  // base at each use (the asm statement keeps the compiler from folding it
  // into 64-bit per-lane pointers held across the loop)
  auto lane_off = [&]() {
    unsigned o = coff;
    asm volatile("" : "+v"(o));
    return o;
  };

  // previous-rotation emission of block b -> LDS (fp16 hi/lo split), T_prev
  // parked in lane-private LDS slots, the next block's T_prev prefetched,
  // then the block's self-heating product into lds_q
  auto block_head = [&](int b, bool more) {
    if (tid < P * NS) {
#pragma unroll
      for (int k = 0; k < BTPM_BLK; ++k) {
        const float t = nprev[k];
        const float e = esia * (t * t) * (t * t);
        const _Float16 hi = (_Float16)e;
        const _Float16 lo = (_Float16)(e - (float)hi);
        const int n = lcr * BTPM_BLK + k;
        lds_b[0][n * kLdsK + j] = hi;
        lds_b[1][n * kLdsK + j] = lo;
      }
    }
#pragma unroll
    for (int k = 0; k < BTPM_BLK; ++k) lds_p[k][tid] = nprev[k];
    if (more) load8(Tin + (size_t)(b + 1) * bstride + lane_off(), nprev);
    __syncthreads();
    crater_product<kMP * kLdsK, kNP * kLdsK, kQCols>(lds_a[0], lds_b[0], lds_q, wave, lane, vf_unscale);
    __syncthreads();
  };
  auto block_tail = [&](int b) {
    if (active) {
      float out[BTPM_BLK];
#pragma unroll
      for (int k = 0; k < BTPM_BLK; ++k) out[k] = lds_p[k][tid];
      store8(Tout + (size_t)b * bstride + lane_off(), out);
    }
  };
  // U *= f = fp32(r0 sig^n) at a rescale, n the steps since the last one; the
  // residual r0 sig^n / f is carried (cc.r0 is double buffered by rescale
  // parity: every lane reads one half, sub-facet 0 writes the other, and the
  // barriers of the blocks in between order them)
  auto block_scale = [&](int n) {
    const double pb = cc.r0[rpar] * cc.pk[n - 1];
    const float f = (float)pb;
    if (j == 0) cc.r0[rpar ^ 1] = fma(pb - (double)f, (double)__builtin_amdgcn_rcpf(f), 1.0);
    rpar ^= 1;
    return f;
  };
  auto after_step = [&](int k, float tp, float t) {
    dl2 = dl;
    dl = t - tp;
    dm = fmaxf(dm, fabsf(dl));
    lds_p[k][tid] = t;  // the slot now holds this rotation's T
  };
  auto next_src = [&](int b, int k) {
    const gfloat* next = srcp + (size_t)(b + 1) * bstride;  // uniform block base
    if (k == BTPM_BLK / 2 - 1) load4(next + lane_off(), nsrc, 0);
    if (k == BTPM_BLK - 1) load4(next + lane_off(), nsrc, 4);
  };

  // the steps of block b, all 57 nodes on the vector ALUs.  FULL: the block
  // has all 8 steps and a successor whose inputs are prefetched (every block
  // but the last), so the unrolled steps carry no step-count tests
  auto valu_steps = [&](int b, auto inst_tag, auto full_tag) {
    constexpr bool INST = decltype(inst_tag)::value;
    constexpr bool FULL = decltype(full_tag)::value;
    const int kend = FULL ? BTPM_BLK : min(BTPM_BLK, ntau - b * BTPM_BLK);
    // this block's row of the scale table (steps since the last rescale)
    const float2* sk8 = &cc.sk[bph * BTPM_BLK];
#pragma unroll
    for (int k = 0; k < BTPM_BLK; ++k) {
      const float tp = lds_p[k][tid];
      if (FULL || k < kend) {
        const double tot = (double)(nsrc[k] + lds_q[k * kQCols + tid]);
        float t;
        if constexpr (INST) {  // roughness_inst_equilibrium, thermal_GPU.cu:581-641
          t = (float)sqrt(sqrt(tot / cc.es));
        } else {
          // the per-step conversions leave out the residual (within 6e-8 of
          // 1): a bounded perturbation of T_1 and T_0, not a gain on the profile
          const float2 sk = sk8[k];
          t = (float)conduct_step<NX>(u, kr, sk.x, sk.y, tot, cc.m1, cc.es, Trefd, cc.tol, cap,
                                      (double)(tp + (2.0f * dl - dl2)));
        }
        after_step(k, tp, t);
      }
      if constexpr (FULL) next_src(b, k);
    }
    asm volatile("" ::: "memory");
    if constexpr (!INST) {
      // every nres blocks, and at the end of the rotation (the profile goes
      // out unscaled)
      if (!FULL || bph + 1 == nres) {
        const float f = block_scale(bph * BTPM_BLK + kend);
#pragma unroll
        for (int i = 0; i < NX; ++i) u[i] *= f;
        bph = 0;
      } else {
        ++bph;
      }
    }
  };

  // the TI = 0 loop is a separate instantiation so the main loop stays lean
  auto rotation = [&](auto inst_tag) {
    for (int b = 0; b + 1 < nb; ++b) {
      block_head(b, true);
      valu_steps(b, inst_tag, std::true_type{});
      block_tail(b);
    }
    block_head(nb - 1, false);
    valu_steps(nb - 1, inst_tag, std::false_type{});
    block_tail(nb - 1);
  };
  if (S.inst) rotation(std::true_type{});
  else rotation(std::false_type{});

  // per-crater freeze test (converged kernel, T175706/thermal_GPU.cu:648-692)
  if (active) {
    if (!S.inst) {
      int cw = c;
      asm volatile("" : "+v"(cw));  // keep the record address out of the step loop
      store_profile<NX>((gfloat*)S.prof + (size_t)cw * BTPM_PSTRIDE, u, Tref);
    }
    atomicMax(&lds_cmax[lcr], __float_as_uint(dm));
  }
  if (tid == 0) lds_cnt = 0;
  __syncthreads();
  if (active && j == 0) {
    const float cm = __uint_as_float(lds_cmax[lcr]);
    S.dmax[g] = cm;
    bool still = true;
    if (check && cm < S.tacc) {
      S.frozen[g] = 1;
      still = false;
    }
    if (still) atomicAdd(&lds_cnt, 1);
  }
  __syncthreads();
  if (tid == 0) {
    S.tile_active[tl.tile] = lds_cnt;
    S.tile_work[tl.tile] = S.inst ? 0 : nwork;
  }
}

// ---------------------------------------------------------------------------
// Crater columns of at most BTPM_LIN_CLASSES FTCS numbers, on the 8-step
// operator (linear_block.h): P craters x 100 sub-facets per workgroup, lane ->
// column in the surface steps, four 16-column tiles per wave in the operator's
// product.  The crater product of block b + 1 needs only the previous
// rotation's temperatures, so it runs beside the surface steps of block b, a
// piece of it in each step (its matrix instructions issue into the waits of
// the balance's dependent FP64 chain), and the emission of block b + 2 is
// split after them: E and Q are double buffered and a block has one barrier.
// The fragments that do not change (the wave's m tiles of VF^T, at P = 2
// the operator too) stay in registers for the whole rotation.  P = 5
// puts 98 % of its lanes to work, two waves to a SIMD; P = 2 spreads few
// craters over more CUs, one wave to a SIMD.  A 650-step rotation, none frozen,
// at P = 2 / 5 and with ten craters a workgroup and the steps on the vector
// ALUs: 80 craters 267 / 389 / 718 us, 512 craters 292 / 403 / 756 us, 640
// craters 525 / 411 / 744 us, 5120 craters 2.58 / 1.69 / 1.73 ms: on a full chip
// the operator only holds what the vector ALUs reach.
// ---------------------------------------------------------------------------
namespace {
template <int P>
struct CraterGroup {
  static constexpr int kThreads = (P * BTPM_NS + 63) / 64 * 64;
  static constexpr int kWaves = kThreads / 64;
  static constexpr int kNT = (P * BTPM_BLK + 15) / 16;  // n tiles of the product
  static constexpr int kQC = kThreads + 4;              // Q row stride in floats
  // E rows: the product's columns, and 8 that the idle lanes write
  static constexpr int kRows = 16 * kNT > 8 * P + 8 ? 16 * kNT : 8 * P + 8;
  static constexpr int kBH = kRows * kLdsK;             // low halves behind the high
  static constexpr int kM = (kMT + kWaves - 1) / kWaves;  // m tiles per wave
  // two waves share a SIMD at P = 5 (256 registers each): the operator's
  // fragments are read from LDS there
  static constexpr bool kOpLds = P > 2;
};

// A fragments of one m tile of VF^T: three K chunks of 32 and the tail 96..99
// as a fourth whose other slots are zero, as in product_strip.
struct VfFrag {
  half8_t hi[4], lo[4];
};
__device__ __forceinline__ VfFrag load_vf(const _Float16* vfA, int mt, int lane) {
  const int r = lane & 15, g = lane >> 4;
  const _Float16* row = vfA + (size_t)(mt * 16 + r) * kKP;
  VfFrag f;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    f.hi[c] = *reinterpret_cast<const half8_t*>(row + 32 * c + 8 * g);
    f.lo[c] = *reinterpret_cast<const half8_t*>(row + kMP * kKP + 32 * c + 8 * g);
  }
  const half8_t zero = {0, 0, 0, 0, 0, 0, 0, 0};  // k >= 100 is zero in the tiles
  f.hi[3] = g == 0 ? *reinterpret_cast<const half8_t*>(row + 96) : zero;
  f.lo[3] = g == 0 ? *reinterpret_cast<const half8_t*>(row + kMP * kKP + 96) : zero;
  return f;
}

// One piece of the product is K chunk c of n tile t for the wave's M m tiles
// (mt0, mt0 + step, ...).  Nothing in it branches, so a piece can be scheduled
// among other work: lanes whose Q does not exist store it behind the row, and
// in the tail chunk the lanes of g > 0 read entries that meet zeros in A (of
// the same column, so a NaN there is one already).
struct EFrag {
  half8_t hi, lo;
};
template <int P>
__device__ __forceinline__ EFrag load_e(const _Float16* lds_b, int t, int c, int lane) {
  using G = CraterGroup<P>;
  const int r = lane & 15, g = lane >> 4;
  const _Float16* row = lds_b + (16 * t + r) * kLdsK + (c < 3 ? 32 * c + 8 * g : 96);
  return EFrag{*reinterpret_cast<const half8_t*>(row),
               *reinterpret_cast<const half8_t*>(row + G::kBH)};
}
template <int P, int M>
__device__ __forceinline__ void product_piece(const VfFrag (&a)[M], const EFrag& e,
                                              float4_t (&acc)[M], int t, int c, int mt0, int step,
                                              float* lds_q, int lane, float unscale) {
  using G = CraterGroup<P>;
  const int r = lane & 15, g = lane >> 4;
  if (c == 0)
#pragma unroll
    for (int m = 0; m < M; ++m) acc[m] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int p = 0; p < 3; ++p)
#pragma unroll
    for (int m = 0; m < M; ++m)
      acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(p == 0 ? a[m].lo[c] : a[m].hi[c],
                                                      p == 1 ? e.lo : e.hi, acc[m], 0, 0, 0);
  if (c < 3) return;
  const int bn = 16 * t + r;  // product column: crater bn / 8, step bn % 8
#pragma unroll
  for (int m = 0; m < M; ++m) {
    const int mt = mt0 + m * step, m0 = mt * 16 + 4 * g;
    const int col = m0 < BTPM_NS && bn < P * BTPM_BLK ? (bn / BTPM_BLK) * BTPM_NS + m0 : G::kThreads;
    *reinterpret_cast<float4*>(&lds_q[(bn & (BTPM_BLK - 1)) * G::kQC + col]) =
        make_float4(acc[m][0] * unscale, acc[m][1] * unscale, acc[m][2] * unscale,
                    acc[m][3] * unscale);
  }
}
}  // namespace

template <int P>
__global__ __launch_bounds__((P * BTPM_NS + 63) / 64 * 64) void btpm_conduct_crater_lin(
    const btpm_tile* __restrict__ tiles, const btpm_set_dev* __restrict__ sets,
    const btpm_status_dev* __restrict__ status) {
  using namespace btpm_lin;
  using G = CraterGroup<P>;
  constexpr int NX = BTPM_NX, NS = BTPM_NS, TH = G::kThreads;
  __shared__ __align__(16) _Float16 lds_b[2][2 * G::kBH];
  __shared__ __align__(16) float lds_q[2][BTPM_BLK * G::kQC];
  __shared__ float lds_t[2][BTPM_BLK][TH];  // T_prev of the next two blocks
  __shared__ __align__(16) _Float16 lds_op[G::kOpLds ? kFrags * kFrag : 8];
  __shared__ unsigned lds_cmax[P];
  __shared__ int lds_cnt;

  const btpm_tile tl = tiles[blockIdx.x];
  const btpm_set_dev& S = sets[tl.set];
  const btpm_status_dev st = status[tl.set];
  if (st.done || st.rev >= S.max_rev) return;
  const bool check = st.rev > S.check_after;
  const int tid = (int)threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g4 = lane >> 4;
  const int norder = st.norder;
  // local crater -> crater through the compacted order (a tile holds craters
  // of one class); idle lanes and empty slots mirror the first crater's columns
  const int first = tl.tile * P < norder ? S.order[tl.tile * P] : -1;
  auto crater = [&](int l) {
    const int slot = tl.tile * P + l;
    return l < P && slot < norder ? S.order[slot] : -1;
  };
  const int lcr = tid / NS, j = tid % NS;
  const int own = crater(lcr);
  const int gr = max(own >= 0 ? own : first, 0);
  const int c = gr * NS + j;
  const bool active = own >= 0 && !S.frozen[gr];
  const int nwork = __syncthreads_count(active);
  if (nwork == 0) {
    if (tid == 0) {
      S.tile_active[tl.tile] = 0;
      S.tile_work[tl.tile] = 0;
    }
    return;
  }
  if (tid < P) lds_cmax[tid] = 0u;
  // E rows of the last n tile's padding and Q slots of the idle lanes are
  // never written by a block
  for (int e = tid; e < 4 * G::kBH; e += TH) (&lds_b[0][0])[e] = (_Float16)0.0f;
  if (tid >= P * NS)
    for (int k = 0; k < BTPM_BLK; ++k) lds_q[0][k * G::kQC + tid] = lds_q[1][k * G::kQC + tid] = 0.0f;
  const _Float16* opk = static_cast<const _Float16*>(S.op) +
                        (S.cls != nullptr ? (size_t)S.cls[first] * BTPM_LIN_OP : 0);
  if constexpr (G::kOpLds)
    for (int e = tid; e < kFrags * 64; e += TH)
      reinterpret_cast<h8*>(lds_op)[e] = reinterpret_cast<const h8*>(opk)[e];
  VfFrag vf[G::kM];
#pragma unroll
  for (int m = 0; m < G::kM; ++m)  // past the last m tile: any tile, its rows are not stored
    vf[m] = load_vf(reinterpret_cast<const _Float16*>(S.vfA), min(wave + m * G::kWaves, kMT - 1),
                    lane);
  const double m1 = (double)S.m1[gr];
  const double es = (double)S.es, tol = (double)S.newton_tol;
  const int cap = S.newton_cap;
  const float esia = S.esia;
  const float vf_unscale = S.vf_unscale;
  const int nb = S.nb, ntau = S.ntau;
  const size_t bstride = (size_t)S.ncols * BTPM_BLK;
  const gfloat* srcp = (const gfloat*)S.src + (size_t)c * BTPM_BLK;
  const gfloat* Tin = (const gfloat*)S.T + (size_t)c * BTPM_BLK;
  gfloat* Tout = (gfloat*)S.T + (size_t)c * BTPM_BLK;
  Surface sf = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  __syncthreads();  // the cleared E rows, the operator

  // emission of a block, fp16 hi / lo, into E buffer i (idle lanes: rows 8P..)
  _Float16* const eb = &lds_b[0][lcr * BTPM_BLK * kLdsK + j];
  auto split_e = [&](int i, const float (&t)[BTPM_BLK]) {
#pragma unroll
    for (int k = 0; k < BTPM_BLK; ++k) {
      const float e = esia * (t[k] * t[k]) * (t[k] * t[k]);
      const _Float16 hi = (_Float16)e;
      _Float16* p = eb + i * 2 * G::kBH + k * kLdsK;
      p[0] = hi;
      p[G::kBH] = (_Float16)(e - (float)hi);
    }
  };
  constexpr int kPieces = 4 * G::kNT;          // of the product, spread over the 8 steps
  constexpr int kPer = (kPieces + 7) / 8;      // at most in one step
  auto first_piece = [](int k) { return kPieces * k / 8; };
  float4_t acc[G::kM];
  EFrag ef[kPer];
  // the E fragments of step k's pieces, read a step ahead; the pieces themselves
  auto load_pieces = [&](int i, int k) {
#pragma unroll
    for (int q = 0; q < kPer; ++q)
      if (first_piece(k) + q < first_piece(k + 1))
        ef[q] = load_e<P>(lds_b[i], (first_piece(k) + q) / 4, (first_piece(k) + q) % 4, lane);
  };
  auto run_pieces = [&](int i, int k) {
#pragma unroll
    for (int q = 0; q < kPer; ++q)
      if (first_piece(k) + q < first_piece(k + 1))
        product_piece<P>(vf, ef[q], acc, (first_piece(k) + q) / 4, (first_piece(k) + q) % 4, wave,
                         G::kWaves, lds_q[i], lane, vf_unscale);
  };
  auto product = [&](int i) {
#pragma unroll
    for (int k = 0; k < BTPM_BLK; ++k) {
      load_pieces(i, k);
      run_pieces(i, k);
    }
  };

  if (S.inst) {  // roughness_inst_equilibrium, thermal_GPU.cu:581-641
    for (int b = 0; b < nb; ++b) {
      float src[BTPM_BLK], t[BTPM_BLK];
      load8(srcp + (size_t)b * bstride, src);
      load8(Tin + (size_t)b * bstride, t);
      split_e(0, t);
      __syncthreads();
      product(0);
      __syncthreads();
      const int kend = min(BTPM_BLK, ntau - b * BTPM_BLK);
#pragma unroll
      for (int k = 0; k < BTPM_BLK; ++k)
        if (k < kend) {
          const float x = (float)sqrt(sqrt((double)(src[k] + lds_q[0][k * G::kQC + tid]) / es));
          sf.dm = fmaxf(sf.dm, fabsf(x - t[k]));
          t[k] = x;
        }
      if (active) store8(Tout + (size_t)b * bstride, t);
    }
  } else {
    const GLOBAL_AS h8* op = (const GLOBAL_AS h8*)opk + lane;
    const h8* lop = reinterpret_cast<const h8*>(lds_op) + lane;
    h8 A[G::kOpLds ? 1 : kFrags];
    if constexpr (!G::kOpLds)
#pragma unroll
      for (int i = 0; i < kFrags; ++i) A[i] = op[i * 64];
    float gain[BTPM_BLK];
#pragma unroll
    for (int k = 0; k < BTPM_BLK; ++k)
      gain[k] = reinterpret_cast<const float*>(opk + kGain)[k];
    const float own_main = reinterpret_cast<const float*>(opk + kOwn)[0];
    const float own_tail = reinterpret_cast<const float*>(opk + kOwn)[1];
    const gfloat* prof = (const gfloat*)S.prof;
    float u[4][16];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int l = 64 * wave + 16 * t + (lane & 15), ct = crater(l / NS);
      const gfloat* rec = prof + (size_t)((ct >= 0 ? ct : first) * NS + l % NS) * BTPM_PSTRIDE;
      load_nodes(rec, g4, rec[NX], u[t]);
    }
    const gfloat* rec = prof + (size_t)c * BTPM_PSTRIDE;
    const float Tref = rec[NX];
    sf.u0 = (rec[0] - Tref) * kScale;
    linear_init<4>(u, op[2 * kFrags * 64], op[(2 * kFrags + 1) * 64]);
    float w[BTPM_BLK];
    surface_out(u, w);

    // T_prev and src of a block (past the last: the last again, never used)
    auto fetch = [&](const gfloat* p, int b, float (&v)[BTPM_BLK]) {
      load8(p + (size_t)min(b, nb - 1) * bstride, v);
    };
    auto park = [&](int i, const float (&v)[BTPM_BLK]) {
#pragma unroll
      for (int k = 0; k < BTPM_BLK; ++k) lds_t[i][k][tid] = v[k];
      asm volatile("" ::: "memory");  // keep them in LDS, not in VGPRs
    };
    float nsrc[BTPM_BLK], nprev[BTPM_BLK];
    fetch(Tin, 0, nprev);
    park(0, nprev);
    split_e(0, nprev);
    fetch(Tin, 1, nprev);
    fetch(srcp, 0, nsrc);
    __syncthreads();
    product(0);
    park(1, nprev);
    split_e(1, nprev);
    fetch(Tin, 2, nprev);
    __syncthreads();

    auto block = [&](int b, auto full_tag) {
      constexpr bool FULL = decltype(full_tag)::value;
      const int i = b & 1;
      float tot[BTPM_BLK], t[BTPM_BLK];
#pragma unroll
      for (int k = 0; k < BTPM_BLK; ++k) {
        tot[k] = nsrc[k] + lds_q[i][k * G::kQC + tid];
        t[k] = lds_t[i][k][tid];
      }
      if (FULL) {
        fetch(srcp, b + 1, nsrc);
        load_pieces(i ^ 1, 0);
      }
      surface_steps<FULL>(sf, w, t, tot, gain, m1, es, (double)Tref, tol, cap,
                          ntau - b * BTPM_BLK, [&](int k) {
                            if (!FULL) return;
                            run_pieces(i ^ 1, k);
                            if (k + 1 < BTPM_BLK) load_pieces(i ^ 1, k + 1);
                            // one matrix instruction, then the balance's
#pragma unroll
                            for (int q = 0; q < 3 * G::kM * kPer; ++q) {
                              __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                              __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
                            }
                          });
      if (active) store8(Tout + (size_t)b * bstride, t);
      if (FULL) {
        park(i, nprev);
        split_e(i, nprev);
        fetch(Tin, b + 3, nprev);
      }
      surface_in(u, w);
    };
    for (int b = 0; b + 1 < nb; ++b) {
      block(b, std::true_type{});
      if constexpr (G::kOpLds) {
        linear_block_pairs(u, own_main, [&](int i) { return lop[i * 64]; });
      } else {
        linear_block<4>(u, own_main, [&](int i) { return A[i]; });
      }
      surface_out(u, w);
      __syncthreads();
    }
    block(nb - 1, std::false_type{});
    linear_block_pairs(u, own_tail, [&](int i) { return (h8)op[(kFrags + i) * 64]; });

#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int l = 64 * wave + 16 * t + (lane & 15), ct = crater(l / NS);
      if (ct < 0 || S.frozen[ct]) continue;
      gfloat* r = (gfloat*)S.prof + (size_t)(ct * NS + l % NS) * BTPM_PSTRIDE;
      store_nodes(r, g4, r[NX], u[t]);
    }
    if (active) ((gfloat*)S.prof)[(size_t)c * BTPM_PSTRIDE] = fmaf(sf.u0, 1.0f / kScale, Tref);
  }

  // per-crater freeze test (converged kernel, T175706/thermal_GPU.cu:648-692)
  if (active) atomicMax(&lds_cmax[lcr], __float_as_uint(sf.dm));
  if (tid == 0) lds_cnt = 0;
  __syncthreads();
  if (active && j == 0) {
    const float cm = __uint_as_float(lds_cmax[lcr]);
    S.dmax[gr] = cm;
    bool still = true;
    if (check && cm < S.tacc) {
      S.frozen[gr] = 1;
      still = false;
    }
    if (still) atomicAdd(&lds_cnt, 1);
  }
  __syncthreads();
  if (tid == 0) {
    S.tile_active[tl.tile] = lds_cnt;
    S.tile_work[tl.tile] = S.inst ? 0 : nwork;
  }
}

template __global__ void btpm_conduct_crater_lin<5>(const btpm_tile*, const btpm_set_dev*,
                                                    const btpm_status_dev*);
template __global__ void btpm_conduct_crater_lin<2>(const btpm_tile*, const btpm_set_dev*,
                                                    const btpm_status_dev*);

// Standalone crater self-heating product (tests, tools and the
// allocation-free entry point):
//   q[n][j] = sum_i VF(j->i) e[n][i],  n < ncol, with the kernel's own split.
// The power-of-two unscale comes by value, or from device memory when
// unscale_p is set (tiles packed on the device).
extern "C" __global__ __launch_bounds__(BTPM_CRATER_THREADS) void btpm_contract_kernel(
    const _Float16* __restrict__ vfA, const float* __restrict__ e, float* __restrict__ q,
    int ncol, float unscale_v, const float* __restrict__ unscale_p) {
  __shared__ _Float16 lds_a[2][kMP * kLdsK];
  __shared__ _Float16 lds_b[2][kNP * kLdsK];
  __shared__ float lds_q[BTPM_BLK * kQCols];
  const float unscale = unscale_p != nullptr ? *unscale_p : unscale_v;
  const int tid = (int)threadIdx.x;
  const int n0 = blockIdx.x * kNP;
  stage_vf(vfA, lds_a, tid);
  for (int x = tid; x < kNP * kLdsK; x += BTPM_CRATER_THREADS) {
    const int n = x / kLdsK, i = x - n * kLdsK;
    float v = 0.0f;
    if (i < BTPM_NS && n0 + n < ncol) v = e[(size_t)(n0 + n) * BTPM_NS + i];
    const _Float16 hi = (_Float16)v;
    lds_b[0][x] = hi;
    lds_b[1][x] = (_Float16)(v - (float)hi);
  }
  __syncthreads();
  crater_product<kMP * kLdsK, kNP * kLdsK, kQCols>(lds_a[0], lds_b[0], lds_q, tid >> 6, tid & 63,
                                                   unscale);
  __syncthreads();
  for (int x = tid; x < kNP * BTPM_NS; x += BTPM_CRATER_THREADS) {
    const int n = x / BTPM_NS, jj = x - n * BTPM_NS;
    if (n0 + n < ncol)
      q[(size_t)(n0 + n) * BTPM_NS + jj] =
          lds_q[(n % BTPM_BLK) * kQCols + (n / BTPM_BLK) * BTPM_NS + jj];
  }
}
