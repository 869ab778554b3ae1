// ed_fp64.hpp -- FP64 contraction on gfx950: split sum on FP64 matrix
// instructions, momentum phases one lattice axis at a time.
//
// For every primary derivative d and pair (e, f)
//   Q_d[e,f,x] = sum_splits c_s sum_c conj(W_{L_s}[e,x,c]) W_{R_s}[f,x,c],
//   E_d[p]     = sum_x Phi_p(x) Q_d[e,f,x].
// The phase is a product over the axes, Phi_n(x) = prod_a (c_a + i sgn(n_a) s_a)
// with c_a, s_a = cos, sin(2 pi |n_a| x_a / L_a), so every momentum is a signed
// sum of real moments
//   M_k = sum_z h_k(z) sum_y g_k(y) sum_x f_k(x) Q_d[e,f,x],
// f, g, h each one of the axis functions.  The x sum needs only the few
// distinct f (1, 3 or 5 for the usual momentum sets) at every site; the y sum
// runs once per line of Lx sites, and the z sum over the planes' x-y sums in a
// second kernel (momenta_kernel).
//
// Why: FP64 matrix and vector instructions run at the same rate on gfx950 and
// share the units (16x16x4: 64 cycles for 1024 multiply-adds, v_fma_f64: 4 for
// 64; two waves of a SIMD running one kind each take the sum of both times), so
// the cost of the contraction is its number of multiply-adds.  Contracting 16
// base momenta per site takes 64 per pair and site; the x sum of 33 momenta
// takes 10, next to 24 to 48 for the split sum.
#pragma once
#include <utility>

#include "ed_kernels.hpp"

namespace ed {
namespace f64 {

// Axis-function slots of one launch: F1 functions of x, the i-th followed by
// cap(i) functions of y (NS products f g in all).  Which functions they are is
// run-time data (Args::xt, yt); unused ones are zero.
template <int... S>
struct Pattern {
  static constexpr int F1 = sizeof...(S);
  static constexpr int NS = (S + ...);
  // x function of product k (compile-time k only)
  __host__ __device__ static constexpr int fx(int k) {
    int i = 0, n = 0;
    ((k >= n ? (i = k < n + S ? i : i + 1, n += S) : 0), ...);
    return i;
  }
};

constexpr int NT_MAX = 4;    // 16 x 16 tiles per workgroup
constexpr int NF_MAX = 96;   // moments per launch
constexpr int CHUNK = 32;    // consecutive items given to one XCD (its CUs)

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>)
template <class F, int... I>
__device__ __forceinline__ void static_for(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
// v[i] without an indexed (scratch) access
__device__ __forceinline__ int pick(const short (&v)[NT_MAX], int i) {
  return i == 0 ? v[0] : i == 1 ? v[1] : i == 2 ? v[2] : v[3];
}
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Tiles of one workgroup: tile q pairs e rows 16 rowL[tile[q] & 15] with f rows
// 16 rowR[tile[q] >> 4]; the nL + nR row blocks are staged once for all tiles.
struct Group {
  short nL, nR, nT, pad;
  short rowL[NT_MAX], rowR[NT_MAX], tile[NT_MAX];
};

// One output momentum from the moments: E[+-p] = even +- odd, where a term is
// i^code times moment k (code even: even sum, odd: odd sum).
struct MomTerm {
  int p, n;
  short k[8], code[8];
};

struct Args {
  Geom g;
  int D, P, nd;
  int gt;            // groups per timeslice, over all primary derivatives
  int NT;            // tiles per workgroup: 1 or NT_MAX
  int nsplit;        // line ranges per group: pps whole planes each, or spp parts
  int pps, spp, lps; // of lps lines of one plane (pps = 1)
  int nwork;         // timeslices x gt x nsplit
  int ngrp[2];       // groups of one derivative: all tiles / tiles te <= tf
  int order;         // 0: CHUNK consecutive items per XCD in turn, 1: round robin
  int nf, ns, nmom, t_out0;
  const DPlan* dplan;  // item0: first tile group of the derivative
  const SplitTerm* splits;
  const Group* grp[2];
  const double* xt;  // [Lx + 1][F1]
  const double* yt;  // [Ly][NS]
  const double* zt;  // [Lz][nf], moments ordered by product slot
  const int* zslot;  // [NS + 1] first moment of each product slot
  const MomTerm* mt; // [nmom]
  const double* wgt; // [Ne][Ne] blending weights or nullptr
  // x-y sums [timeslice][group][plane, part][tile][re, im][NS][4][64]
  double* M;
  double2* out;
};

__device__ __forceinline__ int item_of(const Args& a, int b) {
  const int full = a.nwork / (8 * CHUNK) * (8 * CHUNK);
  if (a.order || b >= full) return b;
  const int k = b >> 3;
  return (k / CHUNK) * (8 * CHUNK) + (b & 7) * CHUNK + k % CHUNK;
}

__host__ __device__ constexpr int k4_of(int NQ) { return (NQ + 1) / 2; }  // 1 KB pieces staged per site and row block

// LDS of a workgroup: all of a CU's for four tiles (8 waves of up to 256
// registers fill it anyway), a quarter for one tile (2 waves: four workgroups
// a CU); and the sites of a stage that fit it three times.
__host__ __device__ constexpr int lds_of(int NT) { return NT == 1 ? 40960 : 163840; }
__host__ __device__ inline int sites_of(int NT, int RT, int K4) {
  const int s = lds_of(NT) / (3 * RT * K4 * 1024);
  return s < 1 ? 1 : s > 8 ? 8 : s;
}

// 64 lanes x 16 bytes from per-lane global addresses to consecutive LDS bytes
// at lds_off, without passing through registers.  Issued as assembly because
// the compiler would drain it before the next LDS read; nothing is returned in
// a register, and stage_wait() runs before the barrier that publishes the data.
__device__ __forceinline__ void stage_16(const double2* p, uint32_t lds_off) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(p), "s"(lds_off) : "memory", "m0");
}
// at most n (uniform) of this wave's latest loads are still in flight
__device__ __forceinline__ void stage_wait(int n) {
  if (n >= 6) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
  else if (n >= 4) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

typedef const __attribute__((address_space(4))) double* cptr;  // uniform table: scalar loads

// One workgroup: up to four 16 x 16 tiles, two waves per tile (one the real,
// one the imaginary part of Q), sweeping the sites of a range of lines.
// NQ: matrix instructions per site and part, K = 4 NQ >= 6 nsplit real terms.
//
// Term j' = 2 j + comp of the split sum multiplies component comp of L_j
// with the same component of R_j for Re conj(L) R, and with the other one
// (sign + for comp 0, - for comp 1) for Im conj(L) R: both parts read the same
// staged (split, colour) pairs j and differ in a lane offset and a sign.
//
// Stage: S sites x (nL + nR) row blocks x K4 pieces of 1 KB (4 pairs j x 16
// rows) in a ring of three.  The operands of a site are read from LDS while the
// matrix instructions of the site before it run, so a stage is used up one
// site early: its barrier comes before its last site's matrix instructions,
// which hide the first reads of the next stage, and a stage has two stage
// times to land.
// Sharing the row blocks among the four tiles halves the bytes per pair
// against one tile per workgroup.
//
// Bound: the FP64 units (62 % of their rate at 32^3, Nev 200, 33 momenta, 13
// derivatives: 167 ms per eight timeslices against 106 for its multiply-adds
// alone; 291 ms for the contraction that formed 16 momenta per site).  The
// rest, from copies of the kernel without one part: issuing the stages' loads
// 11 % (L2 hits or not: 1 %), barriers 3 %, LDS reads 2 %, line ends 5 %, and
// the two waves a SIMD holds (s1 and s2 fill the registers) waiting for the
// same unit.  Registers set four tiles and two waves per SIMD; LDS sets S.
template <class PAT, int NQ, int PART>
__device__ __forceinline__ void contract_body(const double2* __restrict__ Wt, const Args& a, const DPlan& dp,
                                              const Group& gr, char* lds, int l0, int l1, double* __restrict__ Mw) {
  typedef mfma<double>::acc acc_t;
  constexpr int K4 = k4_of(NQ), F1 = PAT::F1, NS = PAT::NS;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, g4 = lane >> 4;
  const int q = wave >> 1;
  const Geom& g = a.g;
  const int J = 3 * dp.nsplit;
  const int RT = gr.nL + gr.nR, S = uni(sites_of(a.NT, RT, K4));
  const int site_e = 3 * g.NeP;  // workspace elements per site
  const int s0 = l0 * g.Lx, nsite = (l1 - l0) * g.Lx, nblk = (nsite + S - 1) / S;

  // staging role: the first half of the waves stages the left row blocks, the
  // second half the right ones, site i of a stage by wave i mod (half)
  const int half = a.NT;  // waves per side
  const bool right = wave >= half;
  const int i0 = right ? wave - half : wave;
  const int nrow = right ? gr.nR : gr.nL;
  const double2* src[K4];  // row block 0, site 0
#pragma unroll
  for (int k = 0; k < K4; ++k) {
    const int j = 4 * k + g4, jj = j < J ? j : 0;  // pairs past the last repeat the first (coefficient 0)
    const SplitTerm st = a.splits[dp.first + jj / 3];
    src[k] = Wt + widx(g, right ? st.nR : st.nL, 0, jj % 3, l16);
  }
  const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)lds;
  const int site_b = RT * K4 * 1024;
  const int nown = i0 < S ? (S - i0 + half - 1) / half : 0;  // sites of a stage this wave loads
  const int nl = nown * nrow * K4;                            // its loads
  int ro[NT_MAX];                                             // first element of each row block
#pragma unroll
  for (int rt = 0; rt < NT_MAX; ++rt) ro[rt] = 16 * (right ? gr.rowR[rt] : gr.rowL[rt]);
  const uint32_t dst0 = lds0 + i0 * site_b + (right ? gr.nL : 0) * K4 * 1024;
  auto stage = [&](int b, int slot) {  // slot = b mod 3
    uint32_t d = dst0 + slot * S * site_b;
    int s = b * S + i0;
    for (int n = 0; n < nown; ++n, s += half, d += half * site_b) {
      const size_t so = (size_t)(s0 + min(s, nsite - 1)) * site_e;  // the last stage repeats its last site
#pragma unroll
      for (int rt = 0; rt < NT_MAX; ++rt) {
        if (rt < nrow) {
          size_t o = so + ro[rt];
          asm volatile("" : "+s"(o));  // no instruction: one offset per row block, not an address per load
#pragma unroll
          for (int k = 0; k < K4; ++k) stage_16(src[k] + o, d + (rt * K4 + k) * 1024);
        }
      }
    }
  };

  // Coefficients of this lane's left values: pair 4 k + g4 of a full piece k
  // (both components, two matrix instructions: NG pieces), and term
  // 8 NG + g4 of a last half piece (REM).
  constexpr int NG = NQ / 2, REM = NQ & 1;
  auto coeff = [&](int j) { return j < J ? (double)a.splits[dp.first + j / 3].coeff : 0.0; };
  const int comp = g4 & 1;
  double cf[NG], cr = 0.0;
#pragma unroll
  for (int k = 0; k < NG; ++k) cf[k] = coeff(4 * k + g4);
  if (REM) cr = (PART && comp ? -1.0 : 1.0) * coeff(4 * NG + (g4 >> 1));
  const bool mine = q < gr.nT;
  const int tile = mine ? pick(gr.tile, q) : 0, tl = tile & 15, tr = tile >> 4;
  // full pieces: 16 bytes per lane, consecutive lanes consecutive; the last
  // half piece: 8 bytes (comp of the left value, for the imaginary part the
  // other component of the right one)
  const int offA = tl * K4 * 1024 + lane * 16, offB = (gr.nL + tr) * K4 * 1024 + lane * 16;
  const int remA = tl * K4 * 1024 + NG * 1024 + (g4 >> 1) * 256 + l16 * 16 + comp * 8;
  const int remB = (gr.nL + tr) * K4 * 1024 + NG * 1024 + (g4 >> 1) * 256 + l16 * 16 + (PART ? 1 - comp : comp) * 8;

  const cptr xt = (cptr)a.xt, yt = (cptr)a.yt;
  double s1[F1][4], s2[NS][4];  // x sums of the line, x-y sums of the plane
#pragma unroll
  for (int r = 0; r < 4; ++r) {
#pragma unroll
    for (int m = 0; m < F1; ++m) s1[m][r] = 0.0;
#pragma unroll
    for (int m = 0; m < NS; ++m) s2[m][r] = 0.0;
  }
  stage(0, 0);
  if (nblk > 1) stage(1, 1);
  if (nblk > 2) stage(2, 2);
  stage_wait(0);
  __syncthreads();
  // Nothing reads stage b any more (its last operands are in registers) and
  // stage b + 1 is about to be read: it has landed here, stage b + 2 may still
  // be in flight, and stage b + 3 takes the place of stage b.
  auto next_stage = [&](int b) {
    if (b + 1 >= nblk) return;
    stage_wait(b + 2 < nblk ? nl : 0);
    // without the wait for scalar and LDS reads in flight that __syncthreads
    // brings: this wave's reads of stage b have returned (settle)
    asm volatile("s_barrier" ::: "memory");
  };
  if (!mine) {
    for (int b = 0, slot = 0; b < nblk; ++b, slot = slot == 2 ? 0 : slot + 1) {
      next_stage(b);
      if (b + 3 < nblk) stage(b + 3, slot);
    }
    return;
  }
  constexpr int NR = NG <= 3 ? NG : 3;  // pieces read ahead (all of them up to four split terms)
  struct Ops {
    double2 A[NR], B[NR];
    double a, b;
  };
  auto load = [&](Ops& o, const char* pb) {
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      o.A[k] = *(const double2*)(pb + offA + k * 1024);
      o.B[k] = *(const double2*)(pb + offB + k * 1024);
    }
    if (REM) {
      o.a = *(const double*)(pb + remA);
      o.b = *(const double*)(pb + remB);
    }
  };
  // One site: its successor's operands are requested, then its matrix
  // instructions and the x sums of the site before (value P, functions f) run,
  // so that neither waits for the other's results.  The two waves of a SIMD
  // (w and w + 4) issue their loads at different sites of a stage: a wave
  // stands while the CU's address path takes them, and the other one keeps the
  // matrix unit busy.
  int blk = 0, i = 0, slot = 0;
  const int issue = right ? (S - 1) >> 1 : S - 1;
  const char* pb = lds;
  auto site = [&](const Ops& cur, Ops& nxt, const acc_t& P, const double* f) {
    const char* const pc = pb;
    const bool last = i + 1 == S;
    auto ahead = [&] {
      if (last) {
        next_stage(blk);
        slot = slot == 2 ? 0 : slot + 1;
        pb = lds + slot * S * site_b;
      } else {
        pb += site_b;
      }
      load(nxt, pb);  // past the last site: a stage no longer in use, read for nothing
    };
    // past four split terms the last operands are still read from this stage
    // below, so its barrier waits for them
    constexpr bool whole = NG <= NR;
    if (whole) {
      ahead();
      __builtin_amdgcn_sched_barrier(0);
    }
    acc_t Q = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
      if (k == 2 * NG) {
        Q = mfma<double>::mac(cr * cur.a, cur.b, Q);
      } else {
        const int m = k >> 1;
        const double2 A = m < NR ? cur.A[m < NR ? m : 0] : *(const double2*)(pc + offA + m * 1024);
        const double2 B = m < NR ? cur.B[m < NR ? m : 0] : *(const double2*)(pc + offB + m * 1024);
        // Re conj(L) R = Lr Rr + Li Ri, Im conj(L) R = Lr Ri - Li Rr
        if (PART == 0) Q = k & 1 ? mfma<double>::mac(cf[m] * A.y, B.y, Q) : mfma<double>::mac(cf[m] * A.x, B.x, Q);
        else Q = k & 1 ? mfma<double>::mac(-cf[m] * A.y, B.x, Q) : mfma<double>::mac(cf[m] * A.x, B.y, Q);
      }
    }
    if (!whole) {
      asm volatile("" : "+v"(Q));  // no instruction: the products above are formed before the barrier
      ahead();
    }
#pragma unroll
    for (int j = 0; j < 4 * F1; ++j) s1[j / 4][j % 4] = fma(f[j / 4], P[j % 4], s1[j / 4][j % 4]);
    if (i == issue) {
      // the stage three ahead of the one last used up, in its place
      const int b = last ? blk + 3 : blk + 2;
      if (b >= 3 && b < nblk) stage(b, slot == 0 ? 2 : slot - 1);
    }
    if (last) {
      ++blk;
      i = 0;
    } else {
      ++i;
    }
    return Q;
  };
  // Operands read a site ago are here (lgkmcnt 0).  Waited for before the next
  // reads are issued: scalar and LDS reads return in no common order, so a wait
  // after that would be for all of them.
  auto settle = [] {
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_sched_barrier(0);
  };
  Ops X, Y;
  load(X, pb);
  int y = l0 % g.Ly;
  for (int line = l0; line < l1; ++line) {
    acc_t P = {0.0, 0.0, 0.0, 0.0};
    double f1[F1];  // x functions of the site P belongs to
#pragma unroll
    for (int m = 0; m < F1; ++m) f1[m] = 0.0;
    cptr xp = xt;
    for (int x = 0; x < g.Lx; x += 2, xp += 2 * F1) {
      double n0[F1], n1[F1];
      settle();
#pragma unroll
      for (int m = 0; m < F1; ++m) {
        n0[m] = xp[m];
        n1[m] = xp[F1 + m];  // the table ends with a row of zeros
      }
      P = site(X, Y, P, f1);
#pragma unroll
      for (int m = 0; m < F1; ++m) f1[m] = n0[m];
      if (x + 1 < g.Lx) {
        settle();
        P = site(Y, X, P, f1);
#pragma unroll
        for (int m = 0; m < F1; ++m) f1[m] = n1[m];
      } else {
        X = Y;
      }
    }
    double gy[NS];
#pragma unroll
    for (int m = 0; m < NS; ++m) gy[m] = yt[y * NS + m];
#pragma unroll
    for (int m = 0; m < F1; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) s1[m][r] = fma(f1[m], P[r], s1[m][r]);
    static_for(std::make_integer_sequence<int, NS>{}, [&](auto k) {
      constexpr int m = decltype(k)::value, xf = PAT::fx(m);
#pragma unroll
      for (int r = 0; r < 4; ++r) s2[m][r] = fma(gy[m], s1[xf][r], s2[m][r]);
    });
#pragma unroll
    for (int m = 0; m < F1; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) s1[m][r] = 0.0;
    if (++y < g.Ly && line + 1 < l1) continue;
    // end of the plane (or of its part in this range)
#pragma unroll
    for (int m = 0; m < NS; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        Mw[(m * 4 + r) * 64 + lane] = s2[m][r];
        s2[m][r] = 0.0;
      }
    Mw += (size_t)a.NT * 2 * NS * 256;
    y = 0;
  }
}

template <class PAT, int NQX>
__global__ __launch_bounds__(128 * NT_MAX, 1) void contract_kernel(const double2* __restrict__ W, Args a) {
  extern __shared__ __align__(16) char lds[];
  const int w = uni(item_of(a, blockIdx.x));
  const int per_t = a.gt * a.nsplit;
  const int tb = w / per_t;
  int r = w - tb * per_t;
  int di = 0;
  while (di + 1 < a.nd && uni(a.dplan[di + 1].item0) * a.nsplit <= r) ++di;
  DPlan dp = a.dplan[di];
  dp.first = uni(dp.first), dp.nsplit = uni(dp.nsplit), dp.mirror = uni(dp.mirror), dp.item0 = uni(dp.item0);
  r -= dp.item0 * a.nsplit;
  const int ng = dp.mirror ? a.ngrp[1] : a.ngrp[0];
  const int split = r / ng, gi = r - split * ng;
  Group gr = (dp.mirror ? a.grp[1] : a.grp[0])[gi];
  gr.nL = (short)uni(gr.nL), gr.nR = (short)uni(gr.nR), gr.nT = (short)uni(gr.nT);
#pragma unroll
  for (int k = 0; k < NT_MAX; ++k)
    gr.rowL[k] = (short)uni(gr.rowL[k]), gr.rowR[k] = (short)uni(gr.rowR[k]), gr.tile[k] = (short)uni(gr.tile[k]);
  // lines of this range: pps whole planes, or part split % spp of one plane
  const int z0 = split / a.spp * a.pps, part = split % a.spp;
  const int l0 = z0 * a.g.Ly + part * a.lps;
  const int l1 = a.spp > 1 ? min(l0 + a.lps, (z0 + 1) * a.g.Ly) : min(z0 + a.pps, a.g.Lz) * a.g.Ly;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const double2* Wt = W + (size_t)tb * a.g.nW * a.g.V3P * 3 * a.g.NeP;
  const int seg = z0 * a.spp + part;
  double* Mw = a.M + (((size_t)(tb * a.gt + dp.item0 + gi) * (a.g.Lz * a.spp) + seg) * a.NT * 2 + wave) * (PAT::NS * 256);
  const int nq = (6 * dp.nsplit + 3) >> 2;
  auto go = [&](auto n) {
    constexpr int NQ = decltype(n)::value;
    if (wave & 1) contract_body<PAT, NQ, 1>(Wt, a, dp, gr, lds, l0, l1, Mw);
    else contract_body<PAT, NQ, 0>(Wt, a, dp, gr, lds, l0, l1, Mw);
  };
  if (NQX > 6 && nq > 6) go(std::integral_constant<int, 12>{});
  else if (nq == 6) go(std::integral_constant<int, 6>{});
  else if (nq == 5) go(std::integral_constant<int, 5>{});
  else if (nq == 3) go(std::integral_constant<int, 3>{});
  else go(std::integral_constant<int, 2>{});
}

// Output momenta of one quarter tile (rows 4 r .. 4 r + 3 of 16 x 16 pairs) of
// one group: the z sums of the planes' x-y sums, then every momentum of the
// launch with its weight and its Hermitian partner.  Bound by HBM (the x-y sums
// and the outputs, once each).
// grid (timeslices x gt x NT x 4), block 256, LDS 2 nf x 64 doubles
__global__ __launch_bounds__(256) void momenta_kernel(Args a) {
  extern __shared__ __align__(16) char lds[];
  double* v = (double*)(void*)lds;  // [re, im][nf][64]
  const int rq = blockIdx.x & 3;
  int b = blockIdx.x >> 2;
  const int q = b % a.NT;
  b /= a.NT;
  const int tb = b / a.gt, gi = b - tb * a.gt;
  int di = 0;
  while (di + 1 < a.nd && a.dplan[di + 1].item0 <= gi) ++di;
  const DPlan dp = a.dplan[di];
  const Group gr = (dp.mirror ? a.grp[1] : a.grp[0])[gi - dp.item0];
  if (q >= gr.nT) return;
  const int tile = pick(gr.tile, q), te = pick(gr.rowL, tile & 15), tf = pick(gr.rowR, tile >> 4);
  const int nseg = a.g.Lz * a.spp, wave = uni(threadIdx.x >> 6);
  const size_t seg_e = (size_t)a.NT * 2 * a.ns * 256;  // doubles per plane part
  constexpr int NZ = 6;                                // z functions of one product per pass over the planes
  for (int row = wave; row < 2 * a.ns; row += 4) {
    const int part = row / a.ns, slot = row - part * a.ns;
    const double* S = a.M + (size_t)b * nseg * seg_e + ((size_t)((q * 2 + part) * a.ns + slot) * 4 + rq) * 64 +
                      (threadIdx.x & 63);
    const int k1 = uni(a.zslot[slot + 1]);
    for (int k0 = uni(a.zslot[slot]); k0 < k1; k0 += NZ) {
      // two chains, the plane parts from the last one down
      double m0[NZ] = {}, m1[NZ] = {};
      auto add = [&](int sg, double (&m)[NZ]) {
        const double s = S[sg * seg_e];
        const double* h = a.zt + (size_t)(sg / a.spp) * a.nf + k0;  // the table ends with NZ zeros
#pragma unroll
        for (int k = 0; k < NZ; ++k) m[k] = fma(h[k], s, m[k]);
      };
      int sg = 0;
#pragma unroll 2
      for (; sg + 1 < nseg; sg += 2) {
        add(nseg - 1 - sg, m0);
        add(nseg - 2 - sg, m1);
      }
      if (sg < nseg) add(nseg - 1 - sg, m0);
#pragma unroll
      for (int k = 0; k < NZ; ++k)
        if (k0 + k < k1) v[(part * a.nf + k0 + k) * 64 + (threadIdx.x & 63)] = m0[k] + m1[k];
    }
  }
  __syncthreads();
  const int pair = threadIdx.x & 63;
  const int e = 16 * te + mfma<double>::row(pair >> 4, rq), f = 16 * tf + (pair & 15);
  const int Ne = a.g.Ne;
  if (e >= Ne || f >= Ne) return;
  const size_t plane = (size_t)Ne * Ne, tbase = (size_t)(a.t_out0 + tb) * a.D * a.P;
  const double wef = a.wgt ? a.wgt[(size_t)e * Ne + f] : 1.0, wfe = a.wgt ? a.wgt[(size_t)f * Ne + e] : 1.0;
  const bool partner = partner_writes(dp, te, tf);
  const double sg = (double)dp.sign;
  for (int m = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); m < a.nmom; m += 4) {
    const MomTerm* mt = &a.mt[m];
    double er = 0.0, ei = 0.0, od_r = 0.0, od_i = 0.0;
    for (int j = 0; j < mt->n; ++j) {
      const int k = mt->k[j], code = mt->code[j];
      const double re = v[k * 64 + pair], im = v[(a.nf + k) * 64 + pair];
      if (code == 0) er += re, ei += im;
      else if (code == 2) er -= re, ei -= im;
      else if (code == 1) od_r -= im, od_i += re;
      else od_r += im, od_i -= re;
    }
    const double epr = er + od_r, epi = ei + od_i, emr = er - od_r, emi = ei - od_i;
    a.out[(tbase + (size_t)dp.d * a.P + mt->p) * plane + (size_t)e * Ne + f] = make_double2(epr * wef, epi * wef);
    // E_{rev d}[p] = sign * E_d[-p]^dagger
    if (partner)
      a.out[(tbase + (size_t)dp.partner * a.P + mt->p) * plane + (size_t)f * Ne + e] =
          make_double2(sg * emr * wfe, -sg * emi * wfe);
  }
}

}  // namespace f64
}  // namespace ed
