// bmg_chain.hip -- the device-resident PMV sampler: FP64 model state in LDS,
// Cholesky add / remove / full refactorisation, sum-tree proposals, the
// moves of src/sampler.hpp:899-1669 and the schedule of src/sampler.cpp:
// 626-834, one workgroup per chain.
//
// All threads of a workgroup run the scalar control flow redundantly on
// identical register copies (the random stream included), so every decision
// is uniform; the O(n k) parts use all 256 threads and the O(k^2) triangular
// and Givens sweeps use wave 0.  Triangular solves and the Cholesky
// factorisation are right-looking: each element receives its subtractions in
// the same order as the netlib loops of the CPU oracle, but fused, with
// reciprocals in place of divisions, and a removal's rotations are found by
// another method, so factors agree to rounding and log-likelihoods to 1e-10.
// Compiled with contraction off, so that only the fused steps written out are
// fused.
#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>

#include <type_traits>
#include "bmg_chain.h"
#include "bmg_device.h"
#include "../../include/bmagwa_hip.h"

using namespace bmg;

#define LOG_HALF (-0.69314718055994528622676398299518041312694549560546875)
#define TLEV_LDS 512

__device__ __forceinline__ int P(int c) { return c * (c + 1) / 2; }

// A log-likelihood that is not finite (+inf when the residual term reaches
// zero, NaN) can only come from rounding in a near-singular design; it is
// taken as -inf, so such a proposal is rejected (as in the oracle).
__device__ __forceinline__ double finite_ll(double v) { return isfinite(v) ? v : -INFINITY; }

// element i (runtime) of a small register array without dynamic indexing,
// which would place the whole per-lane state in scratch memory.  Each
// element passes through an empty register constraint, so the compiler
// cannot fold the selects back into one load at a computed address.
template <typename T, int N>
__device__ __forceinline__ T sel(const T (&a)[N], int i) {
  T r = a[0];
  asm volatile("" : "+v"(r));
#pragma unroll
  for (int q = 1; q < N; ++q) {
    T v = a[q];
    asm volatile("" : "+v"(v));
    r = (i == q) ? v : r;
  }
  return r;
}
template <typename T, int N>
__device__ __forceinline__ void put(T (&a)[N], int i, T v) {
#pragma unroll
  for (int q = 0; q < N; ++q) a[q] = (i == q) ? v : a[q];
}

// A pointer that every lane of a wave holds alike, as a scalar register pair
// into global memory.  The chain's pointers are read from LDS, and the
// compiler would take one for an address anywhere (flat instructions, whose
// waits also cover every LDS access in flight) that may differ by lane.
template <typename T>
__device__ __forceinline__ T* gp(T* p) {
  uint64_t u = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)u);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
  u = (uint64_t)hi << 32 | lo;
  return (T*)(__attribute__((address_space(1))) T*)u;
}

// ------------------------------------------------------------- state -----
// The proposed model's factor (packed upper): an LDS array up to 160
// columns; a larger capacity keeps it in a per-chain global array (L2/HBM),
// whose address thread 0 stores in the LDS member at kernel entry.  The
// member is a plain array in the LDS case (as a base-class member the
// compiler's code for the triangular loops was a fifth slower).
constexpr int KMAX_LDS = 160;
// a chain returns from the 256-column code once its model is this many
// columns inside the smaller capacity (a change costs a store and a load of
// the chain's state, about 20 us; nearly every move adds fewer SNPs)
constexpr int CAP_BACK = 12;
struct GlobalFactor {
  double* p;
  __device__ __forceinline__ operator double*() const { return gp(p); }
};
template <int KMAX>
using FactorT = std::conditional_t<(KMAX <= KMAX_LDS),
                                   double[KMAX * (KMAX + 1) / 2 + (KMAX + 63) / 64 * 64 - KMAX + BMG_LPAD],
                                   GlobalFactor>;

// counters of ChainScal that change in every iteration
struct Counters {
  uint64_t n_accepted, n_acpt[4], n_moves[4];
  uint64_t tr_count, th_count, th_loci_len, th_beta_len;
};

// The dataset's, the chain's and its arrays' descriptions, the counters, the
// move-size tables and the phase clocks are copies too: read through their
// global addresses, each use between two stores was a vector load of several
// hundred cycles in front of the work, and each counter a load-add-store
// that wave 0 waited out.  (With the pointers made global ones and the chain's
// scalars kept in registers as well, 500 iterations of 16 chains at n =
// 10,000, p = 500,000 went from 339 to 309 ms, of 64 chains on four datasets
// of up to 20,000 individuals from 137 to 116 ms.)
template <int KMAX>
struct Smem {
  DevData D;
  ChainConst K;
  ChainArrays A;
  Counters cnt;
  uint64_t prof[24];
  double cdf[3][BMG_MAXMS];              // move-size distributions: add/remove, swap, state change
  double r_ms_sum[BMG_MAXMS], r_ms_n[BMG_MAXMS];
  FactorT<KMAX> L;                       // proposed model's factor (packed upper)
  double xy[KMAX], v[KMAX], d[KMAX];     // proposed model vectors
  double beta[KMAX], mu[KMAX];           // the chain's beta / mu_beta
  double work[KMAX + 64];
  double c_xy[KMAX], c_v[KMAX], c_d[KMAX];
  int32_t slot[KMAX], snp[KMAX];         // per column: slot in xxs, SNP
  int32_t c_slot[KMAX], c_snp[KMAX];
  uint32_t loci[KMAX], c_loci[KMAX];     // per locus
  int32_t xi1[KMAX], xi2[KMAX], c_xi1[KMAX], c_xi2[KMAX];
  int8_t xtype[KMAX], c_xtype[KMAX], tind[KMAX], c_tind[KMAX];
  uint64_t mi[BMG_MAXMS], mi_add[BMG_MAXMS], mi_rem[BMG_MAXMS];
  int64_t mi_map[BMG_MAXMS];
  uint8_t mi_isadd[BMG_MAXMS];
  uint64_t rm_list[2 * BMG_MAXMS];
  uint64_t marks[BMG_MAXMS];
  int32_t mark_val[BMG_MAXMS];
  uint64_t sc_perm[BMG_MAXMS], sc_from[BMG_MAXMS], sc_to[BMG_MAXMS];
  double tlev[2][TLEV_LDS];              // sum-tree levels >= 2 (add, rem)
  int32_t win[512];                      // window of the current model_inds
  // column slots in use (the slot space is that of the per-chain arrays, the
  // same in every capacity, so a chain keeps its slots when it changes it)
  uint64_t slots_cur[BMG_KMAXG / 64], slots_prop[BMG_KMAXG / 64];
  int32_t iacc[KMAX + 1];                // integer column dots of new_column_dots
  int32_t iacc2[KMAX + 1];               // the next addition's dots, formed ahead
  // delayed rejection: factor block and v of the toggled loci's columns, the
  // walk's products of diagonals and residual terms by column, the loci's
  // log d, the prior change by loci added, and the moved SNPs' proposal
  // weights
  double ex_L[BMG_DR_COLS * (BMG_DR_COLS + 1) / 2];
  double ex_v[BMG_DR_COLS], ex_pp[BMG_DR_COLS + 1], ex_ss[BMG_DR_COLS + 1];
  double ex_ld[BMG_DR_MAX], ex_pa[BMG_DR_MAX + 1];
  double dq_add[BMG_DR_MAX], dq_rem[BMG_DR_MAX];
  uint8_t ex_b2n[BMG_DR_MAX];
  // undo journal of an add/remove move's sum-tree writes: the global
  // entries it overwrote (leaf and level 1, in order) and a copy of the LDS
  // levels taken when the move began
  double tj_old[2 * BMG_MAXMS][2];
  uint64_t tj_ind[2 * BMG_MAXMS];        // leaf index, tree in bit 63
  double tj_tlev[2][TLEV_LDS];
  double bq[BMG_MAXMS];                  // proposal weights of the reverse move
  double red[8];
  long long redi[8];
  double bcd[4];
  long long bci[4];
};

// The chain's stream with its next 64 blocks at hand, one in each lane of the
// wave: a Philox block is ten rounds of dependent 32-bit multiplies, about
// 1,000 cycles, and every lane would compute the same one for each draw.  A
// draw is a read of its lane; the stream itself is unchanged.  (With the
// DPP scan below a pick went from 3.6 to 3.0 us, and with the terms' draws in
// parallel 500 iterations of 16 chains over 500,000 SNPs from 122.8 to 118.6 ms.)
struct ChainRng : Rng {
  uint64_t base;                         // counter of lane 0's block
  uint32_t w[4];                         // this lane's block
};
struct Words { uint32_t w[4]; };
static __device__ __noinline__ Words rng_block_at(uint32_t k0, uint32_t k1, uint64_t c, uint32_t c2, uint32_t c3) {
  Words o;
  o.w[0] = (uint32_t)c; o.w[1] = (uint32_t)(c >> 32); o.w[2] = c2; o.w[3] = c3;
  philox10(o.w[0], o.w[1], o.w[2], o.w[3], k0, k1);
  return o;
}
// the lane that holds the next block; the stream moves on by one
__device__ __forceinline__ int rng_next_lane(ChainRng& r) {
  const uint64_t c = (uint64_t)r.c1 << 32 | r.c0;
  uint32_t at = __builtin_amdgcn_readfirstlane(c - r.base < 64 ? (uint32_t)(c - r.base) : 64u);
  if (at >= 64) {
    const Words o = rng_block_at(r.k0, r.k1, c + (threadIdx.x & 63), r.c2, r.c3);
    r.base = c;
#pragma unroll
    for (int q = 0; q < 4; ++q) r.w[q] = o.w[q];
    at = 0;
  }
  if (++r.c0 == 0) ++r.c1;
  return (int)at;
}
__device__ __forceinline__ double rng_u01(ChainRng& r) {
  const int at = rng_next_lane(r);
  return words_u01(__builtin_amdgcn_readlane(r.w[0], at), __builtin_amdgcn_readlane(r.w[1], at));
}

struct Reg {
  ChainRng rng;
  int cols, nloci, Ns[5];
  double syx, ldq, ldl, ll;
  int c_cols, c_nloci, c_Ns[5];
  double c_syx, c_ldq, c_ldl, c_ll;
  double sigma2, alpha, alpha2, ita2[4];
  int beta_len, mu_computed;
  int lmin;
  int n_rm, n_marks;
  int movesize;
  double tot_add, tot_rem;
  int err;
  int learn_on;
  int tj_on, tj_n;                       // journal active, entries
  int job_tr;                            // tree write that waits (-1: none)
  uint64_t job_ind;
  long long warm;                        // SNP a pick has drawn (or -1): see warm_next
  int warm_add;                          // ... for addition
  long long pre_snp;                     // column_key of the dots in iacc2 (or -1)
  int pre_slot;                          // and the slot its value words went to
  double tj_tot[2];                      // tree totals when the move began
};

// how far a chain has come: the next iteration, whether its refresh is done
// already, and whether the other capacity's code takes over there
struct Progress { uint64_t iter; int change, refreshed; };

template <int KMAX>
struct Ctx {
  Smem<KMAX>& S;
  Reg& R;
  const DevData& D;
  const ChainConst& K;
  const ChainArrays& A;
  uint64_t* prof;   // the chain's phase counters (thread 0 writes)
};

__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }
__device__ __forceinline__ int wave_id() { return threadIdx.x >> 6; }

// ------------------------------------------------------------ genotypes ---
// a column of SNP `snp` under one coding, as one number (-1: none)
__device__ __forceinline__ long long column_key(long long snp, int coding) {
  return snp < 0 ? -1 : snp * 4 + coding;
}

// x_j^T y (FP64) of one SNP's packed row, where no table was made at set-up
// (the Model API): lane-strided words, 16 fields each in order, then the
// workgroup sum
__device__ __forceinline__ double dot_y_block(const uint32_t* __restrict__ w, uint32_t W,
                                              const double* __restrict__ y, int coding, double* red) {
  double s = 0.0;
  for (uint32_t k = threadIdx.x; k < W; k += BMG_BLOCK) {
    uint32_t x = w[k];
    const double* yy = y + 16 * (size_t)k;
#pragma unroll
    for (int f = 0; f < 16; ++f) {
      int iv = code_ival((x >> (2 * f)) & 3u, coding);
      if (iv) s += (double)iv * yy[f];
    }
  }
  return block_sum(s, red);
}

// The Makefile compiles this file twice so that the two kernels build in
// parallel: BMG_CHAIN_UNIT 1 holds the sampler's, 2 the Model methods'.
#ifndef BMG_CHAIN_UNIT
#define BMG_CHAIN_UNIT 0
#endif
#define BMG_UNIT(u) (BMG_CHAIN_UNIT == 0 || BMG_CHAIN_UNIT == (u))

template <int KMAX>
__device__ __forceinline__ double snp_dot_y(Ctx<KMAX>& C, uint64_t snp, int coding) {
  const double* pre = gp(C.D.xy[coding]);
  if (pre) return pre[snp];   // made at set-up
  return dot_y_block(gp(C.D.g) + snp * C.D.W32, C.D.W32, gp(C.D.y), coding, C.S.red);
}

// value word of a packed word: the coded genotype (0..2) in each 2-bit field
__device__ __forceinline__ uint32_t value_word(uint32_t w, int coding) {
  const uint32_t lo = w & BMG_EVEN, hi = (w >> 1) & BMG_EVEN;
  const uint32_t het = hi & ~lo, hom = hi & lo;
  // A: het + 2 hom, H: het, D: het + hom, R: hom
  const uint32_t one = (coding == 3 ? 0u : het) | (coding >= 2 ? hom : 0u);
  return one | (coding == 0 ? hom << 1 : 0u);
}

// acc[c] = x_c^T x_new for the constant column c = 0, the model's columns c
// in [me, cols) and the new column itself, c = cols (covariate columns:
// cov_dots).  Exact integer dots: the slot copies of the model's columns hold
// value words, whose even fields (masked in place) and odd fields (the rest,
// four times their value) meet the new column's in two 8-way unsigned 4-bit
// dot products (v_dot8_u32_u4); the odd sum is divided by four at the end.
//
// A group of SPAN lanes (16, 32 or 64, as the columns are short or long)
// holds NP pieces of 16 bytes a lane of the new column, decoded once, and
// streams whole columns past them: consecutive lanes read consecutive 16
// bytes, up to four columns' pieces are in flight while those before are
// summed, and a column's sum meets in its group by DPP adds.  Bound by the
// L2 reads of the columns (2,560 bytes each at n = 10,000).  (With a lane
// reading 64 consecutive bytes, each load instruction touched 32 cache lines
// for a quarter of their bytes, and 40 lanes added their sums to one LDS
// word: 8.7 us per addition at 105 columns on four waves, 12 us on three.)
// Columns longer than SPAN x NP pieces go in several passes.  Threads
// [T0, T0 + NTH) take part (the whole workgroup, or waves 1-3 while wave 0
// runs a triangular sweep); the first group also writes the new column's
// value words to its slot copy xnew.
template <int KMAX, int T0, int NTH, int SPAN, int NP>
__device__ __forceinline__ void column_dots_np(Ctx<KMAX>& C, uint64_t snp_new, int coding, int cols,
                                               uint32_t* __restrict__ xnew, int32_t* acc) {
  constexpr int UC = NP > 3 ? 2 : 4;          // columns in flight
  constexpr int GRP = NTH / SPAN;             // groups side by side
  Smem<KMAX>& S = C.S;
  const uint32_t W = C.D.W32, W4 = W / 4;     // words and 16-byte pieces per column
  const uint4* __restrict__ wn = (const uint4*)(gp(C.D.g) + snp_new * W);
  const char* __restrict__ xcol = (const char*)gp(C.A.xcol);
  const int me = C.D.me;
  const int tid = (int)threadIdx.x - T0;
  const int grp = tid / SPAN, t = tid % SPAN;
  auto group_sum = [](int v) -> int {         // valid in a group's last lane
    v += dpp_i32<0x111, 0xf>(v);
    v += dpp_i32<0x112, 0xf>(v);
    v += dpp_i32<0x114, 0xf>(v);
    v += dpp_i32<0x118, 0xf>(v);
    if (SPAN > 16) v += dpp_i32<0x142, 0xa>(v);
    if (SPAN > 32) v += dpp_i32<0x143, 0xc>(v);
    return v;
  };
  for (uint32_t p0 = 0; p0 < W4; p0 += SPAN * NP) {
    uint32_t ne[NP][4], no[NP][4];            // even / odd fields of the new column
    uint32_t off[NP];                         // byte offset of this lane's pieces in a column
    uint4 raw[NP];
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      const uint32_t pc = p0 + t + q * SPAN;
      off[q] = (pc < W4 ? pc : W4 - 1) * 16;
      raw[q] = wn[off[q] / 16];
    }
    // group g sums columns me + g + GRP k; every group runs group 0's rounds
    const int n_col = cols - me;
    const int rounds = n_col > 0 ? ((n_col + GRP - 1) / GRP + UC - 1) / UC : 0;
    auto column = [&](int r, int u) { return me + grp + (UC * r + u) * GRP; };
    auto load = [&](int r, uint4 (&w)[UC][NP]) {
#pragma unroll
      for (int u = 0; u < UC; ++u) {
        const int c = column(r, u);
        const uint32_t base = (uint32_t)S.slot[c < cols ? c : cols - 1] * W * 4;
#pragma unroll
        for (int q = 0; q < NP; ++q) w[u][q] = *(const uint4*)(xcol + (base + off[q]));
      }
    };
    // the first columns are on their way while the new one arrives (from
    // HBM, where the model's columns are in L2)
    uint4 wa[UC][NP], wb[UC][NP];
    if (rounds > 0) load(0, wa);
    uint32_t s_one = 0, s_self = 0;
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      const bool in = p0 + t + q * SPAN < W4;
      const uint32_t xs[4] = {raw[q].x, raw[q].y, raw[q].z, raw[q].w};
      uint32_t vw[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        vw[u] = in ? value_word(xs[u], coding) : 0u;
        ne[q][u] = vw[u] & 0x33333333u;
        no[q][u] = (vw[u] >> 2) & 0x33333333u;
      }
      if (grp == 0) {
        if (in) *(uint4*)((char*)xnew + off[q]) = make_uint4(vw[0], vw[1], vw[2], vw[3]);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          s_one = __builtin_amdgcn_udot8(0x11111111u, ne[q][u], s_one, false);
          s_one = __builtin_amdgcn_udot8(0x11111111u, no[q][u], s_one, false);
          s_self = __builtin_amdgcn_udot8(ne[q][u], ne[q][u], s_self, false);
          s_self = __builtin_amdgcn_udot8(no[q][u], no[q][u], s_self, false);
        }
      }
    }
    auto put_sum = [&](int c, int v) {
      if (t == SPAN - 1) acc[c] = p0 == 0 ? v : acc[c] + v;
    };
    if (tid < 64) {                           // the wave that holds group 0
      const int a = group_sum((int)s_one), b = group_sum((int)s_self);
      if (grp == 0) { put_sum(0, a); put_sum(cols, b); }
    }
    auto sum = [&](int r, const uint4 (&w)[UC][NP]) {
      int v[UC];
#pragma unroll
      for (int u = 0; u < UC; ++u) {
        uint32_t se = 0, so = 0;
#pragma unroll
        for (int q = 0; q < NP; ++q) {
          const uint32_t xs[4] = {w[u][q].x, w[u][q].y, w[u][q].z, w[u][q].w};
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const uint32_t e = xs[k] & 0x33333333u;
            se = __builtin_amdgcn_udot8(e, ne[q][k], se, false);
            so = __builtin_amdgcn_udot8(xs[k] ^ e, no[q][k], so, false);
          }
        }
        v[u] = (int)(se + (so >> 2));
      }
#pragma unroll
      for (int u = 0; u < UC; ++u) v[u] = group_sum(v[u]);
#pragma unroll
      for (int u = 0; u < UC; ++u) {
        const int c = column(r, u);
        if (c < cols) put_sum(c, v[u]);
      }
    };
    for (int r = 0; r < rounds; r += 2) {
      if (r + 1 < rounds) load(r + 1, wb);
      sum(r, wa);
      if (r + 1 < rounds) {
        if (r + 2 < rounds) load(r + 2, wa);
        sum(r + 1, wb);
      }
    }
  }
}

// the group width and pieces per lane for the column length: the narrowest
// group that holds a column in one piece a lane, and from 64 pieces on two,
// three or five pieces a lane, the fewest of these that hold it; longer columns
// (past 20,480 individuals) go in passes of five.  (A column just past a line
// pays for the pieces that it leaves empty: 300 iterations of 8 chains of
// 50-70 SNPs take 25.0 ms at n = 12,288 and 35.5 at 14,000, 33.2 at 20,480 and
// 45.7 at 20,481, 48.8 at 25,000, 75.5 at 50,000.)
template <int KMAX, int T0, int NTH>
__device__ __forceinline__ void column_dots(Ctx<KMAX>& C, uint64_t snp_new, int coding, int cols, uint32_t* xnew,
                                            int32_t* acc) {
  if ((int)threadIdx.x < T0) return;
  const uint32_t W4 = C.D.W32 / 4;
  if (W4 <= 16) column_dots_np<KMAX, T0, NTH, 16, 1>(C, snp_new, coding, cols, xnew, acc);
  else if (W4 <= 32) column_dots_np<KMAX, T0, NTH, 32, 1>(C, snp_new, coding, cols, xnew, acc);
  else if (W4 <= 64) column_dots_np<KMAX, T0, NTH, 64, 1>(C, snp_new, coding, cols, xnew, acc);
  else if (W4 <= 128) column_dots_np<KMAX, T0, NTH, 64, 2>(C, snp_new, coding, cols, xnew, acc);
  else if (W4 <= 192) column_dots_np<KMAX, T0, NTH, 64, 3>(C, snp_new, coding, cols, xnew, acc);
  else column_dots_np<KMAX, T0, NTH, 64, 5>(C, snp_new, coding, cols, xnew, acc);
}

// S.work[c] = e_c^T x_new for the covariate columns c in [1, me): each
// thread sums over its individuals, then a fixed-order block reduction
template <int KMAX>
__device__ __forceinline__ void cov_dots(Ctx<KMAX>& C, uint64_t snp_new, int coding_new) {
  const int me = C.D.me;
  const uint32_t* __restrict__ wn = gp(C.D.g) + snp_new * C.D.W32;
  for (int c = 1; c < me; ++c) {
    const double* __restrict__ e = gp(C.D.E) + (size_t)(c - 1) * C.D.n_pad;
    double acc = 0.0;
    for (uint32_t i = threadIdx.x; i < C.D.n; i += BMG_BLOCK) {
      const int iv = code_ival((wn[i >> 4] >> (2 * (i & 15))) & 3u, coding_new);
      if (iv > 0) acc += (double)iv * e[i];
    }
    acc = block_sum(acc, C.S.red);
    if (threadIdx.x == 0) C.S.work[c] = acc;
  }
  __syncthreads();
}

// S.work[c] = x_c^T x_new for c in [0, cols] (covariates included), and
// the new column's value words into its slot copy xnew
template <int KMAX>
__device__ __forceinline__ void new_column_dots(Ctx<KMAX>& C, uint64_t snp_new, int coding_new, int cols,
                                                uint32_t* xnew) {
  Smem<KMAX>& S = C.S;
  column_dots<KMAX, 0, BMG_BLOCK>(C, snp_new, coding_new, cols, xnew, S.iacc);
  __syncthreads();
  for (int c = threadIdx.x; c <= cols; c += BMG_BLOCK) S.work[c] = (double)S.iacc[c];
  __syncthreads();
  if (C.D.me > 1) cov_dots(C, snp_new, coding_new);
}

// ----------------------------------------------------- triangular (wave 0)
// value of lane `src` (uniform) of a double held by every lane
__device__ __forceinline__ double readlane_d(double v, int src) {
  int2 h = *reinterpret_cast<int2*>(&v);
  h.x = __builtin_amdgcn_readlane(h.x, src);
  h.y = __builtin_amdgcn_readlane(h.y, src);
  return *reinterpret_cast<double*>(&h);
}

// The triangular sweeps.  Wave 0 only.  Lane l holds the vector's entries
// l + 64 t (t < NT, the fewest that hold the vector) and the reciprocals of
// their rows' diagonal entries in registers; the outer loops over t are
// unrolled so the register arrays are only ever indexed by constants.  Per
// row the owner's scaled entry is read across lanes and every lane subtracts
// its coefficient times it: the serial chain is one multiply, one cross-lane
// read and one fused multiply-subtract, with no division, no branches and no
// masks.  A lane at or past its row reads another column's entry into a value
// it no longer needs (its result was kept when its row came), and rows past
// the vector's end change nothing that is kept, so whole blocks of SWEEP
// rows run.  Bound by that chain: the coefficients of a block are read into
// registers while the block before it is applied, so no row waits for them.
// (Read two rows ahead, each row took half an LDS round trip, 78 ns, and with
// the factor in global memory half an L2 round trip, 125-180 ns.)  Per element
// the subtractions come in row order, as in the sequential loop; the
// reciprocal and the fused update round differently from its divisions (by an
// ulp), which the log-likelihoods' 1e-10 agreement with the oracle absorbs.
constexpr int SWEEP = 8;

// x := T^-T x, T the n x n triangle of the factor L that begins at row and
// column o (dtrsv Upper/Trans order).  ALPHA: a2 of entry i becomes 1 + the
// sum of the squares of the results 0..i.
template <int NT, bool ALPHA>
__device__ __forceinline__ void sweep_ut(const double* L, int o, int n, const double (&dg)[NT], double (&b)[NT],
                                         double (&xo)[NT], double (&a2)[NT]) {
  const int lane = lane_id();
  int base[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int j = lane + 64 * t;
    base[t] = j < n ? P(o + j) + o : 0;
    xo[t] = 0.0;
    if (ALPHA) a2[t] = 1.0;
  }
  double al = 1.0;
#pragma unroll
  for (int ti = 0; ti < NT; ++ti) {
    const int i0 = 64 * ti;
    const int iend = n < 64 * (ti + 1) ? n : 64 * (ti + 1);
    if (i0 >= iend) break;
    double ca[SWEEP][NT], cb[SWEEP][NT];
    auto load = [&](int i, double (&c)[SWEEP][NT]) {
#pragma unroll
      for (int t = ti; t < NT; ++t)
#pragma unroll
        for (int q = 0; q < SWEEP; ++q) c[q][t] = L[base[t] + i + q];
    };
    auto rows = [&](int i, const double (&c)[SWEEP][NT]) {
#pragma unroll
      for (int q = 0; q < SWEEP; ++q) {
        const int owner = (i + q) & 63;
        const double xi = readlane_d(b[ti] * dg[ti], owner);
        xo[ti] = lane == owner ? xi : xo[ti];
        if (ALPHA) {
          al = fma(xi, xi, al);
          a2[ti] = lane == owner ? al : a2[ti];
        }
#pragma unroll
        for (int t = ti; t < NT; ++t) b[t] = fma(-c[q][t], xi, b[t]);
      }
    };
    load(i0, ca);
#pragma unroll 1
    for (int i = i0; i < iend; i += 2 * SWEEP) {
      if (i + SWEEP < iend) load(i + SWEEP, cb);
      rows(i, ca);
      if (i + SWEEP < iend) {
        if (i + 2 * SWEEP < iend) load(i + 2 * SWEEP, ca);
        rows(i + SWEEP, cb);
      }
    }
  }
}

template <int NT>
__device__ __forceinline__ void trsv_ut_nt(const double* L, double* x, int m) {
  const int lane = lane_id();
  double b[NT], dg[NT], xo[NT], a2[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int j = lane + 64 * t;
    b[t] = j < m ? x[j] : 0.0;
    dg[t] = j < m ? 1.0 / L[P(j) + j] : 1.0;
  }
  sweep_ut<NT, false>(L, 0, m, dg, b, xo, a2);
#pragma unroll
  for (int t = 0; t < NT; ++t) { const int j = lane + 64 * t; if (j < m) x[j] = xo[t]; }
}

// x := U^-T x for x[0..m).  Wave 0 only.
template <int KMAX>
__device__ __forceinline__ void trsv_ut_w0(Smem<KMAX>& S, double* x, int m) {
  const double* L = S.L;
  if (m <= 64) trsv_ut_nt<1>(L, x, m);
  else if (KMAX <= 128 || m <= 128) trsv_ut_nt<2>(L, x, m);
  else if (KMAX <= 192 || m <= 192) trsv_ut_nt<3>(L, x, m);
  else trsv_ut_nt<4>(L, x, m);
}

// x := U^-1 x (dtrsv Upper/NoTrans, back substitution): step j subtracts
// column j (consecutive addresses) times the owner's scaled entry, columns
// in descending order.  A zero x_j leaves every entry as it was, as the
// reference's skip of zero entries does.
template <int NT>
__device__ __forceinline__ void trsv_un_nt(const double* L, double* x, int m) {
  const int lane = lane_id();
  double b[NT], rd[NT], xo[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int j = lane + 64 * t;
    b[t] = j < m ? x[j] : 0.0;
    rd[t] = j < m ? 1.0 / L[P(j) + j] : 1.0;
    xo[t] = 0.0;
  }
#pragma unroll
  for (int tj = NT - 1; tj >= 0; --tj) {
    const int j0 = 64 * tj;
    const int jend = m < 64 * (tj + 1) ? m : 64 * (tj + 1);
    if (j0 >= jend) continue;
    double ca[SWEEP][NT], cb[SWEEP][NT];
    // columns j, j - 1, ... (below the first: column 0)
    auto load = [&](int j, double (&c)[SWEEP][NT]) {
#pragma unroll
      for (int s = 0; s < SWEEP; ++s) {
        const int pj = j - s > 0 ? P(j - s) : 0;
#pragma unroll
        for (int q = 0; q <= tj; ++q) c[s][q] = L[pj + lane + 64 * q];
      }
    };
    auto steps = [&](int j, const double (&c)[SWEEP][NT]) {
#pragma unroll
      for (int s = 0; s < SWEEP; ++s) {
        if (j - s >= j0) {
          const int owner = (j - s) & 63;
          const double xj = readlane_d(b[tj] * rd[tj], owner);
          xo[tj] = lane == owner ? xj : xo[tj];
#pragma unroll
          for (int q = 0; q <= tj; ++q) b[q] = fma(-xj, c[s][q], b[q]);
        }
      }
    };
    load(jend - 1, ca);
#pragma unroll 1
    for (int j = jend - 1; j >= j0; j -= 2 * SWEEP) {
      if (j - SWEEP >= j0) load(j - SWEEP, cb);
      steps(j, ca);
      if (j - SWEEP >= j0) {
        if (j - 2 * SWEEP >= j0) load(j - 2 * SWEEP, ca);
        steps(j - SWEEP, cb);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) { const int j = lane + 64 * t; if (j < m) x[j] = xo[t]; }
}

template <int KMAX>
__device__ __forceinline__ void trsv_un_w0(Smem<KMAX>& S, double* x, int m) {
  const double* L = S.L;
  if (m <= 0) return;
  if (m <= 64) trsv_un_nt<1>(L, x, m);
  else if (KMAX <= 128 || m <= 128) trsv_un_nt<2>(L, x, m);
  else if (KMAX <= 192 || m <= 192) trsv_un_nt<3>(L, x, m);
  else trsv_un_nt<4>(L, x, m);
}

// netlib drotg (as the oracle restates it)
__device__ __forceinline__ void drotg(double& a, double& b, double& c, double& s) {
  double sa = a, sb = b;
  double roe = (fabs(sa) > fabs(sb)) ? sa : sb;
  double scale = fabs(sa) + fabs(sb);
  double r, z;
  if (scale == 0.0) { c = 1.0; s = 0.0; r = 0.0; z = 0.0; }
  else {
    double as = sa / scale, bs = sb / scale;
    r = scale * sqrt(as * as + bs * bs);
    r = (roe >= 0.0 ? 1.0 : -1.0) * r;
    c = sa / r; s = sb / r;
    z = 1.0;
    if (fabs(sa) > fabs(sb)) z = s;
    if (fabs(sb) >= fabs(sa) && c != 0.0) z = 1.0 / c;
  }
  a = r; b = z;
}

// Removing column cr of the m x m factor U (the result of LINPACK dchex job
// 2 + drop + sign fix, src/symmmatrix.cpp:166-195): the rows above cr lose the
// column; below, the triangle T of the later columns takes up the row r =
// U[cr, cr+1..] by rotations that zero r entry by entry, T'T'^T = T^T T + r r^T.
// dchex generates rotation k from the entries that rotation k - 1 left, a
// square root and a division in a serial chain per row.  Here the rotations
// are found first: with w = T^-T r, rotation k has cos = alpha_k-1 / alpha_k
// and sin = w_k / alpha_k, alpha_k^2 = 1 + w_0^2 + ... + w_k^2 (Gill, Golub,
// Murray and Saunders 1974, method C1), so the serial chain is one forward
// sweep, the square roots and divisions are a lane per row, and the rotations
// are then applied with every lane going down its own columns: a multiply and
// a fused multiply-add per row in the chain.  cos, sin >= 0 in cos's case
// give positive diagonals, dchex's after its sign fix.  (dchex's order took
// 14 us at 105 columns, 250 ns a row, and 30-40 us with the factor in global
// memory.  Over removals in a row from factors of LD columns up to r =
// 0.999999 both orders' factors, log-determinants and v are equally far from
// 80-bit ones.)
//
// The triangle's new rows go straight to their place in the compacted factor
// (logical column cr + j from physical column cr + 1 + j): a step stores row
// cr + k of a column, which the lane of the column before read as its row at
// an earlier step.  v (U^T v = X^T y) goes through the same rotations, so
// after the removal it solves the new factor's system without a second
// triangular solve (the reference re-solves, src/model.hpp:530-545; the two
// agree to rounding).  Wave 0 only.
template <int KMAX, int NT>
__device__ __forceinline__ void downdate_w0(Smem<KMAX>& S, double* L, int m, int cr) {
  const int lane = lane_id();
  const int o = cr + 1, n = m - 1 - cr;
  double r[NT], b[NT], dg[NT], w[NT], a2[NT], cc[NT], ss[NT], vo[NT], vn[NT];
  int src[NT], dst[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int j = lane + 64 * t;
    const bool on = j < n;
    src[t] = on ? P(o + j) + o : 0;
    dst[t] = on ? P(cr + j) + cr : 0;
    r[t] = b[t] = on ? L[src[t] - 1] : 0.0;
    dg[t] = on ? 1.0 / L[src[t] + j] : 1.0;
    vo[t] = on ? S.v[o + j] : 0.0;
    vn[t] = 0.0;
  }
  double vr = S.v[cr];
  sweep_ut<NT, true>(L, o, n, dg, b, w, a2);
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    a2[t] = sqrt(a2[t]);
    double before = dpp_f64<0x138, 0xf>(a2[t]);          // wave_shr:1
    const double first = t == 0 ? 1.0 : readlane_d(a2[t > 0 ? t - 1 : 0], 63);
    before = lane == 0 ? first : before;
    const double inv = 1.0 / a2[t];
    cc[t] = before * inv;
    ss[t] = w[t] * inv;
  }
#pragma unroll
  for (int ti = 0; ti < NT; ++ti) {
    const int k0 = 64 * ti;
    const int kend = n < 64 * (ti + 1) ? n : 64 * (ti + 1);
    if (k0 >= kend) break;
    double ua[SWEEP][NT], ub[SWEEP][NT];
    auto load = [&](int k, double (&u)[SWEEP][NT]) {
#pragma unroll
      for (int t = ti; t < NT; ++t)
#pragma unroll
        for (int q = 0; q < SWEEP; ++q) u[q][t] = L[src[t] + k + q];
    };
    auto rows = [&](int kb, const double (&u)[SWEEP][NT]) {
#pragma unroll
      for (int q = 0; q < SWEEP; ++q) {
        const int k = kb + q, owner = k & 63;
        const double c = readlane_d(cc[ti], owner), s = readlane_d(ss[ti], owner);
        const double vk = readlane_d(vo[ti], owner);
        const double vnew = fma(c, vk, s * vr);
        vr = fma(c, vr, -(s * vk));
        vn[ti] = lane == owner ? vnew : vn[ti];
#pragma unroll
        for (int t = ti; t < NT; ++t) {
          const int j = lane + 64 * t;
          const double x = fma(c, u[q][t], s * r[t]);
          r[t] = fma(c, r[t], -(s * u[q][t]));
          if (j >= k && j < n) L[dst[t] + k] = x;
        }
      }
    };
    load(k0, ua);
#pragma unroll 1
    for (int k = k0; k < kend; k += 2 * SWEEP) {
      if (k + SWEEP < kend) load(k + SWEEP, ub);
      rows(k, ua);
      if (k + SWEEP < kend) {
        if (k + 2 * SWEEP < kend) load(k + 2 * SWEEP, ua);
        rows(k + SWEEP, ub);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) { const int j = lane + 64 * t; if (j < n) S.v[cr + j] = vn[t]; }
}

// The downdate on wave 0, while wave 1 moves the rows above cr of the later
// columns down by one column, in ascending order of destination (every source
// lies above every earlier destination, so a batch never overwrites what a
// later one reads; the two waves touch disjoint entries).  With work to do
// ahead, which touches neither the factor nor v and lasts longer than the
// downdate, waves 1-3 do that and wave 0 moves the rows afterwards.
// `side`, another wave's worth of such work, is done by the wave that is
// through first.
template <int KMAX, typename Extra, typename Side>
__device__ __forceinline__ void chol_downdate(Smem<KMAX>& S, int m, int cr, bool ahead, Extra extra, Side side) {
  double* L = S.L;
  if (wave_id() == 0) {
    const int n = m - 1 - cr;
    if (n <= 64) downdate_w0<KMAX, 1>(S, L, m, cr);
    else if (KMAX <= 128 || n <= 128) downdate_w0<KMAX, 2>(S, L, m, cr);
    else if (KMAX <= 192 || n <= 192) downdate_w0<KMAX, 3>(S, L, m, cr);
    else downdate_w0<KMAX, 4>(S, L, m, cr);
  }
  if (wave_id() == (ahead ? 0 : 1)) {
    // rows [0, cr) of logical columns [cr, m - 2]: physical column jl + 1
    // -> jl, element k = (jl - cr) * cr + i in ascending order
    constexpr int DEEP = KMAX <= KMAX_LDS ? 4 : 16;
    const int total = (m - 1 - cr) * cr;
    const float rcr = cr > 0 ? 1.0f / (float)cr : 0.0f;
    for (int k0 = 0; k0 < total; k0 += 64 * DEEP) {
      double x[DEEP];
      int to[DEEP];
#pragma unroll
      for (int u = 0; u < DEEP; ++u) {
        const int k = k0 + 64 * u + lane_id();
        int q = (int)((float)k * rcr);
        if (q * cr > k) --q;
        if ((q + 1) * cr <= k) ++q;
        const int jl = cr + q, i = k - q * cr;
        to[u] = P(jl) + i;
        x[u] = k < total ? L[P(jl + 1) + i] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < DEEP; ++u)
        if (k0 + 64 * u + lane_id() < total) L[to[u]] = x[u];
    }
  }
  if (wave_id() == (ahead ? 0 : 3)) side();
  if (ahead && wave_id() != 0) extra();
  __syncthreads();
}

// Full factorisation of S.L (m x m, in place) in panels of CF_PB rows;
// returns 0 if not positive definite.  Per panel [k0, k1): wave 0 factors
// the diagonal block in registers (lane l holds column k0 + l; the pivot
// and each row-k entry reach the other lanes by cross-lane reads, so the
// block needs no barrier); then a thread per later column computes that
// column's panel rows from the block (a forward substitution of CF_PB
// steps); then the trailing update gives a lane to each row i >= k1 and
// the four waves every fourth column j, so a wave's 64 lanes read and
// write 64 consecutive entries of one column and all read the same panel
// entries of column j.  Every element receives the sequential loop's
// subtractions in k order; they are fused, and the pivots' reciprocals (the
// hardware's reciprocal square root and two Newton steps) take the place of
// the square roots and divisions, whose chains of up to 250 cycles per row
// bound the block and the panel.  A refresh of a 135-column model, of which
// this is most, went from 213 to 179 us, of one of 58 two-column terms from
// 183 to 156; a 60-SNP likelihood is as far from the 64-bit one as before
// (1.2e-16).
constexpr int CF_PB = 16;
template <int KMAX>
__device__ __forceinline__ int chol_full(Smem<KMAX>& S, int m) {
  constexpr int PB = CF_PB;
  constexpr int NT = (KMAX + 63) / 64;
  __syncthreads();
  const int lane = lane_id(), wv = wave_id();
  for (int k0 = 0; k0 < m; k0 += PB) {
    const int k1 = k0 + PB < m ? k0 + PB : m;
    const int nb = k1 - k0;
    if (wv == 0) {
      const int j = k0 + lane;
      const bool own = lane < nb;
      double blk[PB];
#pragma unroll
      for (int r = 0; r < PB; ++r) blk[r] = (own && r <= lane) ? S.L[P(j) + k0 + r] : 0.0;
      int ok = 1;
      double rec = 0.0;
#pragma unroll
      for (int kk = 0; kk < PB; ++kk) {
        if (kk < nb) {
          const double akk = readlane_d(blk[kk], kk);
          if (!(akk > 0.0)) { ok = 0; break; }
          // 1 / sqrt(akk): the hardware's estimate and two Newton steps
          double y = __builtin_amdgcn_rsq(akk);
          const double h = 0.5 * akk;
          y = y * fma(-h * y, y, 1.5);
          y = y * fma(-h * y, y, 1.5);
          const double u = blk[kk] * y;        // the pivot's own lane: akk / sqrt(akk)
          rec = lane == kk ? y : rec;
          blk[kk] = lane >= kk ? u : blk[kk];
#pragma unroll
          for (int r = kk + 1; r < PB; ++r) {
            if (r < nb) {
              const double ur = readlane_d(u, r);
              if (lane >= r) blk[r] = fma(-ur, u, blk[r]);
            }
          }
        }
      }
#pragma unroll
      for (int r = 0; r < PB; ++r) if (own && r <= lane) S.L[P(j) + k0 + r] = blk[r];
      if (own) S.work[lane] = rec;
      if (lane == 0) S.bci[0] = ok;
    }
    __syncthreads();
    if (!S.bci[0]) { __syncthreads(); return 0; }
    // the panel rows of the columns past the block
    {
      const int j = k1 + (int)threadIdx.x;
      if (j < m) {
        double c[PB];
        double* col = S.L + P(j) + k0;
#pragma unroll
        for (int r = 0; r < PB; ++r) c[r] = r < nb ? col[r] : 0.0;
#pragma unroll
        for (int i = 0; i < PB; ++i) {
          if (i < nb) {
            const double* bc = S.L + P(k0 + i) + k0;   // block column k0 + i
#pragma unroll
            for (int k = 0; k < i; ++k) c[i] = fma(-bc[k], c[k], c[i]);
            c[i] = c[i] * S.work[i];
          }
        }
#pragma unroll
        for (int r = 0; r < PB; ++r) if (r < nb) col[r] = c[r];
      }
    }
    __syncthreads();
    // trailing update: a_ij -= sum_k u_ki u_kj over the panel, i in [k1, j]
    for (int q = 0; q < NT; ++q) {
      const int i = k1 + lane + 64 * q;
      if (64 * q >= m - k1) break;
      double ui[PB];
#pragma unroll
      for (int k = 0; k < PB; ++k) ui[k] = (i < m && k < nb) ? S.L[P(i) + k0 + k] : 0.0;
      for (int j = k1 + 64 * q + wv; j < m; j += 4) {
        const double* cj = S.L + P(j);
        double uj[PB];
#pragma unroll
        for (int k = 0; k < PB; ++k) uj[k] = k < nb ? cj[k0 + k] : 0.0;
        const int ic = i <= j ? i : j;
        double a = cj[ic];
#pragma unroll
        for (int k = 0; k < PB; ++k) a = fma(-ui[k], uj[k], a);   // rows past the panel: 0
        if (i <= j) S.L[P(j) + i] = a;
      }
    }
    __syncthreads();
  }
  return 1;
}

// ------------------------------------------------------------- sum trees --
// Levels 0 and 1 in global memory, levels >= 2 in LDS; see the oracle's
// orc_sumtree for the definition (64-ary, Hillis-Steele group sums).
template <int KMAX>
__device__ __forceinline__ double tree_val(Ctx<KMAX>& C, int tr, int h, uint64_t i) {
  if (h < 2) {
    const double* base = tr == 0 ? gp(C.A.tree_add) : gp(C.A.tree_rem);
    return base[C.D.lev_off[h] + i];
  }
  return C.S.tlev[tr][C.D.lev_off[h] - C.D.lev_off[2] + i];
}

// a double moved across lanes by a DPP control (both halves; lanes whose
// source is out of range get 0)
template <int CTRL>
__device__ __forceinline__ double dpp_d(double v) {
  int2 h = *reinterpret_cast<int2*>(&v);
  h.x = __builtin_amdgcn_update_dpp(0, h.x, CTRL, 0xf, 0xf, false);
  h.y = __builtin_amdgcn_update_dpp(0, h.y, CTRL, 0xf, 0xf, false);
  return *reinterpret_cast<double*>(&h);
}

// inclusive scan by DPP adds alone (rows of 16, then the rows' totals): the
// picks' descent, which needs the sums only to compare and to carry
__device__ __forceinline__ double dpp_scan(double v) {
  v += dpp_f64<0x111, 0xf>(v);   // row_shr 1, 2, 4, 8
  v += dpp_f64<0x112, 0xf>(v);
  v += dpp_f64<0x114, 0xf>(v);
  v += dpp_f64<0x118, 0xf>(v);
  v += dpp_f64<0x142, 0xa>(v);   // row_bcast 15, 31
  v += dpp_f64<0x143, 0xc>(v);
  return v;
}

// a group's sum in every lane, in the order the trees are built with: the
// last element of the Hillis-Steele scan is a balanced pairwise sum ((v62 +
// v63) + (v60 + v61)) + ..., which a butterfly over pairs, quads, eights, rows
// and halves forms with the same operands (partners by DPP quad permutations
// and mirrors, then lane swaps)
__device__ __forceinline__ double group_total(double v) {
  v = v + dpp_d<0xB1>(v);    // quad_perm [1,0,3,2]
  v = v + dpp_d<0x4E>(v);    // quad_perm [2,3,0,1]
  v = v + dpp_d<0x141>(v);   // row_half_mirror
  v = v + dpp_d<0x140>(v);   // row_mirror
  {
    const bool odd = ((threadIdx.x & 63) >> 4) & 1;
    int2 h = *reinterpret_cast<int2*>(&v), o;
    const auto a = __builtin_amdgcn_permlane16_swap((unsigned)h.x, (unsigned)h.x, false, false);
    const auto b = __builtin_amdgcn_permlane16_swap((unsigned)h.y, (unsigned)h.y, false, false);
    o.x = (int)(odd ? a[0] : a[1]);
    o.y = (int)(odd ? b[0] : b[1]);
    v = v + *reinterpret_cast<double*>(&o);
  }
  return readlane_d(v, 0) + readlane_d(v, 32);
}

// While wave 0 walks a tree for the next pick, wave 1 reads what the SNP of
// the pick before will need (its genotypes if it is to be added, its entries
// in the other tree, its weight there and its x.y), so that HBM's latency, and
// the address translation's, is not waited for when the move is applied.
// The values are dropped: the reads bring the lines into L2.
template <int KMAX>
__device__ __forceinline__ void warm_next(Ctx<KMAX>& C) {
  if (C.R.warm < 0) return;
  if (wave_id() == 1) {
    const int lane = lane_id();
    const uint64_t j = (uint64_t)C.R.warm;
    const double* other = C.R.warm_add ? gp(C.A.tree_rem) : gp(C.A.tree_add);
    const double* w = C.R.warm_add ? gp(C.A.q_rem) : gp(C.A.q_add);
    double x = other[C.D.lev_off[0] + 64 * (j >> 6) + lane] + w[j];
    if (C.D.top >= 1) x += other[C.D.lev_off[1] + 64 * (j >> 12) + lane];
    uint32_t g = 0;
    if (C.R.warm_add) {
      const double* xy = gp(C.D.xy[C.D.type == BMG_AH ? 0 : C.D.type]);
      if (xy) x += xy[j];
      const uint4* row = (const uint4*)(gp(C.D.g) + j * C.D.W32);
      for (uint32_t q = lane; q < C.D.W32 / 4; q += 64) g ^= row[q].x;
    }
    asm volatile("" : : "v"(x), "v"(g));
  }
  C.R.warm = -1;
}

// set leaf i to its weight (unzero) or 0 (zero) and update the path; the
// new total goes to S.bcd[1].  One wave.
template <int KMAX>
__device__ __forceinline__ void tree_set_wave(Ctx<KMAX>& C, int tr, uint64_t i, int zero) {
  double* g0 = tr == 0 ? gp(C.A.tree_add) : gp(C.A.tree_rem);
  const double* w = tr == 0 ? gp(C.A.q_add) : gp(C.A.q_rem);
  double total;
  const int lane = lane_id();
  double nv = zero ? 0.0 : w[i];
  // issue the level-0 and level-1 group loads together
  uint64_t g1 = i >> 6;
  double c0 = g0[C.D.lev_off[0] + 64 * g1 + lane];
  double c1 = C.D.top >= 1 ? g0[C.D.lev_off[1] + 64 * (g1 >> 6) + lane] : 0.0;
  if (C.R.tj_on) {
    const double o0 = readlane_d(c0, (int)(i & 63)), o1 = readlane_d(c1, (int)(g1 & 63));
    if (lane == 0) {
      C.S.tj_old[C.R.tj_n][0] = o0; C.S.tj_old[C.R.tj_n][1] = o1;
      C.S.tj_ind[C.R.tj_n] = i | ((uint64_t)tr << 63);
    }
  }
  if (lane == (int)(i & 63)) c0 = nv;
  double gs = group_total(c0);
  if (lane == 0) g0[C.D.lev_off[0] + i] = nv;
  if (C.D.top == 0) {
    total = gs;
  } else {
    if (lane == 0) g0[C.D.lev_off[1] + g1] = gs;
    if (lane == (int)(g1 & 63)) c1 = gs;
    gs = group_total(c1);
    uint64_t gi = g1 >> 6;   // entry index at level 2
    for (int h = 2; h <= C.D.top; ++h) {
      double* lv = C.S.tlev[tr] + (C.D.lev_off[h] - C.D.lev_off[2]);
      if (lane == 0) lv[gi] = gs;
      uint64_t grp = gi >> 6;
      double c = lv[64 * grp + lane];
      if (lane == (int)(gi & 63)) c = gs;
      gs = group_total(c);
      gi = grp;
    }
    total = gs;
  }
  if (lane == 0) C.S.bcd[1] = total;
}
template <int KMAX>
__device__ __forceinline__ void tree_set_done(Ctx<KMAX>& C, int tr) {
  const double total = C.S.bcd[1];
  if (tr == 0) C.R.tot_add = total; else C.R.tot_rem = total;
  if (C.R.tj_on) C.R.tj_n++;
}
template <int KMAX>
__device__ __forceinline__ void tree_set(Ctx<KMAX>& C, int tr, uint64_t i, int zero) {
  warm_next(C);
  if (wave_id() == 0) tree_set_wave(C, tr, i, zero);
  __syncthreads();
  tree_set_done(C, tr);
  __syncthreads();
}

// A tree write that waits for a wave with nothing to do: an add/remove move
// leaves it here before it changes the model, and the model update's idle
// wave does it beside the sweep or the downdate (two round trips to memory,
// 2.2 us).  With the logarithms of a move's steps taken side by side as well,
// 500 iterations of 16 chains went from 118.6 to 110.5 ms, of 64 chains on four
// datasets from 84.8 to 78.3.  job_wave: by one wave; job_done: by all, after a barrier;
// job_finish: by all, where the update did not come to it.
template <int KMAX>
__device__ __forceinline__ void job_wave(Ctx<KMAX>& C) {
  if (C.R.job_tr >= 0) tree_set_wave(C, C.R.job_tr, C.R.job_ind, 0);
}
template <int KMAX>
__device__ __forceinline__ void job_done(Ctx<KMAX>& C) {
  if (C.R.job_tr >= 0) tree_set_done(C, C.R.job_tr);
  C.R.job_tr = -1;
}
template <int KMAX>
__device__ __forceinline__ void job_finish(Ctx<KMAX>& C) {
  if (C.R.job_tr < 0) return;
  const int tr = C.R.job_tr;
  C.R.job_tr = -1;
  __syncthreads();
  tree_set(C, tr, C.R.job_ind, 0);
}

// Pick a leaf with probability w_i / total and zero it, reusing the groups the
// descent read: the path's sums are recomputed from them in tree_set's order,
// so the tree ends up exactly as after a tree_set(zero) of the leaf.  *w_out:
// the picked leaf's weight.
template <int KMAX>
__device__ __forceinline__ uint64_t tree_pick_zero(Ctx<KMAX>& C, int tr, double u, double* w_out) {
  double* g0 = tr == 0 ? gp(C.A.tree_add) : gp(C.A.tree_rem);
  warm_next(C);
  if (wave_id() == 0) {
    const int lane = lane_id();
    double total = tr == 0 ? C.R.tot_add : C.R.tot_rem;
    double r = u * total, carry = 0.0;
    uint64_t g = 0;
    long long res = 0;
    double cl[BMG_TREE_LEV];             // this lane's value in the group read at each level
#pragma unroll
    for (int h = 0; h < BMG_TREE_LEV; ++h) cl[h] = 0.0;
    for (int h = C.D.top; h >= 0; --h) {
      double c = tree_val(C, tr, h, 64 * g + lane);
#pragma unroll
      for (int q = 0; q < BMG_TREE_LEV; ++q) if (q == h) cl[q] = c;
      double s = dpp_scan(c);
      unsigned long long m1 = __ballot(c > 0.0 && r < carry + s);
      unsigned long long nz = __ballot(c > 0.0);
      int pick = m1 ? (__ffsll((long long)m1) - 1) : (nz ? 63 - __clzll((long long)nz) : -1);
      if (pick < 0) { res = -1; break; }
      double sp = readlane_d(s, pick > 0 ? pick - 1 : 0);   // uniform lane: a scalar read
      if (pick > 0) carry = carry + sp;
      g = 64 * g + (uint64_t)pick;
      res = (long long)g;
    }
    if (res >= 0) {
      const uint64_t i = (uint64_t)res;
      const uint64_t g1 = i >> 6;
      const double wv = readlane_d(cl[0], (int)(i & 63));
      if (C.R.tj_on) {
        const double o1 = C.D.top >= 1 ? readlane_d(cl[1], (int)(g1 & 63)) : 0.0;
        if (lane == 0) {
          C.S.tj_old[C.R.tj_n][0] = wv; C.S.tj_old[C.R.tj_n][1] = o1;
          C.S.tj_ind[C.R.tj_n] = i | ((uint64_t)tr << 63);
        }
      }
      // tree_set(zero) on the groups already read
      double c0 = cl[0];
      if (lane == (int)(i & 63)) c0 = 0.0;
      double gs = group_total(c0);
      if (lane == 0) g0[C.D.lev_off[0] + i] = 0.0;
      if (C.D.top >= 1) {
        if (lane == 0) g0[C.D.lev_off[1] + g1] = gs;
        double c1 = cl[1];
        if (lane == (int)(g1 & 63)) c1 = gs;
        gs = group_total(c1);
        uint64_t gi = g1 >> 6;
        for (int h = 2; h <= C.D.top; ++h) {
          double* lv = C.S.tlev[tr] + (C.D.lev_off[h] - C.D.lev_off[2]);
          if (lane == 0) lv[gi] = gs;
          double c = 0.0;
#pragma unroll
          for (int q = 2; q < BMG_TREE_LEV; ++q) if (q == h) c = cl[q];
          if (lane == (int)(gi & 63)) c = gs;
          gs = group_total(c);
          gi = gi >> 6;
        }
      }
      if (lane == 0) { C.S.bcd[1] = gs; C.S.bcd[2] = wv; }
    }
    if (lane == 0) C.S.bci[1] = res;
  }
  __syncthreads();
  long long r = C.S.bci[1];
  const double total = C.S.bcd[1], wv = C.S.bcd[2];
  __syncthreads();
  if (r < 0) { C.R.err |= ERR_TREE; *w_out = 1.0; return 0; }
  if (tr == 0) C.R.tot_add = total; else C.R.tot_rem = total;
  if (C.R.tj_on) C.R.tj_n++;
  *w_out = wv;
  return (uint64_t)r;
}

// start journalling the sum-tree writes of a move (all threads)
template <int KMAX>
__device__ __forceinline__ void journal_begin(Ctx<KMAX>& C) {
  const int nl = C.D.top >= 2 ? (int)(C.D.lev_off[C.D.top] + C.D.lev_len[C.D.top] - C.D.lev_off[2]) : 0;
  for (int e = threadIdx.x; e < nl; e += BMG_BLOCK) {
    C.S.tj_tlev[0][e] = C.S.tlev[0][e];
    C.S.tj_tlev[1][e] = C.S.tlev[1][e];
  }
  __syncthreads();
  C.R.tj_on = 1; C.R.tj_n = 0;
  C.R.tj_tot[0] = C.R.tot_add; C.R.tj_tot[1] = C.R.tot_rem;
}

// put the trees back as they were when the journal began (all threads):
// the LDS levels from their copy, the global entries from the journal in
// reverse order, the totals
template <int KMAX>
__device__ __forceinline__ void journal_restore(Ctx<KMAX>& C) {
  const int nl = C.D.top >= 2 ? (int)(C.D.lev_off[C.D.top] + C.D.lev_len[C.D.top] - C.D.lev_off[2]) : 0;
  for (int e = threadIdx.x; e < nl; e += BMG_BLOCK) {
    C.S.tlev[0][e] = C.S.tj_tlev[0][e];
    C.S.tlev[1][e] = C.S.tj_tlev[1][e];
  }
  if (threadIdx.x == 0) {
    for (int k = C.R.tj_n - 1; k >= 0; --k) {
      const uint64_t v = C.S.tj_ind[k];
      const uint64_t i = v & ~(1ull << 63);
      double* g0 = (v >> 63) ? gp(C.A.tree_rem) : gp(C.A.tree_add);
      g0[C.D.lev_off[0] + i] = C.S.tj_old[k][0];
      if (C.D.top >= 1) g0[C.D.lev_off[1] + (i >> 6)] = C.S.tj_old[k][1];
    }
  }
  __syncthreads();
  C.R.tot_add = C.R.tj_tot[0]; C.R.tot_rem = C.R.tj_tot[1];
  C.R.tj_on = 0; C.R.tj_n = 0;
}

// -------------------------------------------------------------- model -----
// Column bookkeeping helpers operate on LDS arrays with all threads.
template <int KMAX>
__device__ __forceinline__ int alloc_slot(Ctx<KMAX>& C) {
  // lowest slot free in both the current and proposed models
  int s = -1;
  for (int q = 0; q < BMG_KMAXG / 64 && s < 0; ++q) {
    uint64_t used = C.S.slots_cur[q] | C.S.slots_prop[q];
    if (~used) s = 64 * q + __ffsll((long long)~used) - 1;
  }
  return s;
}

template <int KMAX>
__device__ __forceinline__ void set_slot_bit(Ctx<KMAX>& C, int s, int on) {
  __syncthreads();
  if (threadIdx.x == 0) {
    if (on) C.S.slots_prop[s >> 6] |= (1ull << (s & 63));
    else C.S.slots_prop[s >> 6] &= ~(1ull << (s & 63));
  }
  __syncthreads();
}

// The residual term S = nu s2 + y'y - v'v of the log-likelihood, formed the
// reference's way, cancels when the factor is nearly singular (strongly
// correlated columns: v'v comes close to y'y and rounding can leave S at
// zero or below).  Where it has lost its significant digits (below 1e-8 of
// nu s2 + y'y; a fit that close never occurs otherwise) it is formed
// directly instead, as nu s2 + |y - X mu|^2 + mu'D mu with mu = U^-1 v,
// a sum of non-negative terms equal to it in exact arithmetic.
#define BMG_S_TINY 1e-8
template <int KMAX>
__device__ __forceinline__ void xcoef(Ctx<KMAX>& C, const double* coef, int L, double* out8, int write_yhat);

// out of line (it hardly ever runs), with the model's sizes by value: the
// caller's state must not have its address taken, which would keep it in
// scratch memory instead of registers
template <int KMAX>
__device__ __noinline__ double direct_syx(Smem<KMAX>& S, int k, int nloci) {
  Reg R;
  R.cols = k; R.nloci = nloci;
  Ctx<KMAX> C{S, R, S.D, S.K, S.A, S.prof};
  __syncthreads();
  for (int i = threadIdx.x; i < k; i += BMG_BLOCK) S.work[i] = S.v[i];
  __syncthreads();
  if (wave_id() == 0) trsv_un_w0(S, S.work, k);
  __syncthreads();
  double o[8];
  xcoef(C, S.work, k, o, 0);
  double md = 0.0;
  for (int i = threadIdx.x; i < k; i += BMG_BLOCK) md += S.d[i] * S.work[i] * S.work[i];
  md = block_sum(md, S.red);
  return S.K.nus2 + o[7] + md;
}

template <int KMAX>
__device__ __forceinline__ void guard_syx(Ctx<KMAX>& C) {
  if (!(C.R.syx >= BMG_S_TINY * C.K.nus2_plus_yy)) C.R.syx = direct_syx(C.S, C.R.cols, C.R.nloci);
}

// src/model.hpp:432-506 for one column (type A, H, D or R)
template <int KMAX>
__device__ __forceinline__ void update_on_add(Ctx<KMAX>& C, uint32_t ind, int model_ind, int coding,
                              int is_x_ind2, double dval, long long next = -1) {
  Smem<KMAX>& S = C.S;
  Reg& R = C.R;
  int col = R.cols;
  int slot = alloc_slot(C);
  // dots formed ahead by the previous addition of this move (same column,
  // same slot, every column since unchanged)
  const bool pre = R.pre_snp == column_key((long long)ind, coding) && R.pre_slot == slot;
  R.pre_snp = -1;
  if (slot < 0 || col >= KMAX) {
    // current and proposed models together need more slots than compiled:
    // the proposal is rejected (log-likelihood -inf) and flagged
    R.err |= ERR_CAPACITY;
    R.ll = -INFINITY; R.syx = INFINITY;
    return;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    if (is_x_ind2) S.xi2[model_ind] = col;
    else { S.xi1[model_ind] = col; S.xi2[model_ind] = 0; }
    S.snp[col] = (int32_t)ind;
    S.xtype[col] = (int8_t)coding;
    S.slot[col] = slot;
    S.d[col] = dval;
  }
  __syncthreads();
  set_slot_bit(C, slot, 1);
  R.cols = col + 1;
  if (R.lmin > col) R.lmin = col;
  const uint64_t ta = wall_clock64();
  double xy = snp_dot_y(C, ind, coding);
  const uint64_t tb = wall_clock64();
  // the slot keeps the column's value words (coded genotype in each 2-bit
  // field), which the dot products and X beta read without the coding;
  // the dot products write them as they decode the column
  if (pre) {
    for (int c = threadIdx.x; c <= col; c += BMG_BLOCK) S.work[c] = (double)S.iacc2[c];
    __syncthreads();
  } else {
    new_column_dots(C, ind, coding, col, gp(C.A.xcol) + (size_t)slot * C.D.W32);
  }
  const uint64_t tc = wall_clock64();
  // record the new X^T X row/column in the slot matrix
  for (int c = threadIdx.x; c <= col; c += BMG_BLOCK) {
    int sc = c == col ? slot : S.slot[c];
    gp(C.A.xxs)[(size_t)slot * BMG_KMAXG + sc] = S.work[c];
    gp(C.A.xxs)[(size_t)sc * BMG_KMAXG + slot] = S.work[c];
  }
  if (threadIdx.x == 0) S.xy[col] = xy;
  // the next column that the move adds (next: its column_key): its dots with
  // every column up to this one are formed by waves 1-3 while wave 0 runs this
  // column's sweep (one effect type, no covariates); its slot is the one it
  // will be given, the lowest free once this column's is taken
  int nslot = -1;
  if (next >= 0 && !C.D.mixed && C.D.me <= 1 && col + 1 < KMAX) nslot = alloc_slot(C);
  // bordered update (src/symmmatrix.cpp:144-164)
  for (int i = threadIdx.x; i < col; i += BMG_BLOCK) S.L[P(col) + i] = S.work[i];
  __syncthreads();
  if (wave_id() == 0) {
    trsv_ut_w0(S, S.L + P(col), col);
    if (nslot >= 0) job_wave(C);
  } else if (nslot >= 0) {
    column_dots<KMAX, 64, BMG_BLOCK - 64>(C, (uint64_t)next >> 2, (int)(next & 3), col + 1,
                                          gp(C.A.xcol) + (size_t)nslot * C.D.W32, S.iacc2);
  } else if (wave_id() == 3) {
    job_wave(C);
  }
  __syncthreads();
  job_done(C);
  if (nslot >= 0) { R.pre_snp = next; R.pre_slot = nslot; }
  const uint64_t td = wall_clock64();
  double ll2 = 0.0, lv = 0.0;
  for (int i = threadIdx.x; i < col; i += BMG_BLOCK) {
    double li = S.L[P(col) + i];
    ll2 += li * li;
    lv += li * S.v[i];
  }
  ll2 = block_sum(ll2, S.red);
  lv = block_sum(lv, S.red);
  double lmm2 = S.work[col] + dval - ll2;
  if (lmm2 <= 0) {
    R.ll = -INFINITY; R.syx = INFINITY;
    R.mu_computed = 0;
    __syncthreads();
    return;
  }
  double lcc = sqrt(lmm2);
  double vc = (xy - lv) / lcc;
  __syncthreads();
  if (threadIdx.x == 0) { S.L[P(col) + col] = lcc; S.v[col] = vc; }
  __syncthreads();
  R.syx = R.syx - vc * vc;
  guard_syx(C);
  R.ldq += 0.5 * log(dval);
  R.ldl += log(lcc);
  R.ll = finite_ll(R.ldq - R.ldl + C.K.minus_n_plus_nu_2 * log(R.syx));
  if (threadIdx.x == 0) {
    const uint64_t te = wall_clock64();
    C.prof[8] += tb - ta; C.prof[9] += tc - tb; C.prof[10] += td - tc; C.prof[11] += te - td;
    C.prof[12] += 1;
  }
}

// src/model.hpp:239-268; next: the SNP that the move adds after this one (-1:
// none).  An AH term's second column follows its first in the same way.
// (Before, both columns' dots came ahead of their sweeps: 5.6 + 5.0 us a
// column at 116 columns and n = 5,000, now 7.7 together; 500 iterations of 8
// such chains 120.5 -> 109.6 ms.)
template <int KMAX>
__device__ __forceinline__ void add_term(Ctx<KMAX>& C, uint32_t ind, int t_ind, const double* d2,
                                         long long next = -1) {
  Smem<KMAX>& S = C.S;
  Reg& R = C.R;
  int type = C.D.types[t_ind];
  int is_ah = type == 4;
  if (R.cols + 1 + is_ah > KMAX) {
    R.err |= ERR_CAPACITY;
    R.ll = -INFINITY; R.syx = INFINITY;
    return;
  }
  int model_ind = R.nloci;
  __syncthreads();
  if (threadIdx.x == 0) { S.loci[model_ind] = ind; S.tind[model_ind] = (int8_t)t_ind; }
  __syncthreads();
  R.nloci++;
  put(R.Ns, type, sel(R.Ns, type) + 1);
  R.mu_computed = 0;
  // A then H columns of an AH term (one copy of the update's code)
#pragma unroll 1
  for (int q = 0; q <= is_ah; ++q) {
    const double dq = q ? d2[1] : d2[0];
    if (q == 0 || isfinite(R.syx)) {
      update_on_add(C, ind, model_ind, is_ah ? q : type, q, dq,
                    q < is_ah ? column_key((long long)ind, 1) : column_key(next, is_ah ? 0 : type));
    } else if (R.cols < KMAX && alloc_slot(C) >= 0) {
      // keep the bookkeeping of the second column (not factorised)
      int col = R.cols, slot = alloc_slot(C);
      __syncthreads();
      if (threadIdx.x == 0) {
        S.xi2[model_ind] = col; S.snp[col] = (int32_t)ind; S.xtype[col] = 1;
        S.slot[col] = slot; S.d[col] = dq;
      }
      __syncthreads();
      set_slot_bit(C, slot, 1);
      R.cols = col + 1;
    }
  }
}

// src/model.hpp:508-556
template <int KMAX>
__device__ __forceinline__ void update_on_remove_impl(Ctx<KMAX>& C, int x_ind, long long next);

template <int KMAX>
__device__ __forceinline__ void update_on_remove(Ctx<KMAX>& C, int x_ind, long long next = -1) {
  const uint64_t t0 = wall_clock64();
  update_on_remove_impl(C, x_ind, next);
  if (threadIdx.x == 0) { C.prof[13] += 1; C.prof[14] += wall_clock64() - t0; }
}

template <int KMAX>
__device__ __forceinline__ void update_on_remove_impl(Ctx<KMAX>& C, int x_ind, long long next) {
  Smem<KMAX>& S = C.S;
  Reg& R = C.R;
  int k = R.cols;
  double inv_val = S.d[x_ind];
  int slot_rm = S.slot[x_ind];
  // shift column arrays left (two-phase)
  double a0 = 0, a1 = 0; int i0 = 0, i1 = 0; int8_t t0 = 0;
  int t = threadIdx.x;
  bool mv = t >= x_ind && t < k - 1;
  if (mv) { a0 = S.xy[t + 1]; a1 = S.d[t + 1]; i0 = S.slot[t + 1]; i1 = S.snp[t + 1]; t0 = S.xtype[t + 1]; }
  __syncthreads();
  if (mv) { S.xy[t] = a0; S.d[t] = a1; S.slot[t] = i0; S.snp[t] = i1; S.xtype[t] = t0; }
  __syncthreads();
  set_slot_bit(C, slot_rm, 0);
  R.cols = k - 1;
  if (R.lmin > x_ind) R.lmin = x_ind;
  if (x_ind == R.cols) {
    double lxx = S.L[P(x_ind) + x_ind];
    double vx = S.v[x_ind];
    R.ldl -= log(lxx);
    R.syx += vx * vx;
  } else {
    // the move's first addition after this removal (next >= 0): its column
    // dots with the remaining columns are formed by waves 1-3 during the
    // downdate, into the slot it will be given (as during a forward sweep)
    int nslot = -1;
    if (next >= 0 && !C.D.mixed && C.D.me <= 1 && R.cols < KMAX)
      nslot = alloc_slot(C);
    auto ahead = [&]() {
      column_dots<KMAX, 64, BMG_BLOCK - 64>(C, (uint64_t)next >> 2, (int)(next & 3), R.cols,
                                            gp(C.A.xcol) + (size_t)nslot * C.D.W32, S.iacc2);
    };
    const uint64_t ta = wall_clock64();
    // v follows the downdate's rotations (no re-solve)
    chol_downdate(S, k, x_ind, nslot >= 0, ahead, [&]() { job_wave(C); });
    job_done(C);
    if (nslot >= 0) { R.pre_snp = next; R.pre_slot = nslot; }
    const uint64_t tb = wall_clock64();
    if (threadIdx.x == 0) { C.prof[16] += tb - ta; C.prof[17] += wall_clock64() - tb; }
    double ld = 0.0, vv = 0.0;
    for (int i = threadIdx.x; i < R.cols; i += BMG_BLOCK) {
      ld += log(S.L[P(i) + i]);
      vv += S.v[i] * S.v[i];
    }
    R.ldl = block_sum(ld, S.red);
    vv = block_sum(vv, S.red);
    R.syx = C.K.nus2_plus_yy - vv;
    guard_syx(C);
  }
  R.ldq -= 0.5 * log(inv_val);
  R.ll = finite_ll(R.ldq - R.ldl + C.K.minus_n_plus_nu_2 * log(R.syx));
}

// src/model.hpp:270-312
template <int KMAX>
__device__ __forceinline__ void remove_term(Ctx<KMAX>& C, int model_ind, long long next = -1) {
  Smem<KMAX>& S = C.S;
  Reg& R = C.R;
  int type = C.D.types[S.tind[model_ind]];
  int xi1 = S.xi1[model_ind], xi2 = S.xi2[model_ind];
  uint32_t ind = S.loci[model_ind];
  put(R.Ns, type, sel(R.Ns, type) - 1);
  int nl = R.nloci;
  int xmove = type == 4 ? 2 : 1;
  int t = threadIdx.x;
  bool mv = t >= model_ind && t < nl - 1;
  uint32_t l0 = 0; int8_t ti = 0; int a1 = 0, a2 = 0;
  if (mv) { l0 = S.loci[t + 1]; ti = S.tind[t + 1]; a1 = S.xi1[t + 1] - xmove; a2 = S.xi2[t + 1] - xmove; }
  __syncthreads();
  if (mv) { S.loci[t] = l0; S.tind[t] = ti; S.xi1[t] = a1; S.xi2[t] = a2; }
  if (threadIdx.x == 0) S.rm_list[R.n_rm] = ind;
  __syncthreads();
  R.n_rm++;
  R.nloci = nl - 1;
  // the later column of an AH term first
#pragma unroll 1
  for (int q = 0; q < xmove; ++q)
    update_on_remove(C, type != 4 ? xi1 : ((q == 0) == (xi1 > xi2) ? xi1 : xi2),
                     q + 1 < xmove ? -1 : column_key(next, type == 4 ? 0 : type));
  R.mu_computed = 0;
}

// index of SNP `ind` in the proposed model, or -1 (all threads)
template <int KMAX>
__device__ __forceinline__ int find_locus(Ctx<KMAX>& C, uint64_t ind) {
  __syncthreads();
  if (threadIdx.x == 0) C.S.bci[2] = -1;
  __syncthreads();
  for (int t = threadIdx.x; t < C.R.nloci; t += BMG_BLOCK)
    if (C.S.loci[t] == (uint32_t)ind) C.S.bci[2] = t;
  __syncthreads();
  int r = (int)C.S.bci[2];
  __syncthreads();
  return r;
}

// src/model.hpp:199-237 on the proposed model
template <int KMAX>
__device__ __forceinline__ void compute_log_likelihood(Ctx<KMAX>& C) {
  Smem<KMAX>& S = C.S;
  Reg& R = C.R;
  int k = R.cols;
  if (k < 1) { R.ll = NAN; return; }
  // X'X + D from the slot matrix into the packed factor: a thread per
  // column j, its rows i <= j read eight at a time (row slot(j) of the slot
  // matrix holds column j's entries), so the loads are in flight together
  if ((int)threadIdx.x < k) {
    const int j = (int)threadIdx.x;
    const double* __restrict__ row = gp(C.A.xxs) + (size_t)S.slot[j] * BMG_KMAXG;
    double* col = S.L + P(j);
    for (int i0 = 0; i0 <= j; i0 += 8) {
      double v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = row[S.slot[i0 + u <= j ? i0 + u : j]];   // past j: a valid slot
      const double dj = S.d[j];
      // unconditional stores: a row past j is clamped to j and rewrites the
      // diagonal with the value row j gives it
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int i = i0 + u <= j ? i0 + u : j;
        col[i] = i == j ? v[u] + dj : v[u];
      }
    }
  }
  double ls = 0.0;
  for (int i = 1 + threadIdx.x; i < k; i += BMG_BLOCK) ls += log(S.d[i]);
  ls = block_sum(ls, S.red);
  R.ldq = 0.5 * ls;
  R.lmin = 0;
  if (!chol_full(S, k)) {
    R.ll = -INFINITY; R.syx = INFINITY; R.mu_computed = 0;
    return;
  }
  for (int i = threadIdx.x; i < k; i += BMG_BLOCK) S.v[i] = S.xy[i];
  __syncthreads();
  if (wave_id() == 0) trsv_ut_w0(S, S.v, k);
  __syncthreads();
  double ld = 0.0, vv = 0.0;
  for (int i = threadIdx.x; i < k; i += BMG_BLOCK) {
    ld += log(S.L[P(i) + i]);
    vv += S.v[i] * S.v[i];
  }
  R.ldl = block_sum(ld, S.red);
  vv = block_sum(vv, S.red);
  R.syx = C.K.nus2_plus_yy - vv;
  guard_syx(C);
  R.ll = finite_ll(R.ldq - R.ldl + C.K.minus_n_plus_nu_2 * log(R.syx));
  R.mu_computed = 0;
}

// --------------------------------------------------- commit / restore -----
// Accept (*current = *new) or reject (*new = *current) for the single
// working copy: only factor columns >= lmin differ from the stored current
// factor.

// dst[e] = src[e] for e in [e0, e1) (all threads): eight elements a thread
// are read before any is written, so the reads of one pass are in flight
// together instead of one round trip per element
__device__ __forceinline__ void copy_factor(double* __restrict__ dst, const double* __restrict__ src, int e0,
                                            int e1) {
  for (int base = e0; base < e1; base += BMG_BLOCK * 8) {
    double t[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int e = base + q * BMG_BLOCK + (int)threadIdx.x;
      t[q] = e < e1 ? src[e] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int e = base + q * BMG_BLOCK + (int)threadIdx.x;
      if (e < e1) dst[e] = t[q];
    }
  }
}

template <int KMAX>
__device__ __forceinline__ void commit(Ctx<KMAX>& C) {
  Smem<KMAX>& S = C.S;
  Reg& R = C.R;
  __syncthreads();
  copy_factor(gp(C.A.Lcur), S.L, P(R.lmin < R.cols ? R.lmin : R.cols), P(R.cols));
  for (int i = threadIdx.x; i < R.cols; i += BMG_BLOCK) {
    S.c_xy[i] = S.xy[i]; S.c_v[i] = S.v[i]; S.c_d[i] = S.d[i];
    S.c_slot[i] = S.slot[i]; S.c_snp[i] = S.snp[i]; S.c_xtype[i] = S.xtype[i];
  }
  for (int i = threadIdx.x; i < R.nloci; i += BMG_BLOCK) {
    S.c_loci[i] = S.loci[i]; S.c_xi1[i] = S.xi1[i]; S.c_xi2[i] = S.xi2[i]; S.c_tind[i] = S.tind[i];
  }
  // current model_inds: removed loci first, then the positions of all loci
  for (int i = threadIdx.x; i < R.n_rm; i += BMG_BLOCK) gp(C.A.model_inds)[S.rm_list[i]] = -1;
  __syncthreads();
  for (int i = threadIdx.x; i < R.nloci; i += BMG_BLOCK) gp(C.A.model_inds)[S.loci[i]] = i;
  if (threadIdx.x < BMG_KMAXG / 64) S.slots_cur[threadIdx.x] = S.slots_prop[threadIdx.x];
  __syncthreads();
  R.c_cols = R.cols; R.c_nloci = R.nloci;
  for (int q = 0; q < 5; ++q) R.c_Ns[q] = R.Ns[q];
  R.c_syx = R.syx; R.c_ldq = R.ldq; R.c_ldl = R.ldl; R.c_ll = R.ll;
  R.lmin = KMAX; R.n_rm = 0;
  R.mu_computed = 0;
}

template <int KMAX>
__device__ __forceinline__ void restore(Ctx<KMAX>& C) {
  Smem<KMAX>& S = C.S;
  Reg& R = C.R;
  __syncthreads();
  int lm = R.lmin < R.c_cols ? R.lmin : R.c_cols;
  copy_factor(S.L, gp(C.A.Lcur), P(lm), P(R.c_cols));
  for (int i = threadIdx.x; i < R.c_cols; i += BMG_BLOCK) {
    S.xy[i] = S.c_xy[i]; S.v[i] = S.c_v[i]; S.d[i] = S.c_d[i];
    S.slot[i] = S.c_slot[i]; S.snp[i] = S.c_snp[i]; S.xtype[i] = S.c_xtype[i];
  }
  for (int i = threadIdx.x; i < R.c_nloci; i += BMG_BLOCK) {
    S.loci[i] = S.c_loci[i]; S.xi1[i] = S.c_xi1[i]; S.xi2[i] = S.c_xi2[i]; S.tind[i] = S.c_tind[i];
  }
  if (threadIdx.x < BMG_KMAXG / 64) S.slots_prop[threadIdx.x] = S.slots_cur[threadIdx.x];
  __syncthreads();
  R.cols = R.c_cols; R.nloci = R.c_nloci;
  for (int q = 0; q < 5; ++q) R.Ns[q] = R.c_Ns[q];
  R.syx = R.c_syx; R.ldq = R.c_ldq; R.ldl = R.c_ldl; R.ll = R.c_ll;
  R.lmin = KMAX; R.n_rm = 0;
}

// --------------------------------------------------------------- prior ----
// src/prior.hpp:144-158 (single effect type, Ns[type] == n_loci)
__device__ __forceinline__ double prior_add_untruncated(const ChainConst& K, const int (&Ns)[5], int n_old,
                                                        int type) {
  return (log(K.g_a + n_old) - log(K.g_b + K.m_g - n_old - 1)) +
         (log(K.tp_type + sel(Ns, type)) - log(K.tp_sum + n_old));
}
// with a model-size limit the prior of larger models is 0
__device__ __forceinline__ double prior_add(const ChainConst& K, const int (&Ns)[5], int n_old, int type) {
  if (n_old >= K.max_size) return -INFINITY;
  return prior_add_untruncated(K, Ns, n_old, type);
}
__device__ __forceinline__ double prior_rem(const ChainConst& K, const int (&Ns)[5], int n_old, int type) {
  return (log(K.g_b + K.m_g - n_old) - log(K.g_a + n_old - 1)) +
         (log(K.tp_sum + n_old - 1) - log(K.tp_type + sel(Ns, type) - 1));
}

// Draws on the chain's stream, one per term in term order, a term per thread:
// a thread starts its term where the stream would be if every earlier term of
// the round took one trial (two Philox blocks); the first term after which
// that does not hold ends the round, and the next round restarts from the
// stream position it left.  The draws are the sequential loop's, value for
// value; a draw alone takes about 1.2 us.  draw(r, i): term i's value from the
// stream r; out[0 .. count) receives them (LDS).
template <int KMAX, typename Draw>
__device__ __forceinline__ void draw_terms(Ctx<KMAX>& C, int first, int count, double* out, Draw draw) {
  Smem<KMAX>& S = C.S;
  Reg& R = C.R;
  uint64_t base = (uint64_t)R.rng.c0 | ((uint64_t)R.rng.c1 << 32);
  __syncthreads();
  while (first < count) {
    const int i = first + (int)threadIdx.x;
    long long stop = count;          // first term whose stream use differs
    uint64_t next = 0;
    double v = 0.0;
    if (i < count) {
      const uint64_t start = base + 2ull * (uint64_t)threadIdx.x;
      Rng r = R.rng;
      r.c0 = (uint32_t)start; r.c1 = (uint32_t)(start >> 32);
      v = draw(r, i);
      next = (uint64_t)r.c0 | ((uint64_t)r.c1 << 32);
      if (next - start != 2) stop = i;
      if (i == first + BMG_BLOCK - 1 && stop == count) stop = i;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const long long w = __shfl_xor(stop, o, 64);
      stop = w < stop ? w : stop;
    }
    if (lane_id() == 0) S.redi[wave_id()] = stop;
    __syncthreads();
    stop = S.redi[0];
    for (int w = 1; w < BMG_BLOCK / 64; ++w) stop = S.redi[w] < stop ? S.redi[w] : stop;
    // terms first..stop are final; the stream continues after term stop
    if (i <= stop && i < count) out[i] = v;
    if (i == stop) S.bci[3] = (long long)next;
    __syncthreads();
    if (stop >= count) {
      base += 2ull * (uint64_t)(count - first);
      first = count;
    } else {
      base = (uint64_t)S.bci[3];
      first = (int)stop + 1;
    }
    __syncthreads();
  }
  R.rng.c0 = (uint32_t)base; R.rng.c1 = (uint32_t)(base >> 32);
}

// the prior precisions of the next n_add new terms, in order, in S.mu (whose
// own contents a change of the model makes void); new_term picks the k-th's
template <int KMAX>
__device__ __forceinline__ void draw_new_terms(Ctx<KMAX>& C, int n_add) {
  if (!C.K.use_ind || n_add == 0) return;
  const int w = C.D.type == 4 ? 2 : 1;
  const double a2 = C.R.alpha2;
  draw_terms(C, 0, w * n_add, C.S.mu, [&](Rng& r, int i) {
    const int t = w == 2 ? i & 1 : C.D.type;
    return 1.0 / (a2 * rng_sinvchi2(r, C.K.nu_tau2[t], C.K.s2_tau2[t]));
  });
}
template <int KMAX>
__device__ __forceinline__ void new_term(Ctx<KMAX>& C, int k, double* d2) {
  const int type = C.D.type, w = type == 4 ? 2 : 1;
  for (int q = 0; q < w; ++q)
    d2[q] = C.K.use_ind ? C.S.mu[w * k + q] : sel(C.R.ita2, w == 2 ? q : type);
}

// ------------------------------------------------- beta / sigma2 / pve ----
template <int KMAX>
__device__ __forceinline__ void compute_mu_beta(Ctx<KMAX>& C) {
  if (!C.R.mu_computed) {
    __syncthreads();
    for (int i = threadIdx.x; i < C.R.cols; i += BMG_BLOCK) C.S.mu[i] = C.S.v[i];
    __syncthreads();
    if (wave_id() == 0) trsv_un_w0(C.S, C.S.mu, C.R.cols);
    __syncthreads();
    C.R.mu_computed = 1;
  }
}

// counter-based access to draw `k` of the main stream from its current
// position (the stream itself is sequential: draw k uses counter base + k)
__device__ __forceinline__ double normal_at(const Rng& r, uint32_t k) {
  Rng q = r;
  uint64_t c = ((uint64_t)q.c1 << 32 | q.c0) + k;
  q.c0 = (uint32_t)c; q.c1 = (uint32_t)(c >> 32);
  return rng_normal(q);
}
__device__ __forceinline__ void rng_skip(Rng& r, uint32_t k) {
  uint64_t c = ((uint64_t)r.c1 << 32 | r.c0) + k;
  r.c0 = (uint32_t)c; r.c1 = (uint32_t)(c >> 32);
}

// src/model.hpp:326-342 with src/rand.hpp:61-78,144-168
template <int KMAX>
__device__ __forceinline__ void sample_beta_sigma2(Ctx<KMAX>& C) {
  Reg& R = C.R;
  double nu = C.K.n_plus_nu;
  double s2 = R.syx / C.K.n_plus_nu;
  double val = -1.0;
  for (int trial = 0; trial < BMG_MAX_TRIALS && (val <= 0 || !isfinite(val)); ++trial)
    val = nu * s2 / (2.0 * rng_gamma(R.rng, 0.5 * nu));
  if (!(val > 0) || !isfinite(val)) R.err |= ERR_SIGMA2;
  R.sigma2 = val;
  compute_mu_beta(C);
  R.beta_len = R.cols;
  for (int i = threadIdx.x; i < R.cols; i += BMG_BLOCK) C.S.beta[i] = normal_at(R.rng, i);
  rng_skip(R.rng, R.cols);
  __syncthreads();
  if (wave_id() == 0) trsv_un_w0(C.S, C.S.beta, R.beta_len);
  __syncthreads();
  double sc = sqrt(R.sigma2);
  for (int i = threadIdx.x; i < R.beta_len; i += BMG_BLOCK)
    C.S.beta[i] = sc * C.S.beta[i] + C.S.mu[i];
  __syncthreads();
}

template <int KMAX>
__device__ __forceinline__ void xbeta_impl(Ctx<KMAX>& C, const double* coef, int L, double* out8,
                                           int write_yhat) {
  Smem<KMAX>& S = C.S;
  Reg& R = C.R;
  const double b0 = coef[0];
  const int me = C.D.me;
  const uint32_t n = C.D.n, W = C.D.W32;
  const uint32_t* __restrict__ xcol = gp(C.A.xcol);
  const double* __restrict__ y = gp(C.D.y);
  double* __restrict__ yhat = gp(C.A.y_hat);
  double sxb = 0, sxb2 = 0, sy = 0, sy2 = 0, syx = 0, se = 0, se2 = 0, srr = 0;
  for (uint32_t w = threadIdx.x; w * 16 < n; w += BMG_BLOCK) {
    double acc[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) acc[q] = 0.0;
    for (int c0 = me; c0 < L; c0 += 16) {
      uint32_t wd[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const int c = c0 + u;
        wd[u] = (c < L && coef[c] != 0.0) ? xcol[(size_t)S.slot[c] * W + w] : 0u;
      }
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const int c = c0 + u;
        if (c < L) {
          const double t = coef[c];
          if (t != 0.0) {
            // t * value is exact (value 0, 1 or 2), so the fused form
            // rounds the sum as the multiply-then-add loop does
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[q] = fma(t, (double)((wd[u] >> (2 * q)) & 3u), acc[q]);
          }
        }
      }
    }
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const uint32_t i = w * 16 + q;
      if (i < n) {
        const double a = acc[q];
        sxb += a; sxb2 += a * a;
        // E beta_E of this individual in column order (the constant first)
        double e = b0;
        for (int c = 1; c < me; ++c) e = e + gp(C.D.E)[(size_t)(c - 1) * C.D.n_pad + i] * coef[c];
        se += e; se2 += e * e;
        // with covariates and no loci the reference adds E beta_E to the
        // y_hat it holds (src/model.hpp:369-373 leaves the genetic part
        // unset), and so does this
        const double yh = R.nloci > 0 ? a + e : (me > 1 && write_yhat ? yhat[i] + e : e);
        sy += yh; sy2 += yh * yh;
        syx += (e - y[i]) * a;
        const double ri = y[i] - (R.nloci > 0 ? a + e : e);
        srr += ri * ri;
        if (write_yhat) yhat[i] = yh;
      }
    }
  }
  out8[0] = block_sum(sxb, S.red);
  out8[1] = block_sum(sxb2, S.red);
  out8[2] = block_sum(sy, S.red);
  out8[3] = block_sum(sy2, S.red);
  out8[4] = block_sum(syx, S.red);
  out8[5] = block_sum(se, S.red);
  out8[6] = block_sum(se2, S.red);
  out8[7] = block_sum(srr, S.red);
}

// y_hat = X_g beta_g + E beta_E into the chain's y_hat (write_yhat) and
// out7: sum xb, sum xb^2, sum y_hat, sum y_hat^2, sum (e - y) xb, sum e,
// sum e^2, with xb = X_g beta_g and e = E beta_E (the constant and the
// covariates).  One packed word (16 individuals) per lane: the columns'
// words are fetched sixteen at a time (coalesced across lanes, all in
// flight together) and each individual's sum is formed in model-column
// order, as the per-individual loop does.
template <int KMAX>
__device__ __forceinline__ void xcoef(Ctx<KMAX>& C, const double* coef, int L, double* out8, int write_yhat) {
  xbeta_impl<KMAX>(C, coef, L, out8, write_yhat);
}

template <int KMAX>
__device__ __forceinline__ void xbeta(Ctx<KMAX>& C, double* out8, int write_yhat) {
  xcoef(C, C.S.beta, C.R.beta_len, out8, write_yhat);
}

// A sum kept as an unevaluated pair (Dekker 1971, Knuth's two-sum), about 106
// bits: the quadratic forms below cancel where columns are correlated.
struct Pair { double hi, lo; };
__device__ __forceinline__ void pair_add(Pair& s, double x, double e) {
  const double t = s.hi + x, z = t - s.hi;
  s.lo += ((s.hi - (t - z)) + (x - z)) + e;
  s.hi = t;
}
__device__ __forceinline__ void pair_fma(Pair& s, double x, double y) {
  const double p = x * y;
  pair_add(s, p, fma(x, y, -p));
}
__device__ __forceinline__ void pair_fma(Pair& s, const Pair& x, double y) {
  const double p = x.hi * y;
  pair_add(s, p, fma(x.hi, y, -p) + x.lo * y);
}

// xcoef's sums (all but the residual's, out8[7]) from the model's X^T X and
// X^T y, O(k^2) instead of O(n k): with a = X_g b_g and e = E b_E, sum a^2 =
// b_g' (X_g^T X_g) b_g and so on, every sum a pair.  Lane j of each wave
// takes column j, the waves every fourth row, so a load reads one row of the
// slot matrix.  Bound by those reads (k^2 doubles through L2).  (Formed per
// individual, with a conversion and a fused multiply-add per genotype, the
// sums of a 139-column model at n = 10,000 took 140 us, once per thinned
// sample and once per refresh.)  The entries are whole numbers but the
// covariates'.
template <int KMAX>
__device__ __forceinline__ void xmoments(Ctx<KMAX>& C, const double* coef, int L, double* out8) {
  constexpr int NQ = (KMAX + 63) / 64;
  constexpr int BAT = 8;
  Smem<KMAX>& S = C.S;
  const int me = C.D.me;
  const int lane = lane_id(), w = wave_id();
  const double* __restrict__ xxs = gp(C.A.xxs);
  // sum a, a^2, a e, e, e^2, a y
  Pair m[6];
#pragma unroll
  for (int q = 0; q < 6; ++q) m[q] = Pair{0.0, 0.0};
#pragma unroll 1
  for (int q = 0; q < NQ; ++q) {
    if (64 * q >= L) break;
    const int j = 64 * q + lane;
    const bool on = j < L;
    const int sj = on ? S.slot[j] : S.slot[0];
    const double bj = on ? coef[j] : 0.0;
    Pair ug{0.0, 0.0}, ue{0.0, 0.0};
    double g0 = 0.0;
#pragma unroll 1
    for (int i0 = w; i0 < L; i0 += 4 * BAT) {
      double g[BAT];
#pragma unroll
      for (int u = 0; u < BAT; ++u) {
        const int i = i0 + 4 * u;
        g[u] = xxs[(size_t)S.slot[i < L ? i : 0] * BMG_KMAXG + sj];
      }
#pragma unroll
      for (int u = 0; u < BAT; ++u) {
        const int i = i0 + 4 * u;
        if (i < me) {
          pair_fma(ue, g[u], coef[i]);
          if (i == 0) g0 = g[u];
        } else if (i < L) {
          pair_fma(ug, g[u], coef[i]);
        }
      }
    }
    if (j >= me) {
      pair_fma(m[0], g0, bj);
      pair_fma(m[1], ug, bj);
      pair_fma(m[2], ue, bj);
      if (w == 0 && on) pair_fma(m[5], S.xy[j], bj);
    } else {
      pair_fma(m[3], g0, bj);
      pair_fma(m[4], ue, bj);
    }
  }
  // the lanes' pairs, then the waves', in a fixed order
#pragma unroll
  for (int o = 1; o < 64; o <<= 1)
#pragma unroll
    for (int q = 0; q < 6; ++q) {
      const double h = __shfl_xor(m[q].hi, o, 64), l = __shfl_xor(m[q].lo, o, 64);
      pair_add(m[q], h, l);
    }
  __syncthreads();
  if (lane == 0)
#pragma unroll
    for (int q = 0; q < 6; ++q) { S.work[12 * w + 2 * q] = m[q].hi; S.work[12 * w + 2 * q + 1] = m[q].lo; }
  __syncthreads();
  double v[6];
#pragma unroll
  for (int q = 0; q < 6; ++q) {
    Pair t{S.work[2 * q], S.work[2 * q + 1]};
    for (int ww = 1; ww < BMG_BLOCK / 64; ++ww) pair_add(t, S.work[12 * ww + 2 * q], S.work[12 * ww + 2 * q + 1]);
    v[q] = t.hi + t.lo;
  }
  __syncthreads();
  out8[0] = v[0]; out8[1] = v[1];
  out8[2] = v[0] + v[3]; out8[3] = v[1] + 2.0 * v[2] + v[4];
  out8[4] = v[2] - v[5];
  out8[5] = v[3]; out8[6] = v[4]; out8[7] = 0.0;
}

// src/model.hpp:345-392: shares of var(E beta_E) (covariates beyond the
// constant), var(X_g beta_g) and var(y_hat) in var(y_hat) + sigma2
// (need_y: leave y_hat too; the sums then come with it, and belong to it also
// where a caller has changed its model since it drew beta.  Nothing reads the
// y_hat of a sample that no RB scan follows, and without covariates each is
// formed anew; with them a model without loci adds to the one it holds, so
// every sample's is formed.)
template <int KMAX>
__device__ __forceinline__ void compute_pve(Ctx<KMAX>& C, double* pves, int need_y) {
  double s[8];
  if (need_y || C.D.me > 1) xbeta(C, s, 1);
  else xmoments(C, C.S.beta, C.R.beta_len, s);
  const double n = (double)C.D.n;
  const bool ce = C.D.me > 1, cg = C.R.nloci > 0;
  pves[2] = ce ? (s[6] - s[5] * s[5] / n) / (n - 1) : 0.0;
  pves[1] = cg ? (s[1] - s[0] * s[0] / n) / (n - 1) : 0.0;
  if (!ce && !cg) { pves[0] = pves[1] = pves[2] = 0.0; return; }
  pves[0] = !ce ? pves[1] : (!cg ? pves[2] : (s[3] - s[2] * s[2] / n) / (n - 1));
  const double z = pves[0] + C.R.sigma2;
  pves[0] /= z; pves[1] /= z; pves[2] /= z;
}

// src/prior.cpp:30-141 on the working model
template <int KMAX>
__device__ __forceinline__ void sample_alpha_and_tau2(Ctx<KMAX>& C) {
  Smem<KMAX>& S = C.S;
  Reg& R = C.R;
  const ChainConst& K = C.K;
  // sample_tau2
  double a2s2 = R.alpha2 * R.sigma2;
  if (K.use_ind) {
    // (the covariates' precisions are fixed)
    const double a2 = R.alpha2;
    draw_terms(C, C.D.me, R.beta_len, S.d, [&](Rng& r, int i) {
      const int t = S.xtype[i];
      const double nu = K.nu_tau2[t] + 1.0;
      const double s2 = (K.nus2_tau2[t] + S.beta[i] * S.beta[i] / a2s2) / nu;
      return 1.0 / (a2 * rng_sinvchi2(r, nu, s2));
    });
  } else {
    double b2[4] = {0, 0, 0, 0}; double mt[4] = {0, 0, 0, 0};
    for (int i = C.D.me; i < R.beta_len; ++i) {
      const int xt = S.xtype[i];
      put(b2, xt, sel(b2, xt) + S.beta[i] * S.beta[i]);
      put(mt, xt, sel(mt, xt) + 1.0);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if (!K.allow_terms[t]) continue;
      double nu = K.nu_tau2[t] + mt[t];
      double s2 = (K.nus2_tau2[t] + b2[t] / a2s2) / nu;
      R.ita2[t] = 1.0 / (R.alpha2 * rng_sinvchi2(R.rng, nu, s2));
    }
    __syncthreads();
    for (int i = C.D.me + threadIdx.x; i < R.beta_len; i += BMG_BLOCK) S.d[i] = sel(R.ita2, (int)S.xtype[i]);
  }
  R.mu_computed = 0;
  __syncthreads();
  // sample_alpha
  int nterms = R.beta_len - C.D.me;
  double a = R.alpha;
  double xbxb = 0, ebxb = 0;
  if (nterms > 0) {
    // x_b = X_g beta_g, e_b = E beta_E - y
    double s[8];
    xmoments(C, S.beta, R.beta_len, s);
    ebxb = s[4];
    xbxb = s[1];
  }
  int trials = 0;
  do {
    if (++trials > BMG_MAX_TRIALS) { R.err |= ERR_ALPHA; a = R.alpha; break; }
    if (nterms > 0) {
      if ((a <= 0.0) || log(rng_u01(R.rng)) <= -2.0 * K.mu_alpha * a) a = -a;
      double as2 = a * R.sigma2;
      double var = 1.0 / (1.0 + xbxb / (a * as2));
      double mu = var * (K.mu_alpha - ebxb / as2);
      a = sqrt(var) * rng_normal(R.rng) + mu;
    } else {
      a = rng_normal(R.rng) + K.mu_alpha;
    }
  } while (a == 0 || a * a == 0);
  // set_alpha
  double old = R.alpha2;
  R.alpha = a; R.alpha2 = a * a;
  __syncthreads();
  if (K.use_ind) {
    for (int i = C.D.me + threadIdx.x; i < R.beta_len; i += BMG_BLOCK) S.d[i] = S.d[i] * old / R.alpha2;
  } else {
#pragma unroll
    for (int t = 0; t < 4; ++t) if (K.allow_terms[t]) R.ita2[t] = R.ita2[t] * old / R.alpha2;
    for (int i = C.D.me + threadIdx.x; i < R.beta_len; i += BMG_BLOCK) S.d[i] = sel(R.ita2, (int)S.xtype[i]);
  }
  __syncthreads();
}

// ---------------------------------------------------------------- moves ---
// first i with u * cumsum[m - 1] < cumsum[i], m <= 64 (a lane per entry)
__device__ __forceinline__ int sample_naive(const double* cumsum, int m, double u) {
  const int lane = lane_id();
  const double r = u * cumsum[m - 1];
  const unsigned long long b = __ballot(lane < m && r < cumsum[lane < m ? lane : 0]);
  return b ? __ffsll((long long)b) - 1 : m - 1;
}

// PMV move mix with one effect type (src/sampler.cpp:468-476); with a
// learned table, a drawn swap is a learned swap with probability
// p_learned (both swaps keep the posterior; the choice does not depend
// on the state, and add/remove and state-change moves keep their share).
// 0 add/remove, 1 swap, 2 state change, 3 learned swap
template <int KMAX>
__device__ __forceinline__ int draw_move(const Ctx<KMAX>& C, ChainRng& rng) {
  const double pm[3] = {0.7, 0.7 + 0.15, 0.7 + 0.15 + 0.15};
  const double r = rng_u01(rng) * pm[2];
  int move = r < pm[0] ? 0 : (r < pm[1] ? 1 : 2);
  if (move == 1 && C.R.learn_on && rng_u01(rng) < C.K.p_learned) move = 3;
  return move;
}

// the size of an add/remove (0), swap (1) or state-change (2) move
template <int KMAX>
__device__ __forceinline__ int draw_move_size(const Ctx<KMAX>& C, ChainRng& rng, int move) {
  const ChainConst& K = C.K;
  uint64_t mx = K.max_ms;
  if (move == 1) {
    const uint64_t half = (C.D.p - C.R.c_nloci + 1) / 2;
    mx = (K.max_ms + 1) / 2;
    mx = mx < half ? mx : half;
    mx = mx < (uint64_t)C.R.c_nloci ? mx : (uint64_t)C.R.c_nloci;
  } else if (move == 2) {
    const uint64_t a = (uint64_t)K.max_nbh * 2, b = C.D.p - 1 < K.max_ms ? C.D.p - 1 : K.max_ms;
    mx = a < b ? a : b;
  }
  return sample_naive(C.S.cdf[move], (int)mx, rng_u01(rng)) + 1;
}

template <int KMAX>
__device__ __forceinline__ void undo_dd(Ctx<KMAX>& C, int ms) {
  for (int i = 0; i < ms; ++i) {
    uint64_t ind = C.S.mi[i];
    if (C.S.mi_isadd[i]) { tree_set(C, 0, ind, 0); tree_set(C, 1, ind, 1); }
    else { tree_set(C, 0, ind, 1); tree_set(C, 1, ind, 0); }
  }
}

// ------------------------------------------------ delayed rejection -----
// ExhModel (src/model.hpp:585-844) on the proposed model once every moved SNP
// is in it: loci from position `cl` on are the ones the second stage toggles,
// and their columns c0..cols-1 form the trailing block.  The walk's adjacent
// swaps only permute the rows above c0 of those columns, and its
// log-likelihoods read only the block's diagonal and v, so the block (in
// indices relative to c0) is all that is copied; the working model is left
// as it is.  Wave 0 walks the 2^ms sub-models in the reference's order: the
// scalar state is replicated in its lanes, the swaps give each lane one row
// or column.  Bound by the chain of adjacent swaps: an LDS round trip, a
// reciprocal square root and a few multiplies each.  So nothing else is in
// it: a sub-model's determinant is the running product of its diagonal and
// its residual term the running difference, both kept by column, so a step
// restarts from the columns left of the swap without taking anything back,
// and the logarithms, the prior terms and the precisions' (which depend on
// the set of loci alone) are added afterwards, a thread per sub-model.  (With
// four logarithms, two divisions and a square root in every step the walk
// took 1.2 us a sub-model, and the scoring 140-155 us of an iteration of 235 at
// n = 1,000, p = 10,000 and delay_rejection = 10; now 50.)
template <int KMAX>
__device__ __forceinline__ double& exl(Smem<KMAX>& S, int r, int c) { return S.ex_L[P(c) + r]; }

// orders wave 0's LDS accesses across its lanes
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// src/symmmatrix.cpp:220-265 on the block (columns s, s+1 relative to c0):
// lane r swaps row r < s, lane i - s - 1 rotates column i > s
template <int KMAX>
__device__ __forceinline__ void exh_swapadj(Smem<KMAX>& S, int nT, int s) {
  const int lane = lane_id();
  const int i = s + 1 + lane;
  const bool up = lane < s, on = i < nT;
  const double a = exl(S, s, s + 1), b = exl(S, s + 1, s + 1), dcc = exl(S, s, s);
  const double v1 = S.ex_v[s], v2 = S.ex_v[s + 1];
  const int r = up ? lane : 0, j = on ? i : s + 1;
  const double t0 = exl(S, r, s), t1 = exl(S, r, s + 1);
  const double y1 = exl(S, s, j), y2 = exl(S, s + 1, j);
  wave_sync();
  // the rotation of (a, b), b > 0: 1 / r from the hardware reciprocal square
  // root and two Newton steps, within an ulp or two
  const double q = fma(a, a, b * b);
  double y = __builtin_amdgcn_rsq(q);
  const double h = 0.5 * q;
  y = y * fma(-h * y, y, 1.5);
  y = y * fma(-h * y, y, 1.5);
  const double c = a * y, sn = b * y;
  if (up) { exl(S, r, s) = t1; exl(S, r, s + 1) = t0; }
  if (on) {
    // column s+1 holds (dcc, 0) in rows s, s+1 after the swap
    const double x1 = lane == 0 ? dcc : y1, x2 = lane == 0 ? 0.0 : y2;
    exl(S, s, i) = fma(x2, sn, x1 * c);
    exl(S, s + 1, i) = fma(x1, sn, -(x2 * c));
  }
  if (lane == 0) {
    exl(S, s, s) = q * y;
    S.ex_v[s] = fma(v2, sn, v1 * c);
    S.ex_v[s + 1] = fma(v1, sn, -(v2 * c));
  }
  wave_sync();
}

// columns [vs, vs + w) join the walk's model (src/model.hpp:673-701)
template <int KMAX>
__device__ __forceinline__ void exh_add(Smem<KMAX>& S, int w, int& vs) {
  double pp = S.ex_pp[vs], ss = S.ex_ss[vs];
  for (int q = 0; q < w; ++q) {
    const double l = exl(S, vs, vs), v = S.ex_v[vs];
    pp = pp * l;
    ss = fma(-v, v, ss);
    ++vs;
    S.ex_pp[vs] = pp;
    S.ex_ss[vs] = ss;
  }
  wave_sync();
}

// src/model.hpp:703-832: the last locus of the walk's model moves one
// position left and the locus it passes leaves the model
template <int KMAX>
__device__ __forceinline__ void exh_moveleft(Smem<KMAX>& S, int w, int nT, int& vs) {
  vs -= 2 * w;
  if (w == 2) {
    exh_swapadj(S, nT, vs + 1);
    exh_swapadj(S, nT, vs + 2);
    exh_swapadj(S, nT, vs);
    exh_swapadj(S, nT, vs + 1);
  } else {
    exh_swapadj(S, nT, vs);
  }
  exh_add(S, w, vs);
}

// The walk over all 2^n sub-models (src/sampler.cpp:882-980): additions,
// left moves and "two new + swap" steps in the reference's order.  lp[i]
// receives the product of the sub-model's block diagonal and lp[2^n + i] its
// residual term.  w: columns per locus.  Wave 0 only (lane 0 stores).  Out of
// line: inlined, its registers crowd the kernel's hot loops.
//
// First each column is scaled by a power of two to a diagonal entry in
// [1/2, 1).  The walk's rotations act on rows and do not see it, and its
// products of up to 40 diagonal entries stay far inside the exponent's range
// whatever the precisions (an entry is at least sqrt(d)); the exponents go back
// in with the loci's log d.
template <int KMAX>
__device__ __noinline__ void exh_walk(Smem<KMAX>& S, int nT_any, int w_any, int n_any, double* lp_any) {
  double* lp = gp(lp_any);
  const int nT = __builtin_amdgcn_readfirstlane(nT_any), w = __builtin_amdgcn_readfirstlane(w_any);
  const int n = __builtin_amdgcn_readfirstlane(n_any);
  const int lane = lane_id();
  const bool st = lane == 0;
  const uint64_t all = 1ull << n;
  if (lane < n) {
    int e = 0;
    for (int k = 0; k < w; ++k) e += __builtin_amdgcn_frexp_exp(exl(S, w * lane + k, w * lane + k));
    S.ex_ld[lane] -= (double)e * 0x1.62e42fefa39efp-1;   // ln 2
  }
  for (int c = 0; c < nT; ++c) {
    const int e = __builtin_amdgcn_frexp_exp(exl(S, c, c));
    wave_sync();
    if (lane <= c) exl(S, lane, c) = ldexp(exl(S, lane, c), -e);
  }
  wave_sync();
  unsigned __int128 ci = 0;      // walk order, five bits a position
  for (int i = 0; i < BMG_DR_MAX + 2; ++i) ci |= (unsigned __int128)(unsigned)i << (5 * i);
  // positions k - 1 and k trade places
  auto swap = [&](int k) {
    const unsigned __int128 x = ((ci >> (5 * (k - 1))) ^ (ci >> (5 * k))) & 31;
    ci ^= x << (5 * (k - 1)) | x << (5 * k);
  };
  auto at = [&](int k) { return (int)((unsigned)(ci >> (5 * k)) & 31u); };
  uint64_t cmb = 0;
  int msz = 0, vs = 0;
  auto record = [&]() {
    const double pp = S.ex_pp[vs], ss = S.ex_ss[vs];
    if (st) { lp[cmb] = pp; lp[all + cmb] = ss; }
  };
  auto left = [&]() {
    --msz;
    cmb &= ~(1ull << at(msz - 1));
    swap(msz);
    exh_moveleft(S, w, nT, vs);
    record();
  };
  record();
#pragma unroll 1
  for (int i = 0; i < n; ++i) {
    ++msz;
    if (i > 1) { ++msz; exh_add(S, w, vs); }
    cmb = (1ull << msz) - 1;
    exh_add(S, w, vs);
    record();
#pragma unroll 1
    for (int j = 0; j < i; ++j) left();
    const uint64_t nmodels = (1ull << i) - i - 1;
    uint64_t j = 0, nK = 0;
    int do_lefts = 0;
#pragma unroll 1
    while (j < nmodels) {
      if (do_lefts < 2) {
        ++msz;
        cmb |= 1ull << at(msz);
        swap(msz);
        exh_add(S, w, vs);
        exh_add(S, w, vs);
        exh_moveleft(S, w, nT, vs);
        record();
        ++j; ++do_lefts;
      } else {
        ++nK;
        const int kb = __builtin_ctzll(nK);
#pragma unroll 1
        for (int kk = 0; kk <= kb; ++kk) { left(); ++j; }
        do_lefts = 0;
      }
    }
  }
}

// src/model.hpp:602-671 (ExhModel::update_to_model) and the walk: fills
// lp[0 .. 2^n) with the log posterior (up to a constant) of every sub-model,
// bit i of the index standing for the proposed model's locus cl + i.  All
// threads; returns the largest entry.  (lp: 2^(n + 1) doubles.)
template <int KMAX>
__device__ __forceinline__ double exhaustive_modelset(Ctx<KMAX>& C, int cl, int n, double* lp) {
  Smem<KMAX>& S = C.S;
  Reg& R = C.R;
  const int w = C.D.type == BMG_AH ? 2 : 1;
  const int nT = w * n;                 // the block's columns: the last n loci
  const int c0 = R.cols - nT;           // after the fixed columns and the other loci
  for (int c = 0; c < nT; ++c)
    for (int r = threadIdx.x; r <= c; r += BMG_BLOCK) S.ex_L[P(c) + r] = S.L[P(c0 + c) + c0 + r];
  for (int i = threadIdx.x; i < nT; i += BMG_BLOCK) S.ex_v[i] = S.v[c0 + i];
  // per locus: half its columns' log d, and the prior change of the q-th one
  // (src/prior.hpp:144-158, one effect type: it depends on the number alone)
  if ((int)threadIdx.x < n) {
    const int q = threadIdx.x, type = C.D.type;
    double ld = 0.0;
    for (int k = 0; k < w; ++k) ld += 0.5 * log(S.d[c0 + w * q + k]);
    S.ex_ld[q] = ld;
    int Ns[5] = {0, 0, 0, 0, 0};
    put(Ns, type, cl + q);
    S.ex_pa[q] = prior_add_untruncated(C.K, Ns, cl + q, type);
  }
  double vv = 0.0, ldl = 0.0, ldq = 0.0;
  for (int i = threadIdx.x; i < c0; i += BMG_BLOCK) {
    vv += S.v[i] * S.v[i];
    ldl += log(S.L[P(i) + i]);
    if (i >= 1) ldq += log(S.d[i]);
  }
  vv = block_sum(vv, S.red);
  ldl = block_sum(ldl, S.red);
  ldq = 0.5 * block_sum(ldq, S.red);
  if (threadIdx.x == 0) { S.ex_pp[0] = 1.0; S.ex_ss[0] = C.K.nus2_plus_yy - vv; }
  __syncthreads();
  if (wave_id() == 0) exh_walk(S, nT, w, n, lp);
  __syncthreads();
  // the log posteriors; sub-models past a model-size limit get prior 0 (the
  // walk passes through them)
  const uint64_t all = 1ull << n;
  double mx = -INFINITY;
  for (uint64_t i = threadIdx.x; i < all; i += BMG_BLOCK) {
    double q = ldq, pr = 0.0;
    int k = 0;
    for (int b = 0; b < n; ++b)
      if ((i >> b) & 1) { q += S.ex_ld[b]; pr += S.ex_pa[k]; ++k; }
    double v = q - (ldl + log(lp[i])) + C.K.minus_n_plus_nu_2 * log(lp[all + i]) + pr;
    if (cl + k > C.K.max_size) v = -INFINITY;
    lp[i] = v;
    mx = fmax(mx, v);
  }
  mx = wave_max(mx);
  if (lane_id() == 0) S.red[wave_id()] = mx;
  __syncthreads();
  mx = S.red[0];
  for (int u = 1; u < BMG_BLOCK / 64; ++u) mx = fmax(mx, S.red[u]);
  __syncthreads();
  return mx;
}

// src/sampler.cpp:982-1049 with one effect type: adds the log proposal
// probability of reaching each sub-model by the multi-step add/remove move
// from the current model to lp[i].  Thread per sub-model; the normalisers'
// logarithms are taken as one of their product (at most 20 factors between
// the smallest weight and the trees' totals), the weights' are tabulated.
template <int KMAX>
__device__ __forceinline__ void dr_proposal_probs(Smem<KMAX>& S, int n, double z_add, double z_rem,
                                                  uint64_t cl, uint64_t m_g, double* lp) {
  const uint64_t nmodels = 1ull << n;
  double* la = S.work;                  // log weights
  double* lr = S.work + BMG_DR_MAX;
  if ((int)threadIdx.x < n) {
    la[threadIdx.x] = log(S.dq_add[threadIdx.x]);
    lr[threadIdx.x] = log(S.dq_rem[threadIdx.x]);
  }
  __syncthreads();
  for (uint64_t i = threadIdx.x; i < nmodels; i += BMG_BLOCK) {
    uint64_t max_adds = m_g - cl, max_rems = cl;
    double za = z_add, zr = z_rem;
    uint64_t isadd = 0;
    for (int j = 0; j < n; ++j) {
      const int nind = S.ex_b2n[j];
      if ((i >> j) & 1) {
        za -= S.dq_add[nind]; zr += S.dq_rem[nind];
        ++max_rems; --max_adds;
      } else {
        isadd |= 1ull << nind;
      }
    }
    double acc = lp[i], z = 1.0;
    int lrp = n - 1;
    for (int j = 0; j < n; ++j) {
      if (max_adds > 0 && max_rems > 0) acc += LOG_HALF;
      if ((isadd >> j) & 1) {
        --max_adds;
        acc += la[j];
        z *= za;
        za -= S.dq_add[j];
      } else {
        --max_rems;
        while ((isadd >> lrp) & 1) --lrp;
        acc += lr[lrp];
        z *= zr;
        zr -= S.dq_rem[lrp];
        --lrp;
      }
    }
    lp[i] = acc - log(z);
  }
}

// Second-stage draw (src/sampler.hpp:1008-1028 and 1592-1612): pairs each
// sub-model with its complement, keeps the better of the two with the
// probability of the difference, and draws one pair from the cumulative
// weights (src/utils.cpp:73-100 with `ms/2 - 3` bisection steps).  The
// pairwise transform runs a thread per pair; wave 0 forms the cumulative
// sums, one scan of 64 at a time; the
// linear part of the search is a workgroup minimum over the first index
// whose sum exceeds the draw.
template <int KMAX>
__device__ __forceinline__ uint64_t dr_second_stage(Ctx<KMAX>& C, int n, double max_log, double* p) {
  const uint64_t nmodels = 1ull << n, mask = nmodels - 1, half = nmodels / 2;
  for (uint64_t i = threadIdx.x; i < half; i += BMG_BLOCK) {
    const uint64_t j = (~i) & mask;
    const double pi = p[i], pj = p[j];
    const double a = pj - pi;
    // a pair of two zero-prior sub-models (model-size limit) has weight 0
    if (pi == -INFINITY && pj == -INFINITY) { p[i] = 0.0; p[j] = 1.0; }
    else if (a > 0) { p[i] = exp(pj - max_log) * (1 - exp(-a)); p[j] = -1.0; }
    else { p[i] = exp(pi - max_log) * (1 - exp(a)); p[j] = 1.0; }
  }
  __syncthreads();
  if (wave_id() == 0) {
    const int lane = lane_id();
    double sum = 0.0;
    for (uint64_t base = 0; base < half; base += 64) {
      const uint64_t idx = base + lane;
      const double x = idx < half ? p[idx] : 0.0;
      const double mine = sum + dpp_scan(x);
      sum = readlane_d(mine, 63);
      if (idx < half) p[idx] = mine;
    }
  }
  __syncthreads();
  const double u = rng_u01(C.R.rng);
  const double r = u * p[half - 1];
  int level = n / 2 - 3;
  uint64_t a = 0, b = half - 1;
  while (level > 0) {
    const uint64_t c = (a + b) / 2;
    if (r < p[c]) b = c; else a = c + 1;
    --level;
  }
  long long first = (long long)half;
  for (uint64_t i = a + threadIdx.x; i <= b; i += BMG_BLOCK)
    if (r < p[i]) { first = (long long)i; break; }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const long long w = __shfl_xor(first, o, 64);
    first = w < first ? w : first;
  }
  __syncthreads();
  if (lane_id() == 0) C.S.redi[wave_id()] = first;
  __syncthreads();
  for (int w = 0; w < BMG_BLOCK / 64; ++w) first = C.S.redi[w] < first ? C.S.redi[w] : first;
  uint64_t sm = first < (long long)half ? (uint64_t)first : half - 1;
  if (p[(~sm) & mask] < 0) sm = (~sm) & mask;
  __syncthreads();
  return sm;
}

// the second stage re-adds the SNPs the first stage removed, each with the
// prior precision it has in the current model (src/sampler.hpp:931-960);
// false when the model capacity does not allow it
template <int KMAX>
__device__ __forceinline__ bool readd_removed(Ctx<KMAX>& C, uint64_t ind) {
  Smem<KMAX>& S = C.S;
  const int mi = gp(C.A.model_inds)[ind];
  const int t_ind = S.c_tind[mi];
  double d2[2];
  d2[0] = S.c_d[S.c_xi1[mi]];
  d2[1] = C.D.types[t_ind] == 4 ? S.c_d[S.c_xi2[mi]] : 0.0;
  add_term(C, (uint32_t)ind, t_ind, d2);
  return !(C.R.err & ERR_CAPACITY);
}

// removes the proposed model's loci cl + i whose bit of `sm` is clear
// (src/sampler.hpp:1081-1091)
template <int KMAX>
__device__ __forceinline__ void dr_keep(Ctx<KMAX>& C, int cl, int n, uint64_t sm) {
  uint64_t removals = sm & ((1ull << n) - 1);
  int c = cl;
  for (int i = 0; i < n; ++i) {
    if ((removals & 1) == 0) { remove_term(C, c + i); --c; }
    removals >>= 1;
  }
}

// Second stage of the multi-step add/remove move after a first-stage
// rejection (src/sampler.hpp:931-1099): the removed SNPs are re-added, every
// sub-model between the current and the proposed one is scored with its
// proposal probability, and one is drawn.  Returns the number of moved SNPs
// kept (0: the current model stays).
template <int KMAX>
__device__ __forceinline__ int dr_addrem(Ctx<KMAX>& C, int ms) {
  Smem<KMAX>& S = C.S;
  Reg& R = C.R;
  int ms_rem = 0;
  for (int i = 0; i < ms; ++i) ms_rem += S.mi_isadd[i] ? 0 : 1;
  const int cl = R.c_nloci - ms_rem;
  const int ms_add = ms - ms_rem;
  double z_add = R.tot_add, z_rem = R.tot_rem;
  const uint64_t nmb = (1ull << ms_add) - 1, mask = (1ull << ms) - 1;
  bool ok = true;
  for (int i = 0; i < ms && ok; ++i) {
    const uint64_t ind = S.mi[i];
    if (S.mi_isadd[i]) { z_add += gp(C.A.q_add)[ind]; z_rem -= gp(C.A.q_rem)[ind]; }
    else ok = readd_removed(C, ind);
  }
  if (!ok) { restore(C); undo_dd(C, ms); return 0; }
  for (int i = 0; i < ms; ++i) {
    const uint64_t ind = (uint64_t)S.mi_map[i];
    const int pos = find_locus(C, ind);
    if (threadIdx.x == 0 && pos >= cl && pos - cl < ms) {
      S.ex_b2n[pos - cl] = (uint8_t)i;
      S.dq_add[i] = gp(C.A.q_add)[ind];
      S.dq_rem[i] = gp(C.A.q_rem)[ind];
    }
  }
  __syncthreads();
  double* lp = gp(C.A.dr_lp);
  const uint64_t t0 = wall_clock64();
  const double max_log = exhaustive_modelset(C, cl, ms, lp);
  dr_proposal_probs(S, ms, z_add, z_rem, (uint64_t)cl, C.D.p, lp);
  __syncthreads();
  const uint64_t sm = dr_second_stage(C, ms, max_log, lp);
  if (threadIdx.x == 0) C.prof[19] += wall_clock64() - t0;
  if (sm == ((~nmb) & mask)) { restore(C); undo_dd(C, ms); return 0; }
  int moved = 0;
  for (int i = 0; i < ms; ++i) {
    const int bit = (int)((sm >> i) & 1), nb = (int)((nmb >> i) & 1);
    if (bit == nb) { ++moved; continue; }
    const uint64_t ind = (uint64_t)S.mi_map[S.ex_b2n[i]];
    if (bit) { tree_set(C, 0, ind, 1); tree_set(C, 1, ind, 0); }
    else { tree_set(C, 0, ind, 0); tree_set(C, 1, ind, 1); }
  }
  dr_keep(C, cl, ms, sm);
  if (threadIdx.x == 0) S.r_ms_sum[ms - 1] += (double)moved / (double)ms;
  commit(C);
  return moved;
}

// Second stage of the state-change move (src/sampler.hpp:1547-1667): as
// above, scored by model size instead of proposal probabilities.
template <int KMAX>
__device__ __forceinline__ int dr_statechange(Ctx<KMAX>& C, int ms, int ms_add, int ms_rem) {
  Smem<KMAX>& S = C.S;
  Reg& R = C.R;
  const int cl = R.c_nloci - ms_rem;
  const uint64_t nmb = (1ull << ms_add) - 1, mask = (1ull << ms) - 1;
  for (int i = 0; i < ms_rem; ++i)
    if (!readd_removed(C, S.mi_rem[i])) { restore(C); return 0; }
  double* lp = gp(C.A.dr_lp);
  const uint64_t t0 = wall_clock64();
  const double max_log = exhaustive_modelset(C, cl, ms, lp);
  for (uint64_t i = threadIdx.x; i <= mask; i += BMG_BLOCK) lp[i] -= log((double)(cl + __popcll(i)));
  __syncthreads();
  const uint64_t sm = dr_second_stage(C, ms, max_log, lp);
  if (threadIdx.x == 0) C.prof[19] += wall_clock64() - t0;
  if (sm == ((~nmb) & mask)) { restore(C); return 0; }
  int moved = 0;
  for (int i = 0; i < ms; ++i) {
    const int bit = (int)((sm >> i) & 1), nb = (int)((nmb >> i) & 1);
    if (bit != nb) continue;
    ++moved;
    if (bit) { const uint64_t ind = S.mi_add[i]; tree_set(C, 0, ind, 1); tree_set(C, 1, ind, 0); }
    else { const uint64_t ind = S.mi_rem[i - ms_add]; tree_set(C, 0, ind, 0); tree_set(C, 1, ind, 1); }
  }
  dr_keep(C, cl, ms, sm);
  commit(C);
  return moved;
}

// sum over the steps i < ms of log w_i - log t_i (lane i holds step i's), plus
// log 1/2 before the steps whose bit of `halves` is set, in step order
__device__ __forceinline__ double sum_logs(double w, double t, uint64_t halves, int ms) {
  const double v = lane_id() < ms ? log(w) - log(t) : 0.0;
  double s = 0.0;
  for (int i = 0; i < ms; ++i) {
    if ((halves >> i) & 1) s += LOG_HALF;
    s += readlane_d(v, i);
  }
  return s;
}

// prior change of n_rem removals, then n_add additions, of one effect type
// from a model of n0 loci, ns0 of them of that type: a step per lane, added in
// step order
__device__ __forceinline__ double prior_steps(const ChainConst& K, int n0, int ns0, int n_rem, int n_add, int type) {
  const int k = lane_id(), ms = n_rem + n_add;
  double v = 0.0;
  if (k < ms) {
    const int d = k < n_rem ? -k : k - 2 * n_rem;
    const int n = n0 + d;
    int Ns[5] = {0, 0, 0, 0, 0};
    put(Ns, type, ns0 + d);
    v = k < n_rem ? prior_rem(K, Ns, n, type) : prior_add(K, Ns, n, type);
  }
  double s = 0.0;
  for (int i = 0; i < ms; ++i) s += readlane_d(v, i);
  return s;
}

// src/sampler.hpp:899-1123
template <int KMAX>
__device__ __forceinline__ int move_addrem(Ctx<KMAX>& C) {
  Smem<KMAX>& S = C.S;
  Reg& R = C.R;
  const ChainConst& K = C.K;
  const int type = C.D.type;
  int ms = draw_move_size(C, R.rng, 0);
  R.movesize = ms;
  double lqf = 0, lqb = 0, lmpc = 0;
  // the logarithms of a step's weight and of its normaliser are taken by the
  // step's own lane, all steps at once, and added in step order
  const int lane = lane_id();
  uint64_t halves = 0;                     // steps with a choice of direction
  double my_w = 1.0, my_t = 1.0;
  // the move's tree writes are journalled, so a rejection puts the trees
  // back without recomputing their sums
  const uint64_t tq0 = wall_clock64();
  journal_begin(C);
  const uint64_t tq1 = wall_clock64();
  // prepare_addrem (src/sampler.hpp:1126-1165)
  uint64_t max_adds = C.D.p - R.c_nloci, max_rems = R.c_nloci;
  for (int i = 0; i < ms; ++i) {
    int add;
    if (max_rems == 0) add = 1;
    else if (max_adds == 0) add = 0;
    else { halves |= 1ull << i; add = rng_u01(R.rng) < 0.5; }
    double u = rng_u01(R.rng);
    uint64_t ind;
    double wv;
    const double tot = add ? R.tot_add : R.tot_rem;
    if (add) --max_adds;
    else --max_rems;
    ind = tree_pick_zero(C, add ? 0 : 1, u, &wv);   // wv = q_add[ind] or q_rem[ind]
    if (lane == i) { my_w = wv; my_t = tot; }
    R.warm = (long long)ind; R.warm_add = add;
    if (threadIdx.x == 0) {
      S.mi_isadd[i] = (uint8_t)add; S.mi[i] = ind; S.mi_map[i] = add ? (int64_t)ind : -1;
    }
    __syncthreads();
  }
  warm_next(C);
  lqf = sum_logs(my_w, my_t, halves, ms);
  const uint64_t tq2 = wall_clock64();
  // do_addrem (src/sampler.hpp:1204-1268): removals first; the last removal's
  // downdate also forms the first addition's column dots
  int last_rem = -1;
  long long first_add = -1;
  int ms_rem = 0;
  for (int i = 0; i < ms; ++i) {
    if (!S.mi_isadd[i]) { last_rem = i; ++ms_rem; }
    else if (first_add < 0) first_add = (long long)S.mi[i];
  }
  R.pre_snp = -1;
  int last = ms - 1;
  lmpc = prior_steps(K, R.nloci, sel(R.Ns, type), ms_rem, ms - ms_rem, type);
  for (int i = 0; i < ms; ++i) {
    if (S.mi_isadd[i]) continue;
    uint64_t ind = S.mi[i];
    R.job_tr = 0; R.job_ind = ind;
    while (S.mi_map[last] >= 0) --last;
    __syncthreads();
    if (threadIdx.x == 0) S.mi_map[last] = (int64_t)ind;
    __syncthreads();
    int mind = find_locus(C, ind);
    remove_term(C, mind, i == last_rem ? first_add : -1);
    job_finish(C);
  }
  double d2[2];
  draw_new_terms(C, ms - ms_rem);
  for (int i = 0, k = 0; i < ms; ++i) {
    if (!S.mi_isadd[i]) continue;
    uint64_t ind = S.mi[i];
    long long next = -1;   // the move's next addition, whose dots are formed ahead
    for (int j = i + 1; j < ms; ++j)
      if (S.mi_isadd[j]) { next = (long long)S.mi[j]; break; }
    R.job_tr = 1; R.job_ind = ind;
    new_term(C, k++, d2);
    add_term(C, (uint32_t)ind, 0, d2, next);
    job_finish(C);
  }
  R.pre_snp = -1;
  const uint64_t tq3 = wall_clock64();
  // backward_prepare_addrem (src/sampler.hpp:1168-1202); the reverse
  // move's weights are loaded together first (thread i loads step i's)
  {
    if ((int)threadIdx.x < ms) {
      const int i = (int)threadIdx.x;
      uint64_t ind;
      if (S.mi_isadd[i]) {
        int k = 0;   // step i is the k-th addition; it pairs with the k-th from last
        for (int q = 0; q < i; ++q) k += S.mi_isadd[q];
        int lr = ms - 1, seen = 0;
        for (;; --lr) if (S.mi_isadd[lr] && seen++ == k) break;
        ind = (uint64_t)S.mi_map[lr];
        S.bq[i] = gp(C.A.q_rem)[ind];
      } else {
        ind = (uint64_t)S.mi_map[i];
        S.bq[i] = gp(C.A.q_add)[ind];
      }
    }
    __syncthreads();
    uint64_t madd = C.D.p - R.nloci, mrem = R.nloci;
    double w_add = R.tot_add, w_rem = R.tot_rem;
    halves = 0;
    for (int i = 0; i < ms; ++i) {
      if (madd > 0 && mrem > 0) halves |= 1ull << i;
      const double q = S.bq[i];
      const int add = S.mi_isadd[i];
      if (lane == i) { my_w = q; my_t = add ? w_rem : w_add; }
      if (add) { --mrem; w_rem -= q; }
      else { --madd; w_add -= q; }
    }
    lqb = sum_logs(my_w, my_t, halves, ms);
    __syncthreads();
  }
  double log_r = lqb - lqf;
  log_r += lmpc + R.ll - R.c_ll;
  const uint64_t tq4 = wall_clock64();
  if (threadIdx.x == 0) {
    C.prof[20] += tq2 - tq1; C.prof[21] += tq3 - tq2; C.prof[22] += tq4 - tq3; C.prof[23] += tq1 - tq0;
  }
  if (threadIdx.x == 0) {
    if (K.dr == 0) S.r_ms_sum[ms - 1] += (log_r >= 0 ? 1.0 : exp(log_r));
    S.r_ms_n[ms - 1] += 1.0;
  }
  if (log_r >= 0 || log(rng_u01(R.rng)) <= log_r) {
    R.tj_on = 0;
    commit(C);
    if (K.dr != 0 && threadIdx.x == 0) S.r_ms_sum[ms - 1] += 1.0;
    if (threadIdx.x == 0) C.prof[23] += wall_clock64() - tq4;
    return ms;
  }
  // a proposal past the compiled capacity has no second stage
  if (ms <= K.dr && ms > 1 && !(R.err & ERR_CAPACITY)) {
    R.tj_on = 0;
    const uint64_t t0 = wall_clock64();
    const int moved = dr_addrem(C, ms);
    if (threadIdx.x == 0) C.prof[18] += wall_clock64() - t0;
    return moved;
  }
  restore(C);
  journal_restore(C);
  if (threadIdx.x == 0) C.prof[23] += wall_clock64() - tq4;
  return 0;
}

// is SNP j in the current model (with the switch move's temporary marks)?
template <int KMAX>
__device__ __forceinline__ int cur_in_model(Ctx<KMAX>& C, int64_t j, int64_t wbase) {
  if (j < 0 || j >= (int64_t)C.D.p) return 0;   // outside the genome: stops a walk
  for (int q = 0; q < C.R.n_marks; ++q) if ((int64_t)C.S.marks[q] == j) return 1;
  if (j >= wbase && j < wbase + 512) return C.S.win[j - wbase] >= 0;
  return gp(C.A.model_inds)[j] >= 0;
}

template <int KMAX>
__device__ __forceinline__ void load_window(Ctx<KMAX>& C, int64_t center, int64_t* wbase) {
  int64_t b = center - 256;
  if (b < 0) b = 0;
  __syncthreads();
  for (int t = threadIdx.x; t < 512; t += BMG_BLOCK) {
    int64_t j = b + t;
    C.S.win[t] = (j < (int64_t)C.D.p) ? gp(C.A.model_inds)[j] : -1;
  }
  __syncthreads();
  *wbase = b;
}

// src/sampler.hpp:1271-1418
template <int KMAX>
__device__ __forceinline__ int move_switch(Ctx<KMAX>& C) {
  Smem<KMAX>& S = C.S;
  Reg& R = C.R;
  const ChainConst& K = C.K;
  uint64_t full = C.D.p - R.c_nloci;
  int ms = draw_move_size(C, R.rng, 1);
  R.movesize = ms;
  uint64_t nbh = (full - ms) / 2;
  if (nbh < 1) nbh = 1;
  if (nbh > K.max_nbh) nbh = K.max_nbh;
  int64_t m_g = (int64_t)C.D.p;
  R.n_marks = 0;
  for (int i = 0; i < ms; ++i) {
    int mir = (int)floor(rng_u01(R.rng) * R.nloci);
    int64_t ir = S.loci[mir];
    int64_t wb;
    load_window(C, ir, &wb);
    int64_t ia;
    int j = 0;
    int move = (int)floor(rng_u01(R.rng) * nbh) + 1;
    if (rng_u01(R.rng) < 0.5) {
      ia = ir; j = 0;
      while (j < move) {
        ++ia;
        if (ia < m_g) { if (!cur_in_model(C, ia, wb)) ++j; }
        else break;
      }
      if (ia == m_g) {
        ia = ir; move = move + move - j; j = 0;
        while (j < move) {
          --ia;
          while (cur_in_model(C, ia, wb)) --ia;
          ++j;
        }
      }
    } else {
      ia = ir; j = 0;
      if (ia > 0) {
        while (j < move) {
          --ia;
          if (ia > 0) { if (!cur_in_model(C, ia, wb)) ++j; }
          else break;
        }
      }
      if (j < move) {
        if (!cur_in_model(C, ia, wb)) ++j;
        if (j < move) {
          ia = ir; move = move + move - j; j = 0;
          while (j < move) {
            ++ia;
            while (cur_in_model(C, ia, wb)) ++ia;
            ++j;
          }
        }
      }
    }
    if (ia < 0 || ia >= m_g) { R.err |= ERR_WALK; ia = ia < 0 ? 0 : m_g - 1; }
    int t_ind = S.tind[mir];
    __syncthreads();
    if (threadIdx.x == 0) {
      S.mi_rem[i] = (uint64_t)ir; S.mi_add[i] = (uint64_t)ia;
      S.marks[R.n_marks] = (uint64_t)ia; S.mark_val[R.n_marks] = t_ind;
    }
    __syncthreads();
    R.n_marks++;
    remove_term(C, mir);
  }
  double d2[2];
  draw_new_terms(C, ms);
  for (int i = 0; i < ms; ++i) {
    uint64_t ia = S.mi_add[i];
    int t_ind = S.mark_val[i];
    new_term(C, i, d2);
    add_term(C, (uint32_t)ia, t_ind, d2);
  }
  R.n_marks = 0;
  double log_r = R.ll - R.c_ll;
  if (log_r >= 0 || log(rng_u01(R.rng)) <= log_r) {
    commit(C);
    for (int i = 0; i < ms; ++i) {
      tree_set(C, 0, S.mi_rem[i], 0); tree_set(C, 1, S.mi_rem[i], 1);
      tree_set(C, 0, S.mi_add[i], 1); tree_set(C, 1, S.mi_add[i], 0);
    }
    return 2 * ms;
  }
  restore(C);
  return 0;
}

// Learned swap (no counterpart in the reference): the swap of
// src/sampler.hpp:1271-1418 with the partner of the removed SNP j drawn from
// the frozen weights W[j][.] over the SNPs within lH of j that are not in
// the model, and the exact Hastings ratio
//   log W[k][j] - log Z_r - log W[j][k] + log Z_f
// (Z_f, Z_r: forward / reverse normalisers; the uniform choice of the
// removed SNP and the prior cancel because the size is unchanged).  Column
// c of a weight row is the offset c < lH ? c - lH : c - lH + 1.  Lanes
// gather the masked weights into LDS; every lane then runs the same
// sequential sums, so the draw and the ratio are those of the oracle.
__device__ __forceinline__ int lw_off(int H, int c) { return c < H ? c - H : c - H + 1; }
__device__ __forceinline__ int lw_col(int H, int o) { return o < 0 ? o + H : o + H - 1; }

template <int KMAX>
__device__ __forceinline__ int move_learned_swap(Ctx<KMAX>& C) {
  Smem<KMAX>& S = C.S;
  Reg& R = C.R;
  const int H = C.D.lH;
  const int64_t m_g = (int64_t)C.D.p;
  R.movesize = 1;
  int mir = (int)floor(rng_u01(R.rng) * R.nloci);
  if (mir >= R.nloci) mir = R.nloci - 1;
  const int64_t j = S.loci[mir];
  double* wf = S.work;            // 2H forward weights (0: not a candidate)
  double* wr = S.work + 2 * H;    // 2H reverse weights
  __syncthreads();
  if (threadIdx.x < 2 * H) {
    int64_t k = j + lw_off(H, threadIdx.x);
    double w = 0.0;
    if (k >= 0 && k < m_g && gp(C.A.model_inds)[k] < 0) w = (double)gp(C.D.lw)[(size_t)j * 2 * H + threadIdx.x];
    wf[threadIdx.x] = w;
  }
  __syncthreads();
  double zf = 0.0;
  for (int c = 0; c < 2 * H; ++c) zf += wf[c];
  if (!(zf > 0.0)) return 0;
  double u = rng_u01(R.rng) * zf, acc = 0.0;
  int pick = -1;
  for (int c = 0; c < 2 * H; ++c) {
    if (wf[c] > 0.0) {
      acc += wf[c];
      pick = c;
      if (u < acc) break;
    }
  }
  if (pick < 0) return 0;
  const int64_t k = j + lw_off(H, pick);
  const double wjk = wf[pick];
  __syncthreads();
  if (threadIdx.x < 2 * H) {
    int64_t q = k + lw_off(H, threadIdx.x);
    double w = 0.0;
    if (q >= 0 && q < m_g && (q == j || gp(C.A.model_inds)[q] < 0))
      w = (double)gp(C.D.lw)[(size_t)k * 2 * H + threadIdx.x];
    wr[threadIdx.x] = w;
  }
  __syncthreads();
  double zr = 0.0;
  for (int c = 0; c < 2 * H; ++c) zr += wr[c];
  const double wkj = wr[lw_col(H, (int)(j - k))];
  if (!(wkj > 0.0)) return 0;
  const double lq = log(wkj) - log(zr) - log(wjk) + log(zf);
  const int t_ind = S.tind[mir];
  __syncthreads();
  if (threadIdx.x == 0) { S.mi_rem[0] = (uint64_t)j; S.mi_add[0] = (uint64_t)k; }
  remove_term(C, mir);
  double d2[2];
  draw_new_terms(C, 1);
  new_term(C, 0, d2);
  add_term(C, (uint32_t)k, t_ind, d2);
  double log_r = R.ll - R.c_ll + lq;
  if (log_r >= 0 || log(rng_u01(R.rng)) <= log_r) {
    commit(C);
    tree_set(C, 0, (uint64_t)j, 0); tree_set(C, 1, (uint64_t)j, 1);
    tree_set(C, 0, (uint64_t)k, 1); tree_set(C, 1, (uint64_t)k, 0);
    return 2;
  }
  restore(C);
  return 0;
}

// src/sampler.hpp:1421-1669
template <int KMAX>
__device__ __forceinline__ int move_statechange(Ctx<KMAX>& C) {
  Smem<KMAX>& S = C.S;
  Reg& R = C.R;
  const ChainConst& K = C.K;
  const int type = C.D.type;
  uint64_t m_g = C.D.p;
  int ms = draw_move_size(C, R.rng, 2);
  R.movesize = ms;
  uint64_t nbh = K.max_nbh < m_g / 2 ? K.max_nbh : m_g / 2;
  int mic = (int)floor(rng_u01(R.rng) * R.nloci);
  uint64_t ic = S.loci[mic];
  // partial Fisher-Yates over the 2 nbh offsets (only the first ms entries
  // are used): positions that differ from the identity are kept as a sparse
  // map in LDS by thread 0; every thread consumes the same draws
  __syncthreads();
  int nsw = 0;
  for (int i = 0; i < ms; ++i) {
    uint64_t ind = (uint64_t)floor(rng_u01(R.rng) * (double)(nbh * 2 - i)) + i;
    if (threadIdx.x == 0) {
      uint64_t vi = i, vind = ind;
      for (int q = 0; q < nsw; ++q) {
        if (S.sc_from[q] == (uint64_t)i) vi = S.sc_to[q];
        if (S.sc_from[q] == ind) vind = S.sc_to[q];
      }
      S.sc_perm[i] = vind;
      int found = 0;
      for (int q = 0; q < nsw; ++q) if (S.sc_from[q] == ind) { S.sc_to[q] = vi; found = 1; }
      if (!found) { S.sc_from[nsw] = ind; S.sc_to[nsw] = vi; }
    }
    // every thread tracks the map size identically
    {
      int found = 0;
      __syncthreads();
      for (int q = 0; q < nsw; ++q) if (S.sc_from[q] == ind) found = 1;
      if (!found) ++nsw;
      __syncthreads();
    }
  }
  __syncthreads();
  uint64_t wrap = ic + nbh;
  if (ic < nbh) wrap += (nbh - ic);
  else if (wrap > m_g - 1) wrap = m_g - 1;
  int ms_rem = 0, ms_add = 0;
  for (int i = 0; i < ms; ++i) {
    uint64_t ind = S.sc_perm[i] + ic + 1;
    if (ind > wrap) ind = ic - (ind - wrap);
    if (ind >= m_g) { R.err |= ERR_WALK; ind = m_g - 1; }
    int fl = find_locus(C, ind);
    if (threadIdx.x == 0) {
      if (fl < 0) S.mi_add[ms_add] = ind; else S.mi_rem[ms_rem] = ind;
    }
    if (fl < 0) ++ms_add; else ++ms_rem;
  }
  __syncthreads();
  const double lmpc = prior_steps(K, R.nloci, sel(R.Ns, type), ms_rem, ms_add, type);
  R.pre_snp = -1;
  for (int i = 0; i < ms_rem; ++i) {
    int mir = find_locus(C, S.mi_rem[i]);
    // the last removal's downdate also forms the first addition's dots
    remove_term(C, mir, i + 1 == ms_rem && ms_add > 0 ? (long long)S.mi_add[0] : -1);
  }
  double d2[2];
  int t_ind = 0;
  draw_new_terms(C, ms_add);
  for (int i = 0; i < ms_add; ++i) {
    uint64_t ia = S.mi_add[i];
    new_term(C, i, d2);
    // the next addition's dots are formed during this one's sweep
    add_term(C, (uint32_t)ia, t_ind, d2, i + 1 < ms_add ? (long long)S.mi_add[i + 1] : -1);
  }
  R.pre_snp = -1;
  double log_r = lmpc + R.ll - R.c_ll;
  log_r += log((double)R.c_nloci) - log((double)R.nloci);
  if (log_r >= 0 || log(rng_u01(R.rng)) <= log_r) {
    commit(C);
    for (int i = 0; i < ms_add; ++i) { tree_set(C, 0, S.mi_add[i], 1); tree_set(C, 1, S.mi_add[i], 0); }
    for (int i = 0; i < ms_rem; ++i) { tree_set(C, 0, S.mi_rem[i], 0); tree_set(C, 1, S.mi_rem[i], 1); }
    return ms;
  }
  if (ms <= K.dr && ms > 1 && !(R.err & ERR_CAPACITY)) {
    const uint64_t t0 = wall_clock64();
    const int moved = dr_statechange(C, ms, ms_add, ms_rem);
    if (threadIdx.x == 0) C.prof[18] += wall_clock64() - t0;
    return moved;
  }
  restore(C);
  return 0;
}

// src/sampler.hpp:1728-1769
__device__ __forceinline__ void adapt_jd_mb(double* p_ms, double* q_p0, const double* r_ms, const double* r_n,
                                            int max_ms) {
  double q = 1 - *p_ms;
  double zp = 1 - pow(q, max_ms);
  double q_p = *p_ms / zp;
  for (int i = 0; i < max_ms; ++i) { q_p0[i] += q_p; q_p *= q; }
  double p_best = 0.01, p = 0.01, h_best = -INFINITY, h;
  double step = 0.98 / 49.0, ratio;
  for (int j = 0; j < 50; ++j) {
    h = 0.0; zp = 0.0; q = 1.0 - p; q_p = p;
    for (int i = 0; i < max_ms; ++i) {
      ratio = q_p / q_p0[i];
      h += (i + 1) * r_ms[i] * ratio;
      zp += r_n[i] * ratio;
      q_p *= q;
    }
    h /= zp;
    if (h > h_best) { h_best = h; p_best = p; }
    p += step;
  }
  *p_ms = p_best;
}

__device__ __forceinline__ void geometric_cdf(int maxsize, double p, double* values) {
  double q = 1 - p, qp = q;
  for (int i = 0; i < maxsize; ++i) { values[i] = 1 - q; q *= qp; }
}

// --------------------------------------------------------------- kernel ---

// the descriptions of the chain's dataset, options and arrays into LDS
template <typename T>
__device__ __forceinline__ void copy_words(T& dst, const T* src) {
  static_assert(sizeof(T) % 4 == 0, "whole words");
  uint32_t* d = (uint32_t*)&dst;
  const uint32_t* w = (const uint32_t*)src;
  for (int i = threadIdx.x; i < (int)(sizeof(T) / 4); i += BMG_BLOCK) d[i] = w[i];
}
template <int KMAX>
__device__ __forceinline__ void load_descriptions(Smem<KMAX>& S, const DevData* data, const ChainConst* K,
                                                  const ChainArrays* A) {
  copy_words(S.K, K);
  copy_words(S.A, A);
  copy_words(S.D, data + K->ds);
  __syncthreads();
  if constexpr (KMAX > KMAX_LDS) {
    if (threadIdx.x == 0) S.L.p = S.A.Lwork;
    __syncthreads();
  }
}

template <int KMAX>
__device__ __forceinline__ void load_chain(Ctx<KMAX>& C, const ChainScal& CS) {
  Smem<KMAX>& S = C.S;
  Reg& R = C.R;
  (Rng&)R.rng = rng_make(C.K.seed, C.K.chain_id, 0, 0);
  R.rng.c0 = CS.rng_c0; R.rng.c1 = CS.rng_c1;
  R.rng.base = ((uint64_t)R.rng.c1 << 32 | R.rng.c0) - 64;   // no block at hand
  R.cols = R.c_cols = CS.cols;
  R.nloci = R.c_nloci = CS.nloci;
  for (int q = 0; q < 5; ++q) R.Ns[q] = R.c_Ns[q] = CS.Ns[q];
  R.syx = R.c_syx = CS.syx; R.ldq = R.c_ldq = CS.ldq; R.ldl = R.c_ldl = CS.ldl;
  R.ll = R.c_ll = CS.ll;
  R.sigma2 = CS.sigma2; R.alpha = CS.alpha; R.alpha2 = CS.alpha2;
  for (int q = 0; q < 4; ++q) R.ita2[q] = CS.inv_tau2_alpha2[q];
  R.beta_len = CS.beta_len; R.mu_computed = CS.mu_computed;
  R.lmin = KMAX; R.n_rm = 0; R.n_marks = 0; R.movesize = CS.movesize;
  R.tot_add = CS.tot_add; R.tot_rem = CS.tot_rem;
  R.err = CS.err;
  if (threadIdx.x < 24) S.prof[threadIdx.x] = CS.prof[threadIdx.x];
  if (threadIdx.x < 4) {
    S.cnt.n_acpt[threadIdx.x] = CS.n_acpt[threadIdx.x];
    S.cnt.n_moves[threadIdx.x] = CS.n_moves[threadIdx.x];
  }
  if (threadIdx.x == 0) {
    S.cnt.n_accepted = CS.n_accepted;
    S.cnt.tr_count = CS.tr_count; S.cnt.th_count = CS.th_count;
    S.cnt.th_loci_len = CS.th_loci_len; S.cnt.th_beta_len = CS.th_beta_len;
  }
  if (threadIdx.x < BMG_MAXMS) {
    const double* ad = gp(C.A.adapt) + threadIdx.x;
    for (int q = 0; q < 3; ++q) S.cdf[q][threadIdx.x] = ad[q * 256];
    S.r_ms_sum[threadIdx.x] = ad[3 * 256];
    S.r_ms_n[threadIdx.x] = ad[4 * 256];
  }
  R.learn_on = CS.learn_on && C.D.lw != nullptr && C.D.lH >= 1 && C.D.lH <= BMG_LH_MAX;
  R.tj_on = 0; R.tj_n = 0; R.tj_tot[0] = R.tj_tot[1] = 0.0;
  R.pre_snp = -1; R.pre_slot = -1;
  R.warm = -1; R.warm_add = 0;
  R.job_tr = -1; R.job_ind = 0;
  const double* vec = gp(C.A.vec);
  const int32_t* idx = gp(C.A.idx);
  copy_factor(S.L, gp(C.A.Lcur), 0, P(R.cols));
  for (int i = threadIdx.x; i < KMAX; i += BMG_BLOCK) {
    S.xy[i] = S.c_xy[i] = vec[i];
    S.v[i] = S.c_v[i] = vec[BMG_KMAXG + i];
    S.d[i] = S.c_d[i] = vec[2 * BMG_KMAXG + i];
    S.beta[i] = vec[3 * BMG_KMAXG + i];
    S.mu[i] = vec[4 * BMG_KMAXG + i];
    S.loci[i] = S.c_loci[i] = (uint32_t)idx[i];
    S.xi1[i] = S.c_xi1[i] = idx[BMG_KMAXG + i];
    S.xi2[i] = S.c_xi2[i] = idx[2 * BMG_KMAXG + i];
    S.slot[i] = S.c_slot[i] = idx[3 * BMG_KMAXG + i];
    S.snp[i] = S.c_snp[i] = idx[4 * BMG_KMAXG + i];
    S.xtype[i] = S.c_xtype[i] = (int8_t)idx[5 * BMG_KMAXG + i];
    S.tind[i] = S.c_tind[i] = (int8_t)idx[6 * BMG_KMAXG + i];
  }
  if (threadIdx.x < BMG_KMAXG / 64) S.slots_cur[threadIdx.x] = 0;
  __syncthreads();
  for (int i = threadIdx.x; i < R.cols; i += BMG_BLOCK)
    atomicOr((unsigned long long*)&S.slots_cur[S.slot[i] >> 6], 1ull << (S.slot[i] & 63));
  __syncthreads();
  if (threadIdx.x < BMG_KMAXG / 64) S.slots_prop[threadIdx.x] = S.slots_cur[threadIdx.x];
  // sum-tree levels >= 2
  if (C.D.top >= 2) {
    uint64_t o2 = C.D.lev_off[2];
    for (uint64_t e = threadIdx.x; e < C.D.lds_lev_size; e += BMG_BLOCK) {
      S.tlev[0][e] = gp(C.A.tree_add)[o2 + e];
      S.tlev[1][e] = gp(C.A.tree_rem)[o2 + e];
    }
  }
  __syncthreads();
}

template <int KMAX>
__device__ __forceinline__ void store_chain(Ctx<KMAX>& C, ChainScal& CS) {
  Smem<KMAX>& S = C.S;
  Reg& R = C.R;
  __syncthreads();
  double* vec = gp(C.A.vec);
  int32_t* idx = gp(C.A.idx);
  for (int i = threadIdx.x; i < KMAX; i += BMG_BLOCK) {
    vec[i] = S.c_xy[i]; vec[BMG_KMAXG + i] = S.c_v[i]; vec[2 * BMG_KMAXG + i] = S.c_d[i];
    vec[3 * BMG_KMAXG + i] = S.beta[i]; vec[4 * BMG_KMAXG + i] = S.mu[i];
    idx[i] = (int32_t)S.c_loci[i]; idx[BMG_KMAXG + i] = S.c_xi1[i]; idx[2 * BMG_KMAXG + i] = S.c_xi2[i];
    idx[3 * BMG_KMAXG + i] = S.c_slot[i]; idx[4 * BMG_KMAXG + i] = S.c_snp[i];
    idx[5 * BMG_KMAXG + i] = S.c_xtype[i]; idx[6 * BMG_KMAXG + i] = S.c_tind[i];
  }
  if (C.D.top >= 2) {
    uint64_t o2 = C.D.lev_off[2];
    for (uint64_t e = threadIdx.x; e < C.D.lds_lev_size; e += BMG_BLOCK) {
      gp(C.A.tree_add)[o2 + e] = S.tlev[0][e];
      gp(C.A.tree_rem)[o2 + e] = S.tlev[1][e];
    }
  }
  if (threadIdx.x == 0) {
    CS.rng_c0 = R.rng.c0; CS.rng_c1 = R.rng.c1;
    CS.cols = R.c_cols; CS.nloci = R.c_nloci;
    for (int q = 0; q < 5; ++q) CS.Ns[q] = R.c_Ns[q];
    CS.syx = R.c_syx; CS.ldq = R.c_ldq; CS.ldl = R.c_ldl; CS.ll = R.c_ll;
    CS.sigma2 = R.sigma2; CS.alpha = R.alpha; CS.alpha2 = R.alpha2;
    for (int q = 0; q < 4; ++q) CS.inv_tau2_alpha2[q] = R.ita2[q];
    CS.beta_len = R.beta_len; CS.mu_computed = R.mu_computed;
    CS.movesize = R.movesize;
    CS.tot_add = R.tot_add; CS.tot_rem = R.tot_rem;
    CS.err = R.err;
    CS.n_accepted = S.cnt.n_accepted;
    CS.tr_count = S.cnt.tr_count; CS.th_count = S.cnt.th_count;
    CS.th_loci_len = S.cnt.th_loci_len; CS.th_beta_len = S.cnt.th_beta_len;
  }
  if (threadIdx.x < 24) CS.prof[threadIdx.x] = S.prof[threadIdx.x];
  if (threadIdx.x < 4) {
    CS.n_acpt[threadIdx.x] = S.cnt.n_acpt[threadIdx.x];
    CS.n_moves[threadIdx.x] = S.cnt.n_moves[threadIdx.x];
  }
  if (threadIdx.x < BMG_MAXMS) {
    double* ad = gp(C.A.adapt) + threadIdx.x;
    ad[3 * 256] = S.r_ms_sum[threadIdx.x];
    ad[4 * 256] = S.r_ms_n[threadIdx.x];
  }
  __syncthreads();
}

// the tau2/alpha refresh at the top of an iteration (src/sampler.cpp:628-635)
// acts on the current model; here the working copy equals it, and the
// refreshed model is committed in full
template <int KMAX>
__device__ __forceinline__ void refresh_tau2(Ctx<KMAX>& C) {
  Reg& R = C.R;
  // a refresh whose factorisation fails is undone (as in the oracle): the
  // previous tau2 / alpha and the committed model are kept
  const double al = R.alpha, al2 = R.alpha2;
  double ita[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) ita[q] = R.ita2[q];
  const uint64_t t0 = wall_clock64();
  sample_alpha_and_tau2(C);
  if (threadIdx.x == 0) C.prof[15] += wall_clock64() - t0;
  compute_log_likelihood(C);
  R.lmin = 0;
  if (isfinite(R.ll)) {
    commit(C);
  } else {
    restore(C);
    R.alpha = al; R.alpha2 = al2;
#pragma unroll
    for (int q = 0; q < 4; ++q) R.ita2[q] = ita[q];
  }
}

// Columns that the next move can add to the current model at its largest:
// the move and its size follow from the stream's next draws, read ahead here
// on a copy of the stream.  Swaps remove before they add.
template <int KMAX>
__device__ __forceinline__ int next_growth(Ctx<KMAX>& C) {
  Reg& R = C.R;
  ChainRng q = R.rng;
  const int move = draw_move(C, q);
  if (move == 1 || move == 3) return 0;
  const int ms = draw_move_size(C, q, move);
  const int wide = C.D.type == BMG_AH ? 2 : 1;
  if (move == 2 || R.c_cols + wide * ms <= KMAX_LDS) return wide * ms;
  // an add/remove move: only the SNPs drawn for addition
  uint64_t max_adds = C.D.p - R.c_nloci, max_rems = R.c_nloci;
  int adds = 0;
  for (int i = 0; i < ms; ++i) {
    int add = 1;
    if (max_rems == 0) add = 1;
    else if (max_adds == 0) add = 0;
    else add = rng_u01(q) < 0.5;
    rng_skip(q, 1);
    if (add) { --max_adds; ++adds; }
    else --max_rems;
  }
  return wide * adds;
}

// Iterations of one chain from g.iter up to `end`, to the next RB point, or
// until the model's size asks for the other capacity's code (g.change; `cap`:
// the launch's capacity, in the 256-column code the one to go back to, or
// 256).
template <int KMAX>
__device__ __forceinline__ void run_iterations(Ctx<KMAX>& C, ChainScal& CS, Progress& g, uint64_t end, int cap) {
  Smem<KMAX>& S = C.S;
  Reg& R = C.R;
  const ChainConst& K = C.K;
  double* adapt = gp(C.A.adapt);
  uint64_t pr[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  uint64_t iter = g.iter;
  int refreshed = g.refreshed;
  g.change = g.refreshed = 0;
  for (; iter < end; ++iter) {
    // a chain whose current model turned non-finite stops here; the host
    // reports it (the oracle stops with an error at the same point)
    if (R.err & ERR_STOP) break;
    const uint64_t t_it = wall_clock64();
    uint64_t t0 = t_it;
    if ((iter + 1) % K.n_st == 0 && !refreshed) {
      refresh_tau2(C);
      if (!isfinite(R.c_ll)) R.err |= ERR_NONFINITE;
      uint64_t t1 = wall_clock64(); pr[0] += t1 - t0; t0 = t1;
    }
    refreshed = 0;
    // a model that the move may take past the capacity continues in the
    // 256-column code from here, before any of the move's draws, so the
    // trajectory is the one a 256-column launch gives; it comes back once
    // it is CAP_BACK columns inside again and the move fits.  (Deciding by
    // the largest move there can be, max_move_size, kept chains past 139
    // columns, 119 with two a SNP, out of the LDS code: 500 iterations of 8
    // chains with two columns a SNP took 148 ms instead of 135, of 16 chains at
    // n = 10,000, p = 500,000 139 instead of 135.)
    if (cap < BMG_KMAXG) {
      const int most = (int)K.max_ms * (C.D.type == BMG_AH ? 2 : 1);
      if (KMAX < BMG_KMAXG ? R.c_cols + most > cap && R.c_cols + next_growth(C) > cap
                           : R.c_cols + CAP_BACK <= cap && R.c_cols + next_growth(C) <= cap) {
        g.change = 1;
        g.refreshed = (iter + 1) % K.n_st == 0;
        break;
      }
    }
    const int move = draw_move(C, R.rng);
    int jd = 0;
    if (move == 3) {
      if (R.c_nloci > 0) jd = move_learned_swap(C);
    } else if (move == 0) jd = move_addrem(C);
    else if (move == 1) {
      if (R.c_nloci > 0 && (uint64_t)R.c_nloci < C.D.p - 1) jd = move_switch(C);
    } else {
      if (R.c_nloci > 0 && C.D.p > 2) jd = move_statechange(C);
    }
    {
      const uint64_t t1 = wall_clock64(), dt = t1 - t0;
      if (move == 0) pr[1] += dt;
      else if (move == 1) pr[2] += dt;
      else if (move == 2) pr[3] += dt;
      else pr[4] += dt;
      t0 = t1;
    }
    if (threadIdx.x == 0) {
      S.cnt.n_moves[move]++;
      S.cnt.n_acpt[move] += jd > 0;
      S.cnt.n_accepted += jd > 0;
    }
    if ((iter + 1) % K.thin == 0 || (iter + 2) % K.n_st == 0) {
      sample_beta_sigma2(C);
      uint64_t t1 = wall_clock64(); pr[5] += t1 - t0; t0 = t1;
    }
    if (K.trace_iter && threadIdx.x == 0) {
      uint64_t t = S.cnt.tr_count;
      if (t < K.tr_cap) {
        gp(C.A.tr_move)[t] = (uint8_t)move; gp(C.A.tr_jd)[t] = (uint8_t)jd;
        gp(C.A.tr_ms)[t] = (uint8_t)R.movesize; gp(C.A.tr_size)[t] = (uint32_t)R.c_nloci;
        gp(C.A.tr_ll)[t] = R.c_ll;
      } else {
        R.err |= ERR_TRACE;
      }
      S.cnt.tr_count = t + 1;
    }
    if ((iter + 1) % K.thin == 0) {
      double pves[3];
      compute_pve(C, pves, (iter + 1) % K.n_rao == 0);
      const uint64_t t = S.cnt.th_count, ll0 = S.cnt.th_loci_len, b0 = S.cnt.th_beta_len;
      const bool fits = t < K.th_cap && ll0 + R.c_nloci <= K.th_loci_cap;
      // save_beta (src/sampler.cpp:710-713): the beta drawn for this sample
      const bool keep_beta = fits && K.th_beta_cap != 0 && b0 + R.beta_len <= K.th_beta_cap;
      if (fits)
        for (int q = threadIdx.x; q < R.c_nloci; q += BMG_BLOCK) gp(C.A.th_loci)[ll0 + q] = S.c_loci[q];
      if (keep_beta)
        for (int q = threadIdx.x; q < R.beta_len; q += BMG_BLOCK) gp(C.A.th_beta)[b0 + q] = S.beta[q];
      __syncthreads();
      if (threadIdx.x == 0) {
        if (fits) {
          gp(C.A.th_size)[t] = (uint32_t)R.c_nloci;
          gp(C.A.th_ll)[t] = R.c_ll; gp(C.A.th_s2)[t] = R.sigma2; gp(C.A.th_alpha)[t] = R.alpha;
          gp(C.A.th_pve)[3 * t] = pves[0]; gp(C.A.th_pve)[3 * t + 1] = pves[1]; gp(C.A.th_pve)[3 * t + 2] = pves[2];
          S.cnt.th_count = t + 1; S.cnt.th_loci_len = ll0 + R.c_nloci;
          if (keep_beta) S.cnt.th_beta_len = b0 + R.beta_len;
        }
        if (!fits || (K.th_beta_cap != 0 && !keep_beta)) R.err |= ERR_TRACE;
        CS.pves[0] = pves[0]; CS.pves[1] = pves[1]; CS.pves[2] = pves[2];
      }
      uint64_t t1 = wall_clock64(); pr[6] += t1 - t0; t0 = t1;
    }
    pr[7] += wall_clock64() - t_it;
    if ((iter + 1) % K.n_rao == 0) {
      // decide the RB block now; the scan and proposal update run as
      // separate kernels before the next iteration (src/sampler.cpp:731-811)
      if (threadIdx.x == 0) {
        CS.rb_pending = 1;
        CS.rb_do_scan = (!K.flat || CS.n_rao_burnin <= 0);
        if (CS.rb_do_scan) { CS.rb_call_idx = CS.rb_calls; CS.rb_calls++; }
        if (CS.n_rao_burnin <= 0) {
          CS.rb_accum_rao = 1;
          CS.rao_z1 = (double)(CS.p_rao_n + 1);
          CS.rao_z2 = (double)CS.p_rao_n / CS.rao_z1;
          CS.p_rao_n++;
        } else {
          CS.rb_accum_rao = 0;
          CS.n_rao_burnin--;
        }
        CS.rb_update_prop = 0; CS.rb_rebuild = 0;
        if (K.adaptation || CS.n_rao_burnin > 0) {
          if (!K.flat) {
            CS.rb_update_prop = 1;
            CS.prop_z1 = (double)(CS.p_proposal_n + 1);
            CS.prop_z2 = (double)CS.p_proposal_n / CS.prop_z1;
          }
          if (K.adapt_p_ms) {
            if (K.acpt_goal > 0) {
              double t = fmax(1.0, K.k_move_size * (double)CS.p_proposal_n);
              double ar = (double)S.cnt.n_acpt[0] / (double)S.cnt.n_moves[0];
              double pm2 = CS.p_ms + (K.acpt_goal - ar) / (2.0 + t);
              CS.p_ms = fmax(fmin(pm2, 0.99), 0.01);
              S.cnt.n_acpt[0] = 1; S.cnt.n_moves[0] = 2;
            } else {
              double pms = CS.p_ms;
              adapt_jd_mb(&pms, adapt + 5 * 256, S.r_ms_sum, S.r_ms_n, (int)K.max_ms);
              CS.p_ms = pms;
            }
            geometric_cdf((int)K.max_ms, CS.p_ms, adapt);
          }
          CS.p_proposal_n++;
          if (!K.flat) CS.rb_rebuild = 1;
        }
      }
      ++iter;
      break;   // the RB block runs before the next iteration
    }
  }
  if (threadIdx.x == 0) {
    CS.n_iter = iter;
#pragma unroll
    for (int q = 0; q < 8; ++q) S.prof[q] += pr[q];
  }
  __syncthreads();
  g.iter = iter;
}

// The chain in the code of one capacity: load, set up (mode 1) or iterate,
// store.  Out of line: with both codes in one body the compiler runs out of
// registers.
template <int KMAX>
__device__ __noinline__ Progress run_capacity(Smem<KMAX>& S, KernelArgs args, Progress g, uint64_t end) {
  const int c = blockIdx.x;
  ChainScal& CS = args.scal[c];
  load_descriptions(S, args.data, args.consts + c, args.arrays + c);
  Reg R;
  Ctx<KMAX> C{S, R, S.D, S.K, S.A, S.prof};
  load_chain(C, CS);
  if (KMAX < BMG_KMAXG && args.mode == 1) {
    // setup (src/sampler.cpp:591-620): state was initialised on the host
    // with an empty model; compute its factor, then sample
    compute_log_likelihood(C);
    commit(C);
    sample_beta_sigma2(C);
    refresh_tau2(C);
  } else {
    run_iterations(C, CS, g, end, args.capacity);
  }
  store_chain(C, CS);
  return g;
}

// A workgroup runs its chain to the end of the segment.  The kernel holds two
// codes, one with the factor in LDS for up to KMAX_LDS columns and the
// 256-column one with the factor in HBM, and a chain changes between them
// where its model's size asks for it without leaving its workgroup, so a
// launch lasts as long as its slowest chain.
#if BMG_UNIT(1)
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void k_chains(KernelArgs args) {
  __shared__ union {
    Smem<KMAX_LDS> small;
    Smem<BMG_KMAXG> large;
  } U;
  // (a workgroup has a compute unit to itself)
  static_assert(sizeof(U) <= 160 * 1024, "a workgroup has 160 KB of LDS");
  const int c = blockIdx.x;
  if (c >= args.n_chains) return;
  const ChainScal& CS = args.scal[c];
  if (args.mode == 0 && CS.rb_pending) return;   // the RB block must run first
  Progress g{CS.n_iter, 0, 0};
  const uint64_t end = g.iter + args.n_iter;
  int large = args.mode == 0 && (args.capacity == BMG_KMAXG || CS.cols + CAP_BACK > args.capacity);
  for (;;) {
    g = large ? run_capacity(U.large, args, g, end) : run_capacity(U.small, args, g, end);
    if (!g.change) break;
    large ^= 1;
  }
}
#endif

// ------------------------------------------------------- model op kernel --

template <int KMAX>
__device__ __forceinline__ void swapadj_w0(Smem<KMAX>& S, int m, int col) {
  if (threadIdx.x == 0) {
    // src/symmmatrix.cpp:220-265 on the packed factor and v
    for (int i = 0; i < col; ++i) {
      double t = S.L[P(col) + i]; S.L[P(col) + i] = S.L[P(col + 1) + i]; S.L[P(col + 1) + i] = t;
    }
    double a = S.L[P(col + 1) + col];   // old (col, col+1)
    double b = S.L[P(col + 1) + col + 1];
    double dcc = S.L[P(col) + col];
    S.L[P(col + 1) + col] = dcc;         // column col+1 gets old column col
    S.L[P(col + 1) + col + 1] = 0.0;
    double c, s;
    drotg(a, b, c, s);
    if (a < 0) { a = -a; s = -s; c = -c; }
    S.L[P(col) + col] = a;
    for (int i = col + 1; i < m; ++i) {
      double x1 = S.L[P(i) + col], x2 = S.L[P(i) + col + 1];
      double tmp = x1 * s - x2 * c;
      S.L[P(i) + col] = x2 * s + x1 * c;
      S.L[P(i) + col + 1] = tmp;
    }
    double x1 = S.v[col], x2 = S.v[col + 1];
    double tmp = x1 * s - x2 * c;
    S.v[col] = x2 * s + x1 * c;
    S.v[col + 1] = tmp;
  }
  __syncthreads();
}

#if BMG_UNIT(2)
__global__ __launch_bounds__(256) void k_model_op(ModelOpArgs a) {
  constexpr int KMAX = KMAX_LDS;
  __shared__ Smem<KMAX> S;
  ChainScal& CS = a.scal[0];
  load_descriptions(S, a.data, a.consts, a.arrays);
  Reg R;
  Ctx<KMAX> C{S, R, S.D, S.K, S.A, S.prof};
  load_chain(C, CS);
  R.err &= ~ERR_CAPACITY;   // a capacity error belongs to the call that hit it
  if (a.op == 0) {
    double d2[2] = {a.d0, a.d1};
    add_term(C, a.ind, a.t_ind, d2);
  } else if (a.op == 1) {
    remove_term(C, a.model_ind);
  } else if (a.op == 2) {
    compute_log_likelihood(C);
  } else if (a.op == 3) {
    swapadj_w0(S, R.cols, a.model_ind);
    R.lmin = a.model_ind;
  } else if (a.op == 4) {
    sample_beta_sigma2(C);   // from the model's own stream
  } else if (a.op == 5) {
    double pv[3];
    compute_pve(C, pv, 1);   // leaves y_hat = X beta
    if (threadIdx.x == 0) { CS.pves[0] = pv[0]; CS.pves[1] = pv[1]; CS.pves[2] = pv[2]; }
  }
  R.lmin = 0;
  commit(C);
  store_chain(C, CS);
  if (threadIdx.x == 0) {
    a.out->ll = R.c_ll;
    a.out->cols = R.c_cols; a.out->nloci = R.c_nloci; a.out->err = R.err;
    if (a.op == 5)
      for (int q = 0; q < 3; ++q) a.out->pves[q] = CS.pves[q];
  }
}
#endif
