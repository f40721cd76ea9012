// Data-flow path loop: one persistent kernel simulates the path nodes, every
// node as soon as its neighbours hold values, without FFTs (gfx950).
//
// Schedule. Workgroups take tickets by (dependency level, path index); a
// ticket is one of G slices (parts of the TI's valid positions) of a node. A
// node's neighbours are of lower levels, so their tickets were taken before and
// run on resident workgroups: waiting for their values in the simulation grid (a
// bounded poll of device-scope atomics) always ends, and there are neither
// launches nor barriers between dependent nodes. The grid cell itself is the
// message: a 32-bit word per variable, kPending until the node is written, so
// nothing else has to be ordered with it. The last slice of a node polls the
// other slices' K best (64-bit words, all-ones until written), merges, draws
// and writes. Levels rather than path indices: the nodes that others wait for
// come first (151 ms against 182 for 220 x 220 nodes of a 1000 x 1000 image).
//
// Scan (k_flow_direct). With x_j the neighbours' values and w_j >= 0 their
// weights, the map is, up to a constant of the node,
//     E(p) = -sum_j w_j (x_j - y(p + d_j))^2 - sum_j w_j [class differs],
// so a partial sum of the cost -E bounds it from below. A wavefront sums two
// tiles of 16 x 4 positions (2 per lane) over the neighbours, most unusual
// values first, eight at a time, and drops them together once every partial
// sum is above the bound: the K-th smallest cost known so far, seeded by the
// positions the neighbours themselves were copied from. Positions within the
// bound plus the FP32 error of both sums are kept, and the K best of them are
// decided in FP64 by the same sum, in the same order, as everywhere else in
// the library (exact_value in qsmi_band.hip), so the selected positions are
// those of the exact selection.
//   Bound by issue: a pair is a 4-byte load, two (weights of 1) to four vector
//   and about one scalar instruction; on the 1000 x 1000 log-normal image with n
//   = 80 the vector, the scalar and the load unit are each busy for 0.6 of the
//   time (loads alone: 34 TB/s of L1 on 256 CUs, 8.5 T pairs/s). A node needs
//   17-30 % of its 80 M pairs there and half of them in white noise, where waves
//   of transforms are the faster ones: run_flow leaves such paths to them.
//
// Scan (k_flow_count). Categorical variables under one kernel weight: E is
// the weight times the number of agreeing neighbours. The TI is held as one
// bit plane per class; a lane adds the n shifted 32-bit words of 32 positions
// into bit-sliced counters (carry-save adders of two v_bitop3_b32 each), about
// 3 instructions a neighbour for 32 positions where the FFT route needs ~8000
// a position block, and compares them with the K-th count known so far.
//   Bound by L1 bandwidth: 16 bytes a load feed three words of 32 positions
//   (8-byte loads, one word each, run at half the rate: 83 ms against 44 for
//   the 24 x 24 x 12 part of a 180 x 150 x 120 image).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "qsmi_internal.hpp"
#include "qsmi_flow.hpp"
#include "qsmi_select.hpp"

namespace qsmi {

namespace {

constexpr uint32_t kPending = 0xFFFFFFFFu;  // grid word of a variable not simulated yet
constexpr uint32_t kEmpty = 0x7FC00000u;    // simulated, but no position was valid
constexpr uint32_t kNone = 0xFFFFFFFFu;
constexpr uint32_t kNoTicket = 0x40000000u;  // above every ticket of a launch (nodes x slices)
// The word that says so stands in a cache line of its own: waits look at it, and
// beside the ticket, which every block adds to, that look slowed the tickets
// (500 x 500, a continuous and a 4-class variable, 60 x 60 nodes: 30 -> 20 ms).
constexpr int kGaveUp = 64, kCtlWords = 128;
constexpr unsigned long long kOpen = ~0ull;  // slice result not written yet
constexpr int kThreads = 256, kWaves = kThreads / 64;
// A wavefront sums kPair tiles of kTileX x kTileY positions side by side; the
// units run down the box in strips, so that the rows a unit reads stay in L1
// for the units below it. Every G-th run of kRun units belongs to a slice (the
// cost of a position varies over the TI; handing the runs out from a counter
// evens the slices, but device-scope atomics cost more than that gains: 199 ms
// against 170 ms on a 1000 x 1000 image with 16 slices).
constexpr int kTileX = 16, kTileY = 4, kPair = 2, kRun = 16;
constexpr int kStep = 8;        // terms between two looks at the bound
constexpr int kWaveList = 256;  // kept positions of a wavefront before they are scored
constexpr int kFlowStats = 7;
constexpr int kSources = 32;    // neighbours whose source positions seed the bound

struct FlowParams {
  int D, nVar, nExp, n, K, G, circSim;
  float kf;
  int sd[3], s[3];
  int types[8], e0[8], nCat[8], cat0[8];  // first expanded index, classes, first class value of a variable
  int expVar[16], expCat[16];
  int kdK[8][3];
  long long kerOff[8];
  float rare[kFlowMaxCat];  // per class: 1 - its share of the TI
  const float* quant;       // [nVar][kFlowQuant] quantiles of the continuous variables, ascending
  int S;
  const int* order;  // path nodes by (dependency level, path index)
  const unsigned* cells;
  const float* seeds;
  const int* nbIdx;
  const int* nbCnt;
  const int* offs;
  const float* kern;
  const float* catvals;
  const float* pathK;
  const int* nodeKer;
  const float* planes;  // [nVar][S]: values (continuous), class numbers (categorical)
  const uint32_t* bits;  // count form: [classes + 1][rows][W0], the last plane zero
  int W0, planeWords, zeroPlane;
  const float* tiVals;
  const float* di;    // the grid as given
  uint32_t* work;     // the grid under simulation
  uint32_t* index;
  int* ctl;           // [0] ticket (kNoTicket and above: none left), [kGaveUp] a wait was given up
  int polls;          // polls after which a wait is given up
  unsigned long long* slots;
  unsigned long long* stats;  // [kFlowStats]: nodes, positions scored, 0, flushes; tiles, their steps, without the bound
  int node0, nNodes;
};

// The kernel's parameters, read from the kernel argument segment anew for
// every node (args() hides where they come from): held across the loop they
// would fill the scalar registers and spill into vector registers.
typedef const __attribute__((address_space(4))) FlowParams FlowArgs;
__device__ __forceinline__ FlowArgs* args() {
  FlowArgs* p = (FlowArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return p;
}

__device__ __forceinline__ uint32_t ld_agent(const uint32_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent(uint32_t* p, uint32_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long ld_agent64(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent64(unsigned long long* p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Bounded wait step: false when the wait is given up. Then every other wait of
// the kernel ends as well, and the next node that is written ends the tickets
// (end_tickets): what the other nodes would be simulated from is not valid.
__device__ __forceinline__ bool poll_again(int& polls, int bound, int* err) {
  if (++polls >= bound) {
    st_agent((uint32_t*)err, 1u);
    return false;
  }
  if ((polls & 63) == 0 && ld_agent((const uint32_t*)err)) return false;
  __builtin_amdgcn_s_sleep(2);
  return true;
}

__device__ __forceinline__ uint32_t wait_word(const uint32_t* p, int bound, int* err) {
  uint32_t b = ld_agent(p);
  for (int polls = 0; b == kPending;) {
    if (!poll_again(polls, bound, err)) return kEmpty;
    b = ld_agent(p);
  }
  return b;
}

__device__ __forceinline__ unsigned long long wait_word64(const unsigned long long* p, int bound, int* err) {
  unsigned long long b = ld_agent64(p);
  for (int polls = 0; b == kOpen;) {
    if (!poll_again(polls, bound, err)) return kOpen;
    b = ld_agent64(p);
  }
  return b;
}

__device__ __forceinline__ uint32_t seed_bits_of(float seed) {
  if (!isfinite(seed) || seed <= 0.f) return 0u;
  if (seed >= 1.f) return 0xFFFFFFFFu;
  return (uint32_t)floor((double)seed * 4294967295.0);
}

__device__ __forceinline__ int take_ticket(int* ctl) {
  return __hip_atomic_fetch_add(&ctl[0], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Block-shared state of the current node.
struct FlowShared {
  int tick;
  int box[kWaves][6];
  int src[kSources][3];  // source positions of the nearest neighbours, moved back by their offsets
  uint32_t srcPos[kSources];
  float srcCost[kSources];
  float f[kWaves];
  int m[kWaves];
  float thr;
  uint32_t bound;  // smallest K-th cost a wavefront of the block knows
  int unit;        // units handed out
  int flushed;     // a wavefront has scored positions before the end
  uint32_t few[16];  // the positions left at the end of a slice, and their values
  double fewVal[16];
  float delta0;
  uint32_t pos[kMaxK];
};

// The node's neighbours, in list order (dynamic LDS).
struct FlowNb {
  int* d0;   // [n] offset along dimension 0
  int* row;  // [n] d1 + s1 d2
  float* x;  // [n][nVar] value; class number of a categorical variable
  float* w;  // [n][nVar] weight, 0: no value
  float* dt;  // [nVar][n] delta0 terms (direct form)
};

// Writes TI position p (kNone: none was valid) into the cell's missing
// variables, which releases the nodes that wait for them, and into the index
// image (include/simulation.hpp:658-666). Thread 0 of the node's last slice.
__device__ void write_cell(FlowArgs& P, unsigned cell, uint32_t p) {
  const long long c = (long long)cell * P.nVar;
  if (p != kNone) st_agent(&P.index[cell], p);
  for (int v = 0; v < P.nVar; ++v) {
    if (!isnan(P.di[c + v])) continue;  // a given value is kept
    st_agent(&P.work[c + v], p == kNone ? kEmpty : __float_as_uint(P.tiVals[(long long)p * P.nVar + v]));
  }
}

// No block takes another ticket once a wait has been given up. Looked at once a
// node, by the thread that has written it: with every ticket that look cost up
// to half of the loop's rate.
__device__ __forceinline__ void end_tickets(FlowArgs& P) {
  if (ld_agent((const uint32_t*)&P.ctl[kGaveUp])) st_agent((uint32_t*)&P.ctl[0], kNoTicket);
}

// The rank draw over the K best (best first), as draw_write of qsmi_select.hpp.
__device__ uint32_t draw_rank(FlowArgs& P, int i, float seed, const uint32_t* pos) {
  const float kl = P.pathK ? P.pathK[i] : 0.f;
  const float kk = kl > 0.f ? kl : P.kf;
  int r = (int)floorf(seed * kk * (ceilf(1.f / kk) / 1.f));
  if (r > (int)ceilf(kk) - 1) r = (int)ceilf(kk) - 1;
  if (r > P.K - 1) r = P.K - 1;
  if (r < 0) r = 0;
  return pos[r];
}

// NV: at least the number of variables.
// Reads the node's neighbours (waiting for their values) into LDS, and their
// bounding box -> lo / n of the valid box. Every thread of the block calls
// it; ends with a barrier. delta0 terms: the reference reads the expanded
// value at the original variable's index (include/
// quantileSamplingModule.hpp:368-457).
template <bool DIRECT, int NV>
__device__ __forceinline__ void gather_node(FlowArgs& P, int i, unsigned cell, int cnt, const FlowNb& nb,
                                            FlowShared* sh, int (&lo)[3], int (&n)[3]) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int cc[3] = {0, 0, 0};
  {
    unsigned rem = cell;
    for (int d = 0; d < P.D; ++d) {
      cc[d] = (int)(rem % (unsigned)P.sd[d]);
      rem /= (unsigned)P.sd[d];
    }
  }
  const int kk = P.nodeKer ? P.nodeKer[i] : 0;
  const float* __restrict__ kn = P.kern + P.kerOff[kk];
  const int kd0 = P.kdK[kk][0], kd1 = P.kdK[kk][1], kd2 = P.kdK[kk][2];
  int mn[3] = {0, 0, 0}, mx[3] = {0, 0, 0};
  for (int j = tid; j < cnt; j += kThreads) {
    const int* dp = P.offs + (long long)P.nbIdx[(long long)i * P.n + j] * P.D;
    const int dd[3] = {dp[0], P.D > 1 ? dp[1] : 0, P.D > 2 ? dp[2] : 0};
    int x[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      mn[d] = min(mn[d], dd[d]);
      mx[d] = max(mx[d], dd[d]);
      x[d] = cc[d] + dd[d];
      if (P.circSim) x[d] = ((x[d] % P.sd[d]) + P.sd[d]) % P.sd[d];
    }
    const unsigned t = (unsigned)x[0] + (unsigned)P.sd[0] * ((unsigned)x[1] + (unsigned)P.sd[1] * (unsigned)x[2]);
    const int k0 = kd0 / 2 + dd[0], k1 = kd1 / 2 + dd[1], k2 = kd2 / 2 + dd[2];
    const bool inK = k0 >= 0 && k0 < kd0 && k1 >= 0 && k1 < kd1 && k2 >= 0 && k2 < kd2;
    const float* kw = kn + ((long long)(inK ? k2 : 0) * kd1 + (inK ? k1 : 0)) * (long long)kd0 * P.nExp +
                      (long long)(inK ? k0 : 0) * P.nExp;
    nb.d0[j] = dd[0];
    nb.row[j] = dd[1] + P.s[1] * dd[2];
    const uint32_t* wp = P.work + (long long)t * P.nVar;
    uint32_t bits[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v)
      if (v < P.nVar) bits[v] = ld_agent(&wp[v]);
    // the position the neighbour was copied from, moved back by its offset
    // (hard data and stale entries give 0: any position may seed the bound)
    unsigned sp = ld_agent(&P.index[t]);
    bool waited = false;
    float val[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      if (v >= P.nVar) continue;
      uint32_t b = bits[v];
      if (b == kPending && t != cell) {
        b = wait_word(&wp[v], P.polls, &P.ctl[kGaveUp]);
        waited = true;
      }
      val[v] = (b == kPending || b == kEmpty) ? NAN : __uint_as_float(b);
    }
    if (j >= 1 && j <= kSources) {
      if (waited) sp = ld_agent(&P.index[t]);
      sh->src[j - 1][0] = (int)(sp % (unsigned)P.s[0]) - dd[0];
      sh->src[j - 1][1] = (int)((sp / (unsigned)P.s[0]) % (unsigned)P.s[1]) - dd[1];
      sh->src[j - 1][2] = (int)(sp / ((unsigned)P.s[0] * (unsigned)P.s[1])) - dd[2];
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      if (v >= P.nVar) continue;
      float xv = val[v];
      float w = (inK && !isnan(xv)) ? kw[P.e0[v]] : 0.f;
      if (P.types[v] != 0) {
        int code = -1;
        for (int q = 0; q < P.nCat[v]; ++q)
          if (P.catvals[P.cat0[v] + q] == xv) code = q;
        if (code < 0) w = 0.f;  // agrees with no TI cell
        xv = (float)code;
      }
      nb.x[j * P.nVar + v] = w != 0.f ? xv : 0.f;
      nb.w[j * P.nVar + v] = w;
      if (DIRECT) {
        float tv = 0.f;
        if (P.types[v] == 0) {
          float xe = 0.f;
#pragma unroll
          for (int q = 0; q < NV; ++q)
            if (q == P.expVar[v]) xe = val[q];
          if (P.expCat[v] >= 0) xe = (xe == P.catvals[P.expCat[v]]) ? 1.f : 0.f;
          if (inK && !isnan(xe)) tv = -1.f * (kw[v % P.nExp] * xe * xe);
        }
        nb.dt[v * P.n + j] = tv;
      }
    }
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      mn[d] = min(mn[d], __shfl_xor(mn[d], off));
      mx[d] = max(mx[d], __shfl_xor(mx[d], off));
    }
  }
  if (lane == 0) {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      sh->box[wave][d] = mn[d];
      sh->box[wave][3 + d] = mx[d];
    }
  }
  __syncthreads();
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    int a = 0, b = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      a = min(a, sh->box[w][d]);
      b = max(b, sh->box[w][3 + d]);
    }
    lo[d] = __builtin_amdgcn_readfirstlane(-a);
    n[d] = __builtin_amdgcn_readfirstlane(max(0, P.s[d] - b + a));
  }
}

// Source position m of the node's nearest neighbours as a TI position, or
// kNone when it is not valid or an earlier neighbour gives the same. cntS:
// source positions read. One thread per m; the block synchronises around it.
__device__ __forceinline__ uint32_t source_pos(FlowArgs& P, const FlowShared* sh, int m, int cntS,
                                               const int (&lo)[3], const int (&n)[3]) {
  if (m >= cntS) return kNone;
  const int c0 = sh->src[m][0], c1 = sh->src[m][1], c2 = sh->src[m][2];
  if (c0 < lo[0] || c0 >= lo[0] + n[0] || c1 < lo[1] || c1 >= lo[1] + n[1] || c2 < lo[2] || c2 >= lo[2] + n[2])
    return kNone;
  for (int q = 0; q < m; ++q)
    if (sh->src[q][0] == c0 && sh->src[q][1] == c1 && sh->src[q][2] == c2) return kNone;
  return (uint32_t)(c0 + P.s[0] * (c1 + P.s[1] * c2));
}

// ---------------------------------------------------------------------------
// Direct form
// ---------------------------------------------------------------------------

// Exact value of position p (the sum and order of exact_value in
// qsmi_band.hip), one position per lane.
template <int NV>
__device__ double exact_lane(FlowArgs& P, const FlowNb& nb, int cnt, double delta0, uint32_t p) {
  double acc = delta0;
  const int s0 = P.s[0];
#pragma unroll 4
  for (int j = 0; j < cnt; ++j) {
    const int t = (int)p + nb.d0[j] + s0 * nb.row[j];
    for (int v = 0; v < (NV == 1 ? 1 : P.nVar); ++v) {
      const int jv = NV == 1 ? j : j * P.nVar + v;
      const float w = nb.w[jv], x = nb.x[jv];
      if (w == 0.f) continue;  // block-uniform; adds nothing
      const float y = P.planes[(long long)v * P.S + t];
      if (NV == 1 || P.types[v] == 0) {
        acc = __dadd_rn(acc, __dmul_rn((double)(-w), (double)__fmul_rn(y, y)));
        acc = __dadd_rn(acc, __dmul_rn((double)(2.f * __fmul_rn(w, x)), (double)y));
      } else {
        acc = __dadd_rn(acc, y == x ? (double)w : 0.0);
      }
    }
  }
  return acc;
}

__device__ __forceinline__ double readlane64(double v, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                          __builtin_amdgcn_readlane(__double2loint(v), l));
}

// The same value by a whole wavefront (at most two variables): the products
// of 64 neighbours at a time, then the sum in list order. Few kept positions
// are the rule, and a lane alone would wait for every neighbour's load.
template <int NV>
__device__ double exact_wave(FlowArgs& P, const FlowNb& nb, int cnt, double delta0, uint32_t p, int lane) {
  double acc = delta0;
  constexpr int NW = NV == 1 ? 1 : 2;
  const int s0 = P.s[0], nVar = NV == 1 ? 1 : P.nVar;
  for (int j0 = 0; j0 < cnt; j0 += 64) {
    double a[NW], b[NW];
#pragma unroll
    for (int v = 0; v < NW; ++v) a[v] = b[v] = 0.0;
    const int j = j0 + lane;
    if (j < cnt) {
      const int t = (int)p + nb.d0[j] + s0 * nb.row[j];
#pragma unroll
      for (int v = 0; v < NW; ++v) {
        if (v >= nVar) continue;
        const float w = nb.w[j * nVar + v], x = nb.x[j * nVar + v];
        if (w == 0.f) continue;
        const float y = P.planes[(long long)v * P.S + t];
        if (NV == 1 || P.types[v] == 0) {
          a[v] = __dmul_rn((double)(-w), (double)__fmul_rn(y, y));
          b[v] = __dmul_rn((double)(2.f * __fmul_rn(w, x)), (double)y);
        } else {
          a[v] = y == x ? (double)w : 0.0;
        }
      }
    }
    const int m = min(64, cnt - j0);
    for (int q = 0; q < m; ++q)
#pragma unroll
      for (int v = 0; v < NW; ++v)
        if (v < nVar) acc = __dadd_rn(__dadd_rn(acc, readlane64(a[v], q)), readlane64(b[v], q));
  }
  return acc;
}

// Largest FP32 cost a position of the K best can have when K positions cost
// at most c. With u = 2^-24, W = sum w x^2 and T terms, the FP32 cost and the
// exact value (whose squares, products and weights are rounded to FP32 first)
// differ by at most u (5 W + (T + 12) c); twice that, with a margin of a quarter,
// plus what a flushed denormal could lose.
__device__ __forceinline__ float cost_limit(float c, float W, int T) {
  return c + 1.25f * 1.1920929e-7f * (6.f * W + (float)(T + 12) * c) + 1e-34f;
}

template <int KT>
__device__ __forceinline__ float kth_of(const float (&b)[KT], int K) {
  float r = b[0];
#pragma unroll
  for (int k = 1; k < KT; ++k)
    if (k == K - 1) r = b[k];
  return r;
}

// Scores a wavefront's kept positions in FP64: those still within lim into
// the lanes' lists. Returns how many were scored.
template <int NV, int KT>
__device__ int score_list(FlowArgs& P, const FlowNb& nb, int cnt, double delta0, uint32_t seedbits,
                          const uint32_t* pos, const float* cost, int len, float lim, int lane, TopK64<KT>& tk) {
  int live = 0;
  for (int q0 = 0; q0 < len; q0 += 64) {
    const int q = q0 + lane;
    const bool ok = q < len && cost[q] <= lim;
    unsigned long long m = __ballot(ok);
    const int c = __popcll(m);
    live += c;
    if (c == 0) continue;
    const uint32_t mine = ok ? pos[q] : 0u;
    if (c <= 12 && NV <= 2) {
      while (m) {
        const int l = __ffsll((long long)m) - 1;
        m &= m - 1;
        const uint32_t p = __builtin_amdgcn_readlane(mine, l);
        Cand64 cd;
        cd.val = exact_wave<NV>(P, nb, cnt, delta0, p, lane);
        cd.pos = p;
        cd.h = tie_hash(seedbits, p);
        if (lane == l) tk.push(cd);
      }
    } else if (ok) {
      Cand64 cd;
      cd.val = exact_lane<NV>(P, nb, cnt, delta0, mine);
      cd.pos = mine;
      cd.h = tie_hash(seedbits, mine);
      tk.push(cd);
    }
  }
  return live;
}

// Half width of the smallest interval around x that holds kNearQuant of the
// variable's quantiles: the squared distance that most positions exceed, i.e.
// how much a neighbour of value x tells them apart.
constexpr int kNearQuant = kFlowQuant * 3 / 10;
__device__ __forceinline__ float near_radius(const float* q, float x) {
  int lo = 0, hi = kFlowQuant - kNearQuant;  // smallest L with x - q[L] <= q[L + kNearQuant - 1] - x
  while (lo < hi) {
    const int m = (lo + hi) >> 1;
    if (x - q[m] <= q[m + kNearQuant - 1] - x)
      hi = m;
    else
      lo = m + 1;
  }
  const int b = min(lo, kFlowQuant - kNearQuant);
  const float r1 = fmaxf(x - q[b], q[b + kNearQuant - 1] - x);
  if (b == 0) return r1;
  return fminf(r1, fmaxf(x - q[b - 1], q[b + kNearQuant - 2] - x));
}

// One step of the scan: kStep terms for the wavefront's kPair tiles, every
// load issued before the first sum. The addresses are a scalar base per term
// (tile and offset) and the lane's place in the tile, so that they cost no
// vector instruction: two (UNIT: weights of 1) to four a (position, term) pair.
template <bool MIXED, bool UNIT>
__device__ __forceinline__ void add_step(const char* tile, const int (&o)[kStep], const float (&x)[kStep],
                                         const float (&w)[kStep], const float (&c)[kStep], const uint32_t (&vo)[kPair],
                                         float (&acc)[kPair]) {
  uint32_t v[kPair];
#pragma unroll
  for (int r = 0; r < kPair; ++r) {
    v[r] = vo[r];
    asm volatile("" : "+v"(v[r]));  // keeps the 32-bit lane offset in the load's own block (scalar base addressing)
  }
  float y[kPair][kStep];
#pragma unroll
  for (int e = 0; e < kStep; ++e) {
    const char* b = tile + o[e];
#pragma unroll
    for (int r = 0; r < kPair; ++r) y[r][e] = *reinterpret_cast<const float*>(b + v[r]);
  }
#pragma unroll
  for (int e = 0; e < kStep; ++e)
#pragma unroll
    for (int r = 0; r < kPair; ++r) {
      const float d = y[r][e] - x[e];
      if (MIXED)
        acc[r] = fmaf(w[e], fminf(d * d, c[e]), acc[r]);
      else
        acc[r] = fmaf(UNIT ? d : w[e] * d, d, acc[r]);
    }
}

__device__ __forceinline__ float uniform(float v) {
  return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v)));
}

// FORM 0: continuous, every weight 1 or 0 (no value); 1: continuous; 2: with
// categorical variables. NV: 1 for one variable, else at least their number.
// COUNT: tiles and steps are counted (a scalar more in the tile loop, 1 % of the
// scan, so only the segments that are judged by them do).
// Wavefronts a SIMD: six where the tile loop fits 80 registers, five for the
// mixed form (two more registers spill into the loop: 543 -> 556 ms on 500 x 500
// with a continuous and a 4-class variable, 225,000 nodes).
template <int FORM, int NV, int KT, bool COUNT>
__global__ void __launch_bounds__(kThreads, KT <= 2 ? (NV == 1 ? 6 : 5) : 4) k_flow_direct(FlowParams kernArgs) {
  constexpr bool MIXED = FORM == 2;
  extern __shared__ __align__(16) char dyn[];
  __shared__ FlowShared sh;
  __shared__ uint32_t lPos[kWaves][kWaveList];
  __shared__ float lCost[kWaves][kWaveList];
  __shared__ Cand64 red[kWaves];
  __shared__ Cand64 best[kMaxK];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  FlowArgs& P0 = *args();
  const int nVar = NV == 1 ? 1 : P0.nVar;
  const int nv = P0.n * nVar, T8 = ((nv + 7) & ~7) + 8;
  // terms in scan order (16-byte aligned), then the neighbours in list order
  int* tOff = reinterpret_cast<int*>(dyn);
  float* tX = reinterpret_cast<float*>(tOff + T8);
  float* tW = tX + T8;
  float* tC = tW + T8;  // MIXED: 1 for a categorical term, infinity otherwise
  float* key = tC + T8;
  float* quant = key + T8;  // [nVar][kFlowQuant]
  FlowNb nb;
  nb.x = quant + nVar * kFlowQuant;
  nb.w = nb.x + nv;
  nb.dt = nb.w + nv;
  nb.d0 = reinterpret_cast<int*>(nb.dt + nv);
  nb.row = nb.d0 + P0.n;
  __builtin_amdgcn_s_setprio(3);
  for (int t = tid; t < nVar * kFlowQuant; t += kThreads) quant[t] = P0.quant[t];  // first read after a barrier
  unsigned long long nScored = 0, nNodesDone = 0, nFlush = 0;
  // tiles of the block's nodes, their steps without the bound, and the steps this wavefront took
  unsigned long long nTiles = 0, nFull = 0, nSteps = 0;
  for (;;) {
    FlowArgs& P = *args();
    const int s0 = P.s[0], s1 = P.s[1], K = P.K, G = P.G;
    __syncthreads();  // the previous node's shared state is read no more
    if (tid == 0) sh.tick = take_ticket(P.ctl);
    __syncthreads();
    const int tick = __builtin_amdgcn_readfirstlane(sh.tick);
    const int q = tick / G, slice = tick - q * G;
    if (q >= P.nNodes) break;
    const int i = P.order[P.node0 + q];
    const unsigned cell = P.cells[i];
    const float seed = P.seeds[i];
    const uint32_t seedbits = seed_bits_of(seed);
    const int cnt = P.nbCnt[i];
    if (cnt <= 1) {  // block-uniform
      bool given = false;
      if (cnt == 1)
        for (int v = 0; v < nVar; ++v) given |= !isnan(P.di[(long long)cell * nVar + v]);
      if (!given) {
        // no neighbour, no value: drawn from the marginal (include/simulation.hpp:586-606)
        if (slice == G - 1 && tid == 0) write_cell(P, cell, (uint32_t)(int)floorf(seed * (float)P.S));
        continue;
      }
    }
    int lo[3], n[3];
    gather_node<true, NV>(P, i, cell, cnt, nb, &sh, lo, n);
    // order of the terms: what most positions cost them, largest first
    const int T = cnt * nVar;
    float wx = 0.f;
    int nPos = 0;
    for (int t = tid; t < T; t += kThreads) {
      const int v = t % nVar;
      const float w = nb.w[t], x = nb.x[t];
      float kv = -1.f;
      if (w > 0.f) {
        ++nPos;
        if (P.types[v] == 0) {
          const float r = near_radius(quant + v * kFlowQuant, x);
          kv = w * (r * r);
          wx += w * x * x;
        } else {
          kv = w * fmaxf(0.f, 2.f * P.rare[P.cat0[v] + (int)x] - 1.f);
        }
      }
      key[t] = kv;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      wx += __shfl_xor(wx, off);
      nPos += __shfl_xor(nPos, off);
    }
    if (lane == 0) {
      sh.f[wave] = wx;
      sh.m[wave] = nPos;
    }
    // delta0 in the reference's order, by the last wavefront
    if (wave == kWaves - 1) {
      float d = 0.f;
      for (int v = 0; v < nVar; ++v) {
        if (P.types[v] != 0) continue;
        for (int j0 = 0; j0 < cnt; j0 += 64) {
          const int tb = __float_as_int(j0 + lane < cnt ? nb.dt[v * P.n + j0 + lane] : 0.f);
          const int m = min(64, cnt - j0);
          for (int u = 0; u < m; ++u) d += __int_as_float(__builtin_amdgcn_readlane(tb, u));
        }
      }
      if (lane == 0) sh.delta0 = d;
    }
    if (tid >= 64 && tid < 68) key[T + tid - 64] = -1.f;
    if (tid < kSources) sh.srcPos[tid] = source_pos(P, &sh, tid, min(cnt - 1, kSources), lo, n);
    __syncthreads();
    const float W = sh.f[0] + sh.f[1] + sh.f[2] + sh.f[3];
    const int Tn = __builtin_amdgcn_readfirstlane(sh.m[0] + sh.m[1] + sh.m[2] + sh.m[3]);
    for (int t = tid; t < T; t += kThreads) {
      const float kv = key[t];
      if (!(kv >= 0.f)) continue;
      int rank = 0;
      for (int u = 0; u < T; u += 4) {  // keys past T are -1
        const float4 k4 = *reinterpret_cast<const float4*>(&key[u]);
        rank += (k4.x > kv || (k4.x == kv && u < t)) ? 1 : 0;
        rank += (k4.y > kv || (k4.y == kv && u + 1 < t)) ? 1 : 0;
        rank += (k4.z > kv || (k4.z == kv && u + 2 < t)) ? 1 : 0;
        rank += (k4.w > kv || (k4.w == kv && u + 3 < t)) ? 1 : 0;
      }
      const int j = t / nVar, v = t - j * nVar;
      tOff[rank] = (v * P.S + nb.d0[j] + s0 * nb.row[j]) * 4;
      tX[rank] = nb.x[t];
      tW[rank] = nb.w[t];
      if (MIXED) tC[rank] = P.types[v] == 0 ? INFINITY : 1.f;
    }
    if (tid < kStep) {  // padding to whole steps
      tOff[Tn + tid] = 0;
      tX[Tn + tid] = 0.f;
      tW[Tn + tid] = 0.f;
      if (MIXED) tC[Tn + tid] = INFINITY;
    }
    __syncthreads();
    const char* pl = reinterpret_cast<const char*>(P.planes);
    // the K-th smallest cost of the source positions: eight lanes each
    {
      const int m = tid >> 3, sub = tid & 7;
      const uint32_t sp = sh.srcPos[m];
      float c = 0.f;
      if (sp != kNone) {
        const char* b = pl + (size_t)sp * 4;
#pragma unroll 4
        for (int t = sub; t < Tn; t += 8) {
          const float d = *reinterpret_cast<const float*>(b + tOff[t]) - tX[t];
          float d2 = d * d;
          if (MIXED) d2 = fminf(d2, tC[t]);
          c = fmaf(tW[t], d2, c);
        }
      }
#pragma unroll
      for (int off = 1; off < 8; off <<= 1) c += __shfl_xor(c, off);
      if (sub == 0) sh.srcCost[m] = sp != kNone ? c : INFINITY;
      if (tid == 0) {
        sh.thr = INFINITY;
        sh.bound = 0x7F800000u;
        sh.unit = 0;
        sh.flushed = 0;
      }
      __syncthreads();
      if (tid < kSources) {
        const float mine = sh.srcCost[tid];
        int rank = 0;
        for (int u = 0; u < kSources; ++u) rank += (sh.srcCost[u] < mine || (sh.srcCost[u] == mine && u < tid)) ? 1 : 0;
        if (rank == K - 1) sh.thr = mine;
      }
      __syncthreads();
    }
    const float thr0 = sh.thr;
    const double delta0 = (double)sh.delta0;
    const bool box = n[0] > 0 && n[1] > 0 && n[2] > 0;
    float bk[KT];
#pragma unroll
    for (int k = 0; k < KT; ++k) bk[k] = INFINITY;
    float thr = thr0;  // at least K positions cost no more
    float lim = cost_limit(thr, W, Tn);
    int len = 0;  // kept positions of this wavefront
    TopK64<KT> tk;
    tk.init();
    const int NX = (n[0] + kTileX * kPair - 1) / (kTileX * kPair), NY = (n[1] + kTileY - 1) / kTileY;
    const int units = box ? NX * NY * n[2] : 0;
    if (COUNT && slice == G - 1) {
      nTiles += (unsigned)units;
      nFull += (unsigned long long)units * ((unsigned)(Tn + kStep - 1) / kStep);
    }
    // a node's dependents wait for everything but the scan's share of the
    // other nodes: the scan yields to the short phases around it
    __builtin_amdgcn_s_setprio(0);
    if (slice * kRun < units) {
      const int lx = lane & (kTileX - 1), ly = lane / kTileX;
      const uint32_t laneVo = (uint32_t)(lx + s0 * ly) * 4u;
      // exact quotients by NY and n[2] for numerators below 2^32 / divisor
      const uint32_t mY = 0xFFFFFFFFu / (uint32_t)NY + 1u, mZ = 0xFFFFFFFFu / (uint32_t)n[2] + 1u;
      // the first step's terms in scalar registers
      const bool full = Tn >= kStep;
      int fo[kStep];
      float fx[kStep], fw[kStep], fc[kStep];
#pragma unroll
      for (int e = 0; e < kStep; ++e) {
        fo[e] = __builtin_amdgcn_readfirstlane(tOff[e]);
        fx[e] = uniform(tX[e]);
        fw[e] = FORM == 0 ? 1.f : uniform(tW[e]);
        fc[e] = MIXED ? uniform(tC[e]) : 0.f;
      }
      unsigned terms = 0;  // of this wavefront's units, in whole steps
      int k = 0;  // the slice's units, handed out to its wavefronts one by one
      if (lane == 0) k = atomicAdd(&sh.unit, 1);
      for (;;) {
        k = __builtin_amdgcn_readfirstlane(k);
        const int run = (k / kRun * G + slice) * kRun, u = run + k % kRun;
        if (run >= units) break;
        if (lane == 0) k = atomicAdd(&sh.unit, 1);
        if (u >= units) continue;
        const int uq = NY == 1 ? u : (int)__umulhi((uint32_t)u, mY), uy = u - uq * NY;
        const int ux = n[2] == 1 ? uq : (int)__umulhi((uint32_t)uq, mZ), uz = uq - ux * n[2];
        const int x0 = ux * kTileX * kPair, y0 = uy * kTileY;
        const int pu = lo[0] + x0 + s0 * (lo[1] + y0 + s1 * (lo[2] + uz));
        const char* tile = pl + (long long)pu * 4;
        uint32_t vo[kPair];
        float acc[kPair];
        if (x0 + kTileX * kPair <= n[0] && y0 + kTileY <= n[1]) {
#pragma unroll
          for (int r = 0; r < kPair; ++r) {
            vo[r] = laneVo + (uint32_t)(r * kTileX * 4);
            acc[r] = 0.f;
          }
        } else {  // lanes outside the box read its nearest position and never count
          const int ey = min(ly, n[1] - 1 - y0);
#pragma unroll
          for (int r = 0; r < kPair; ++r) {
            const int xr = lx + r * kTileX, ex = min(xr, n[0] - 1 - x0);
            vo[r] = (uint32_t)(ex + s0 * ey) * 4u;
            acc[r] = (ex == xr && ey == ly) ? 0.f : INFINITY;
          }
        }
        if (FORM != 0 || full) {
          add_step<MIXED, FORM == 0>(tile, fo, fx, fw, fc, vo, acc);
        } else {  // the padding of a lone step has weight 0
          float w[kStep];
#pragma unroll
          for (int e = 0; e < kStep; ++e) w[e] = tW[e];
          add_step<false, false>(tile, fo, fx, w, fc, vo, acc);
        }
        // wave-uniform: a position can still be within the limit
        bool on = __any(fminf(acc[0], acc[1]) <= lim);
        int t = kStep;
        for (; t < Tn && on; t += kStep) {
          int o[kStep];
          float x[kStep], w[kStep], c[kStep];
#pragma unroll
          for (int e = 0; e < kStep; ++e) {
            o[e] = __builtin_amdgcn_readfirstlane(tOff[t + e]);
            x[e] = tX[t + e];
            w[e] = FORM == 0 ? 1.f : tW[t + e];
            c[e] = MIXED ? tC[t + e] : 0.f;
          }
          if (FORM != 0 || t + kStep <= Tn) {
            add_step<MIXED, FORM == 0>(tile, o, x, w, c, vo, acc);
          } else {
#pragma unroll
            for (int e = 0; e < kStep; ++e) w[e] = tW[t + e];
            add_step<false, false>(tile, o, x, w, c, vo, acc);
          }
          on = __any(fminf(acc[0], acc[1]) <= lim);
        }
        if (COUNT) terms += (unsigned)t;
        if (!on) continue;
#pragma unroll
        for (int r = 0; r < kPair; ++r) {
          const bool hit = acc[r] <= lim && acc[r] < INFINITY;
          unsigned long long m = __ballot(hit);
          if (hit) {
            const int e = len + __popcll(m & ((1ull << lane) - 1ull));
            lPos[wave][e] = (uint32_t)pu + (vo[r] >> 2);
            lCost[wave][e] = acc[r];
          }
          len += __popcll(m);
          bool better = false;
          while (m) {
            const int l = __ffsll((long long)m) - 1;
            m &= m - 1;
            float cst = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(acc[r]), l));
            if (!(cst < kth_of<KT>(bk, K))) continue;
            better = true;
#pragma unroll
            for (int k = 0; k < KT; ++k)
              if (cst < bk[k]) {
                const float o = bk[k];
                bk[k] = cst;
                cst = o;
              }
          }
          if (better) {
            const float kth = kth_of<KT>(bk, K);
            if (kth < thr) {
              thr = kth;
              lim = cost_limit(thr, W, Tn);
              if (lane == 0) atomicMin(&sh.bound, __float_as_uint(kth));  // costs are >= 0: ordered as integers
            }
          }
        }
        if (len > kWaveList - 64 * kPair) {  // wave-uniform: score what is kept so far
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          nScored += score_list<NV, KT>(P, nb, cnt, delta0, seedbits, lPos[wave], lCost[wave], len, lim, lane, tk);
          ++nFlush;
          sh.flushed = 1;
          len = 0;
        }
        // what the other wavefronts of the block know
        const float known = __uint_as_float(__builtin_amdgcn_readfirstlane(*(volatile uint32_t*)&sh.bound));
        if (known < thr) {
          thr = known;
          lim = cost_limit(thr, W, Tn);
        }
      }
      if (COUNT) nSteps += terms / kStep;
    }
    __builtin_amdgcn_s_setprio(3);
    // the slice's bound: every wavefront's K-th cost holds for all
    if (lane == 0) sh.f[wave] = thr;
    __syncthreads();
    lim = cost_limit(fminf(fminf(sh.f[0], sh.f[1]), fminf(sh.f[2], sh.f[3])), W, Tn);
    // few positions are left as a rule: into one list, scored by all wavefronts
    int kept = 0;
    for (int e = lane; e < len; e += 64) kept += lCost[wave][e] <= lim ? 1 : 0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) kept += __shfl_xor(kept, off);
    if (lane == 0) sh.m[wave] = kept;
    __syncthreads();
    const int total = __builtin_amdgcn_readfirstlane(sh.m[0] + sh.m[1] + sh.m[2] + sh.m[3]);
    const bool flushed = __builtin_amdgcn_readfirstlane(sh.flushed) != 0;
    if (total <= 16 && !flushed && NV <= 2) {  // block-uniform
      int at = 0;
      for (int w = 0; w < wave; ++w) at += sh.m[w];
      for (int e0 = 0; e0 < len; e0 += 64) {
        const int e = e0 + lane;
        const bool ok = e < len && lCost[wave][e] <= lim;
        const unsigned long long m = __ballot(ok);
        if (ok) sh.few[at + __popcll(m & ((1ull << lane) - 1ull))] = lPos[wave][e];
        at += __popcll(m);
      }
      __syncthreads();
      for (int e = wave; e < total; e += kWaves) {
        const double v = exact_wave<NV>(P, nb, cnt, delta0, __builtin_amdgcn_readfirstlane(sh.few[e]), lane);
        if (lane == 0) sh.fewVal[e] = v;
      }
      nScored += wave == 0 ? total : 0;
      __syncthreads();
      if (tid < 64) {  // rank of each among all
        Cand64 c = worst_cand64();
        if (lane < total) {
          c.val = sh.fewVal[lane];
          c.pos = sh.few[lane];
          c.h = tie_hash(seedbits, c.pos);
        }
        int rank = 0;
        for (int e = 0; e < total; ++e) {
          Cand64 o;
          o.val = readlane64(c.val, e);
          o.h = (uint32_t)__builtin_amdgcn_readlane((int)c.h, e);
          o.pos = (uint32_t)__builtin_amdgcn_readlane((int)c.pos, e);
          rank += cand64_better(o, c) ? 1 : 0;
        }
        if (lane < total) {
          if (rank < K) best[rank] = c;
        } else if (lane < K) {
          best[lane] = c;
        }
      }
      __syncthreads();
    } else {
      nScored += score_list<NV, KT>(P, nb, cnt, delta0, seedbits, lPos[wave], lCost[wave], len, lim, lane, tk);
      block_topk64<KT>(tk, K, best, red);
    }
    if (G > 1) {
      unsigned long long* sl = P.slots + (long long)q * (G - 1) * K * 2;
      if (slice < G - 1) {
        if (tid < K) {
          st_agent64(&sl[((long long)slice * K + tid) * 2 + 1], (unsigned long long)best[tid].pos);
          st_agent64(&sl[((long long)slice * K + tid) * 2], (unsigned long long)__double_as_longlong(best[tid].val));
        }
        continue;
      }
      tk.init();
      if (tid < K) tk.push(best[tid]);
      for (int e = tid; e < (G - 1) * K; e += kThreads) {
        Cand64 c;
        c.pos = (uint32_t)wait_word64(&sl[(long long)e * 2 + 1], P.polls, &P.ctl[kGaveUp]);
        c.val = __longlong_as_double((long long)wait_word64(&sl[(long long)e * 2], P.polls, &P.ctl[kGaveUp]));
        c.h = tie_hash(seedbits, c.pos);
        if (c.pos != kNone) tk.push(c);
      }
      __syncthreads();  // best[] has been read
      block_topk64<KT>(tk, K, best, red);
    }
    if (tid < K) sh.pos[tid] = best[tid].pos;
    __syncthreads();
    if (tid == 0) {
      write_cell(P, cell, draw_rank(P, i, seed, sh.pos));
      end_tickets(P);
    }
    ++nNodesDone;
  }
  if (lane == 0 && nScored) atomicAdd(&P0.stats[1], nScored);
  if (lane == 0 && nFlush) atomicAdd(&P0.stats[3], nFlush);
  if (tid == 0 && nNodesDone) atomicAdd(&P0.stats[0], nNodesDone);
  if (COUNT && lane == 0 && nSteps) atomicAdd(&P0.stats[5], nSteps);
  if (COUNT && tid == 0 && nTiles) {
    atomicAdd(&P0.stats[4], nTiles);
    atomicAdd(&P0.stats[6], nFull);
  }
}

// ---------------------------------------------------------------------------
// Count form
// ---------------------------------------------------------------------------
constexpr int kWords = 3;

__device__ __forceinline__ void csa(uint32_t& h, uint32_t& l, uint32_t a, uint32_t b, uint32_t c) {
  h = __builtin_amdgcn_bitop3_b32(a, b, c, 0xE8);  // majority
  l = __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);  // parity
}

struct BitTerms {
  int* off;  // word offset of the plane, the row and the word of the box's first position (bytes)
  int* sh;   // bit of the box's first position in that word
};

// Number of agreeing neighbours at the box position (c0, row address rb).
__device__ __forceinline__ int count_at(const char* bits, const BitTerms& bt, int T, int c0, uint32_t rb, int t0,
                                        int step) {
  int c = 0;
#pragma unroll 4
  for (int t = t0; t < T; t += step) {
    const int b = c0 + bt.sh[t];
    const uint32_t w = *reinterpret_cast<const uint32_t*>(bits + bt.off[t] + rb + (uint32_t)(b >> 5) * 4u);
    c += (w >> (b & 31)) & 1u;
  }
  return c;
}

template <int NP, int NV, int KT>
__global__ void __launch_bounds__(kThreads) k_flow_count(FlowParams kernArgs) {
  extern __shared__ __align__(16) char dyn[];
  __shared__ FlowShared sh;
  __shared__ int sNt;
  __shared__ unsigned long long red[kWaves];
  __shared__ unsigned long long bestR[kMaxK];
  __shared__ uint32_t redP[kWaves];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  FlowArgs& P0 = *args();
  const int nVar = NV == 1 ? 1 : P0.nVar;
  const int nv = P0.n * nVar, T8 = ((nv + 7) & ~7) + 8;
  BitTerms bt;
  bt.off = reinterpret_cast<int*>(dyn);
  bt.sh = bt.off + T8;
  FlowNb nb;
  nb.x = reinterpret_cast<float*>(bt.sh + T8);
  nb.w = nb.x + nv;
  nb.dt = nullptr;
  nb.d0 = reinterpret_cast<int*>(nb.w + nv);
  nb.row = nb.d0 + P0.n;
  for (;;) {
    FlowArgs& P = *args();
    const int s0 = P.s[0], s1 = P.s[1], K = P.K, G = P.G, W0 = P.W0;
    const char* bits = reinterpret_cast<const char*>(P.bits);
    __syncthreads();  // the previous node's shared state is read no more
    if (tid == 0) {
      sh.tick = take_ticket(P.ctl);
      sNt = 0;
    }
    __syncthreads();
    const int tick = __builtin_amdgcn_readfirstlane(sh.tick);
    const int q = tick / G, slice = tick - q * G;
    if (q >= P.nNodes) break;
    const int i = P.order[P.node0 + q];
    const unsigned cell = P.cells[i];
    const float seed = P.seeds[i];
    const uint32_t seedbits = seed_bits_of(seed);
    const int cnt = P.nbCnt[i];
    if (cnt <= 1) {  // block-uniform
      bool given = false;
      if (cnt == 1)
        for (int v = 0; v < nVar; ++v) given |= !isnan(P.di[(long long)cell * nVar + v]);
      if (!given) {
        // no neighbour, no value: drawn from the marginal (include/simulation.hpp:586-606)
        if (slice == G - 1 && tid == 0) write_cell(P, cell, (uint32_t)(int)floorf(seed * (float)P.S));
        continue;
      }
    }
    int lo[3], n[3];
    gather_node<false, NV>(P, i, cell, cnt, nb, &sh, lo, n);
    // terms: neighbours that hold a class (their order does not matter)
    for (int t = tid; t < cnt * nVar; t += kThreads) {
      if (nb.w[t] == 0.f) continue;
      const int j = t / nVar, v = t - j * nVar;
      const int e = atomicAdd(&sNt, 1);
      const int b = lo[0] + nb.d0[j];  // >= 0 whenever the box holds a position
      bt.off[e] = ((P.cat0[v] + (int)nb.x[t]) * P.planeWords + nb.row[j] * W0 + (b >> 5)) * 4;
      bt.sh[e] = b & 31;
    }
    if (tid < kSources) sh.srcPos[tid] = source_pos(P, &sh, tid, min(cnt - 1, kSources), lo, n);
    __syncthreads();
    const int T = __builtin_amdgcn_readfirstlane(sNt);
    if (tid < 8) {  // padding to whole rounds of eight terms: the zero plane
      bt.off[T + tid] = P.zeroPlane * P.planeWords * 4;
      bt.sh[T + tid] = 0;
    }
    const int Nv = n[0] > 0 && n[1] > 0 && n[2] > 0 ? n[0] * n[1] * n[2] : 0;
    __syncthreads();
    // the K-th largest count of the source positions: eight lanes each
    int thr = 0;
    {
      const int m = tid >> 3, sub = tid & 7;
      const uint32_t sp = sh.srcPos[m];
      int c = 0;
      if (sp != kNone) {
        const int c0 = (int)(sp % (uint32_t)s0) - lo[0];
        c = count_at(bits, bt, T, c0, (sp / (uint32_t)s0) * (uint32_t)W0 * 4u, sub, 8);
      }
#pragma unroll
      for (int off = 1; off < 8; off <<= 1) c += __shfl_xor(c, off);
      if (sub == 0) sh.srcCost[m] = sp != kNone ? (float)c : -1.f;
      if (tid == 0) {
        sh.thr = 0.f;
        sh.m[0] = 0;
        sh.unit = 0;
      }
      __syncthreads();
      if (tid < kSources) {
        const float mine = sh.srcCost[tid];
        int rank = 0;
        for (int u = 0; u < kSources; ++u) rank += (sh.srcCost[u] > mine || (sh.srcCost[u] == mine && u < tid)) ? 1 : 0;
        if (rank == K - 1) sh.thr = fmaxf(mine, 0.f);
      }
      __syncthreads();
      thr = __builtin_amdgcn_readfirstlane((int)sh.thr);
    }
    // a lane sums kWords words of 32 positions: one 16-byte load a term feeds
    // them (bits past the row's end belong to no valid position)
    const int W = (n[0] + 31) >> 5, WU = (W + kWords - 1) / kWords;
    const int units = Nv > 0 ? WU * n[1] * n[2] : 0;
    // K best of this lane: rank (count, hash) and position; the hash is a
    // bijection of the position, so ranks are distinct
    unsigned long long br[KT];
    uint32_t bp[KT];
#pragma unroll
    for (int k = 0; k < KT; ++k) {
      br[k] = 0ull;
      bp[k] = kNone;
    }
    __builtin_amdgcn_s_setprio(0);
    // every G-th run of 64 units belongs to the slice, handed out to its wavefronts
    for (;;) {
      int k = 0;
      if (lane == 0) k = atomicAdd(&sh.unit, 1);
      k = __builtin_amdgcn_readfirstlane(k);
      const int ub = (k * G + slice) * 64;
      if (ub >= units) break;
      const int u = min(ub + lane, units - 1);
      const bool in = ub + lane < units;
      const int row = u / WU, w0 = (u - row * WU) * kWords;
      const int r2 = row / n[1], r1 = row - r2 * n[1];
      const int line = lo[1] + r1 + s1 * (lo[2] + r2);
      const uint32_t ab = (uint32_t)(line * W0 + w0) * 4u;
      uint32_t c[kWords][NP];
#pragma unroll
      for (int x = 0; x < kWords; ++x)
#pragma unroll
        for (int k2 = 0; k2 < NP; ++k2) c[x][k2] = 0u;
      for (int t = 0; t < T; t += 8) {
        uint4 y[8];
        int h[8];
        uint32_t av = ab;
        asm volatile("" : "+v"(av));  // scalar base addressing, as in add_step
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const char* b = bits + __builtin_amdgcn_readfirstlane(bt.off[t + e]);
          h[e] = __builtin_amdgcn_readfirstlane(bt.sh[t + e]);
          __builtin_memcpy(&y[e], b + av, 16);
        }
#pragma unroll
        for (int x = 0; x < kWords; ++x) {
          uint32_t z[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const uint32_t lw = x == 0 ? y[e].x : x == 1 ? y[e].y : y[e].z;
            const uint32_t hw = x == 0 ? y[e].y : x == 1 ? y[e].z : y[e].w;
            z[e] = __builtin_amdgcn_alignbit(hw, lw, h[e]);
          }
          uint32_t t2a, t2b, f4a, f4b, e8;
          csa(t2a, c[x][0], c[x][0], z[0], z[1]);
          csa(t2b, c[x][0], c[x][0], z[2], z[3]);
          csa(f4a, c[x][1], c[x][1], t2a, t2b);
          csa(t2a, c[x][0], c[x][0], z[4], z[5]);
          csa(t2b, c[x][0], c[x][0], z[6], z[7]);
          csa(f4b, c[x][1], c[x][1], t2a, t2b);
          csa(e8, c[x][2], c[x][2], f4a, f4b);
#pragma unroll
          for (int k2 = 3; k2 < NP; ++k2) {
            const uint32_t carry = c[x][k2] & e8;
            c[x][k2] ^= e8;
            e8 = carry;
          }
        }
      }
      bool found = false;
#pragma unroll
      for (int x = 0; x < kWords; ++x) {
        // positions of the box whose count reaches the K-th known one
        const int left = n[0] - 32 * (w0 + x);
        uint32_t ge = 0u, eq = !in || left <= 0 ? 0u : left >= 32 ? 0xFFFFFFFFu : (1u << left) - 1u;
#pragma unroll
        for (int k2 = NP - 1; k2 >= 0; --k2) {
          if ((thr >> k2) & 1) {  // uniform
            eq &= c[x][k2];
          } else {
            ge |= eq & c[x][k2];
            eq &= ~c[x][k2];
          }
        }
        ge |= eq;
        if (__ballot(ge != 0u) == 0ull) continue;
        found = true;
        const uint32_t pb = (uint32_t)(lo[0] + 32 * (w0 + x) + s0 * line);
        while (ge) {
          const int b = __ffs(ge) - 1;
          ge &= ge - 1u;
          uint32_t cv = 0u;
#pragma unroll
          for (int k2 = 0; k2 < NP; ++k2) cv |= ((c[x][k2] >> b) & 1u) << k2;
          const uint32_t p = pb + (uint32_t)b;
          unsigned long long r = ((unsigned long long)(cv + 1u) << 32) | tie_hash(seedbits, p);
          if (!(r > br[KT - 1])) continue;
          uint32_t pp = p;
#pragma unroll
          for (int k2 = 0; k2 < KT; ++k2)
            if (r > br[k2]) {
              const unsigned long long tr = br[k2];
              const uint32_t tp = bp[k2];
              br[k2] = r;
              bp[k2] = pp;
              r = tr;
              pp = tp;
            }
        }
      }
      if (found) {
        // a lane that holds K positions bounds the K-th count
        int kc = 0;
#pragma unroll
        for (int k2 = 0; k2 < KT; ++k2)
          if (k2 == K - 1) kc = (int)(br[k2] >> 32) - 1;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) kc = max(kc, __shfl_xor(kc, off));
        if (kc > thr && lane == 0) atomicMax(&sh.m[0], kc);
        thr = max(thr, kc);
      }
      // what the other wavefronts of the block know
      thr = __builtin_amdgcn_readfirstlane(max(thr, *(volatile int*)&sh.m[0]));
    }
    __builtin_amdgcn_s_setprio(3);
    // K rounds of block maxima
    auto block_best = [&]() {
      for (int k = 0; k < K; ++k) {
        unsigned long long m = br[0];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
          const unsigned long long o = __shfl_xor(m, off);
          m = o > m ? o : m;
        }
        if (br[0] == m && m != 0ull) redP[wave] = bp[0];
        if (lane == 0) red[wave] = m;
        __syncthreads();
        unsigned long long bm = 0ull;
        uint32_t bpos = kNone;
#pragma unroll
        for (int x = 0; x < kWaves; ++x)
          if (red[x] > bm) {
            bm = red[x];
            bpos = redP[x];
          }
        if (tid == 0) {
          bestR[k] = bm;
          sh.pos[k] = bpos;
        }
        if (br[0] == bm && bm != 0ull) {
#pragma unroll
          for (int x = 0; x < KT - 1; ++x) {
            br[x] = br[x + 1];
            bp[x] = bp[x + 1];
          }
          br[KT - 1] = 0ull;
          bp[KT - 1] = kNone;
        }
        __syncthreads();
      }
    };
    block_best();
    if (G > 1) {
      unsigned long long* sl = P.slots + (long long)q * (G - 1) * K;
      if (slice < G - 1) {
        if (tid < K) st_agent64(&sl[(long long)slice * K + tid], (bestR[tid] >> 32 << 32) | sh.pos[tid]);
        continue;
      }
#pragma unroll
      for (int k = 0; k < KT; ++k) {
        br[k] = 0ull;
        bp[k] = kNone;
      }
      auto push = [&](unsigned long long cp) {
        if ((cp >> 32) == 0ull || cp == kOpen) return;
        uint32_t pp = (uint32_t)cp;
        unsigned long long r = (cp >> 32 << 32) | tie_hash(seedbits, pp);
#pragma unroll
        for (int k = 0; k < KT; ++k)
          if (r > br[k]) {
            const unsigned long long tr = br[k];
            const uint32_t tp = bp[k];
            br[k] = r;
            bp[k] = pp;
            r = tr;
            pp = tp;
          }
      };
      if (tid < K) push((bestR[tid] >> 32 << 32) | sh.pos[tid]);
      for (int e = tid; e < (G - 1) * K; e += kThreads) push(wait_word64(&sl[e], P.polls, &P.ctl[kGaveUp]));
      __syncthreads();  // bestR and sh.pos have been read
      block_best();
    }
    if (tid == 0) {
      write_cell(P, cell, draw_rank(P, i, seed, sh.pos));
      end_tickets(P);
    }
  }
}

// ---------------------------------------------------------------------------
// Set-up and finish
// ---------------------------------------------------------------------------
// the tickets of the next launch; none after a given-up wait
__global__ void k_flow_next(int* ctl) {
  if (ctl[kGaveUp] == 0) ctl[0] = 0;
}

__global__ void k_flow_grid(const float* __restrict__ di, uint32_t* __restrict__ work, long long n) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) work[i] = isnan(di[i]) ? kPending : __float_as_uint(di[i]);
}

// simulated values into the grid; a cell without a valid position keeps what it held
__global__ void k_flow_finish(float* __restrict__ di, const uint32_t* __restrict__ work, long long n) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || !isnan(di[i])) return;
  const uint32_t w = work[i];
  if (w != kPending && w != kEmpty) di[i] = __uint_as_float(w);
}

// variable-planar copy of the TI; categorical variables as class numbers
__global__ void k_flow_planes(const float* __restrict__ ti, int S, int nVar, int v, int cat, int cat0, int nCat,
                              const float* __restrict__ catvals, float* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= S) return;
  const float y = ti[(long long)i * nVar + v];
  if (!cat) {
    out[i] = y;
    return;
  }
  int code = -1;
  for (int q = 0; q < nCat; ++q)
    if (catvals[cat0 + q] == y) code = q;
  out[i] = (float)code;
}

// bit planes of one categorical variable: word w of a row holds cells 32 w .. 32 w + 31
__global__ void k_flow_bits(const float* __restrict__ ti, int s0, int rows, int nVar, int v, int cat0, int nCat,
                            const float* __restrict__ catvals, int W0, int planeWords, uint32_t* __restrict__ bits) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= rows * W0) return;
  const int row = e / W0, w = e - row * W0;
  for (int q = 0; q < nCat; ++q) {
    const float cv = catvals[cat0 + q];
    uint32_t m = 0u;
    for (int b = 0; b < 32; ++b) {
      const int c = 32 * w + b;
      if (c < s0 && ti[((long long)row * s0 + c) * nVar + v] == cv) m |= 1u << b;
    }
    bits[(long long)(cat0 + q) * planeWords + e] = m;
  }
}

template <typename F>
hipError_t launch_persistent(F kernel, const FlowParams& P, size_t lds, int maxBlocks, int cus, hipStream_t st) {
  int per = 0;
  hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, kThreads, lds);
  if (e != hipSuccess) return e;
  const int blocks = std::max(1, std::min(maxBlocks, std::max(1, per) * cus));
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kThreads), lds, st, P);
  return hipGetLastError();
}

}  // namespace

// Slices per node. A slice should run for some tens of microseconds: shorter
// ones spend their time on reading the neighbours, longer ones leave the chip
// idle where few nodes are independent.
static int flow_slices(const FlowPlan& F, long long S, int terms) {
  const long long pairs = S * terms;
  const long long per = F.count ? 1000000 : 160000;
  return (int)std::max<long long>(1, std::min<long long>(48, pairs / per));
}

// Polls of a wait: above any real one, which is what the nodes in flight take
// one after another in the worst case, every slice summing all of its pairs at
// 2 G pairs/s (a block alone reaches 10 and more). A poll takes at least its
// s_sleep(2), 128 cycles: 53 ns at 2.4 GHz.
static int flow_polls(const FlowPlan& F, long long S, int terms, int G, int cus) {
  const double slice = (double)S * terms / G / 2e9;
  const double nodes = std::min<double>(F.inFlight, 8.0 * cus / G + 1.0);  // at most 8 blocks per CU
  return (int)std::min(2e9, (0.5 + nodes * slice) / 53e-9);
}

// The direct scan against the waves, for what is left of a path. The waves'
// transforms cost the same for every image, the direct scan less the sooner
// its bound rules a position out, so the choice is made between segments from
// the tiles and steps that the kernel counted (not from a clock: the same
// request takes the same route under any load).
//
// A chip full of nodes takes kTileUs a tile and stepUs a step; where a level
// has few nodes, it takes a node from its last neighbour's value to its own:
// 50 us, 0.2 us a term (gather, order, merge) and, one after another, the
// steps of one of the node's 4 G wavefronts, 0.45 us each. Measured against
// that, us a node (K <= 2, white noise unless said):
//   1000 x 1000, 1 variable, n 20 / 80 / 250: 2.0 / 4.9 / 16.4 (13.2 K / 40.7 K / 139 K steps)
//   the same, n 80, correlation length 20 / 8: 1.8-3.0 / 2.1-3.7 (11-24 K / 14-30 K steps)
//   1000 x 1000, 2 variables, n 60: 9.9 (63.9 K); with 4 classes, n 80: 18.6 (129 K), smooth 6.3 (41 K)
//   levels of few nodes, us a level: 530 (1000 x 1000, n 250, 139 K steps), 800 (two variables), 316 and 805
//   (1500 x 1500, n 80 and 250, 84 K and 289 K), 154 and 175 (120 x 120 and 250 x 250, n 500)
// More than two best positions cost registers and list flushes: 0.135 ns a
// step instead of 0.105 at 3, 0.25 at 10 (two variables 0.145, 0.19, 0.7).
constexpr double kTileUs = 0.88e-4;
struct FlowCost {
  double nodeUs, levelUs;
};
static FlowCost flow_cost(double tiles, double steps, int terms, int nVar, int K, int G) {
  const double one = nVar == 1 ? 1.05e-4 : 1.45e-4;
  const double stepUs = K <= 2 ? one : nVar == 1 ? (K <= 4 ? 1.35e-4 : 2.5e-4) : (K <= 4 ? 1.9e-4 : 7.0e-4);
  return {tiles * kTileUs + steps * stepUs, 50.0 + 0.2 * terms + 0.45 * (stepUs / one) * steps / (kWaves * G)};
}

// The nodes of R's order from `first` on. A level's nodes wait for the one
// before; at most inFlight of them run at a time.
static double flow_path_us(const FlowPlan& F, const ResidentLoop& R, size_t first, const FlowCost& c) {
  double us = 0.0;
  const size_t nW = R.waveLevel.size();
  for (size_t w = 0; w < nW;) {
    const int level = R.waveLevel[w];
    size_t b = (size_t)R.waveStart[w];
    while (w < nW && R.waveLevel[w] == level) ++w;
    const size_t e = (size_t)R.waveStart[w];
    if (e <= first) continue;
    const double m = (double)(e - std::max(b, first));
    us += std::max(m * c.nodeUs, std::ceil(m / F.inFlight) * c.levelUs);
  }
  return us;
}
static double wave_path_us(const FlowPlan& F, const ResidentLoop& R, size_t first) {
  double us = F.waveSetupUs;
  for (size_t w = 0; w < R.waveLevel.size(); ++w) {
    const size_t b = std::max((size_t)R.waveStart[w], first), e = (size_t)R.waveStart[w + 1];
    if (e > b) us += F.waveUs + (double)(e - b) * F.waveNodeUs;
  }
  return us;
}
constexpr double kHandOver = 1.05;  // the models are good to some 10 %; a segment decides anew

int run_flow(qsmi_ti* t, const ResidentLoop& R, const FlowPlan& F, double* kernelMs, long long* stats, size_t* doneOut,
             bool* gaveUp) {
  hipStream_t st = t->stream;
  *gaveUp = false;
  *doneOut = 0;
  const size_t nPath = (size_t)F.nPath;
  FlowParams P;
  memset(&P, 0, sizeof(P));
  P.D = t->D;
  P.nVar = R.nVar;
  P.nExp = R.nExp;
  P.n = R.n;
  P.K = (int)std::ceil(std::max(R.k, R.kMax));
  P.kf = R.k;
  P.circSim = R.circSim ? 1 : 0;
  for (int d = 0; d < 3; ++d) {
    P.sd[d] = d < t->D ? R.sd[d] : 1;
    P.s[d] = t->s[d];
    P.kdK[0][d] = d < t->D ? R.kd[d] : 1;
  }
  for (int q = 1; q < R.nKer; ++q) {
    for (int d = 0; d < 3; ++d) P.kdK[q][d] = d < t->D ? R.kdK[q][d] : 1;
    P.kerOff[q] = R.kerOff[q];
  }
  for (int v = 0; v < R.nVar; ++v) {
    P.types[v] = R.types[v];
    P.e0[v] = F.e0[v];
    P.nCat[v] = F.nCat[v];
    P.cat0[v] = F.cat0[v];
  }
  for (int e = 0; e < R.nExp; ++e) {
    P.expVar[e] = R.expVar[e];
    P.expCat[e] = R.expCat[e];
  }
  for (int q = 0; q < kFlowMaxCat; ++q) P.rare[q] = F.rare[q];
  P.S = (int)t->S;
  P.order = R.dOrder;
  P.cells = R.dPathCells;
  P.seeds = R.dPathSeeds;
  P.nbIdx = R.dNbIdx;
  P.nbCnt = R.dNbCnt;
  P.offs = R.dOffs;
  P.kern = R.dKernel;
  P.catvals = R.dCatvals;
  P.pathK = R.dPathK;
  P.nodeKer = R.dNodeKer;
  P.tiVals = R.dTi;
  P.di = R.dDi;
  P.index = R.dIndex;
  const int terms = R.n * R.nVar;
  P.G = flow_slices(F, t->S, terms);
  P.W0 = (t->s[0] + 31) / 32;
  const int rows = t->s[1] * t->s[2];
  P.planeWords = rows * P.W0;
  P.zeroPlane = F.nClasses;
  const size_t SD = (size_t)P.sd[0] * P.sd[1] * P.sd[2];
  // one launch simulates a segment of the path (slots and tickets of its own),
  // a shorter one when progress is reported between them
  const size_t seg = std::min<size_t>(std::max<size_t>(nPath, 1),
                                      (size_t)(R.progressSec > 0 ? std::min(F.segment, 8192) : F.segment));
  const size_t slotWords = (size_t)seg * (P.G - 1) * P.K * (F.count ? 1 : 2);
  struct Mem {
    std::vector<void*> p;
    ~Mem() {
      for (void* x : p) (void)hipFree(x);
    }
  } mem;
  auto alloc = [&](size_t bytes) -> void* {
    void* p = nullptr;
    if (hipMalloc(&p, std::max<size_t>(bytes, 16)) != hipSuccess) return nullptr;
    mem.p.push_back(p);
    return p;
  };
  P.work = (uint32_t*)alloc(SD * R.nVar * sizeof(uint32_t));
  P.ctl = (int*)alloc(kCtlWords * sizeof(int));
  P.stats = (unsigned long long*)alloc(kFlowStats * sizeof(unsigned long long));
  P.slots = (unsigned long long*)alloc(slotWords * sizeof(unsigned long long));
  float* planes = F.count ? nullptr : (float*)alloc((size_t)R.nVar * t->S * sizeof(float));
  uint32_t* bits = F.count ? (uint32_t*)alloc(((size_t)(F.nClasses + 1) * P.planeWords + 4) * sizeof(uint32_t)) : nullptr;
  if (!P.work || !P.ctl || !P.stats || !P.slots || (F.count ? !bits : !planes))
    return fail(QSMI_ERR_NOMEM, "path loop: out of device memory");
  P.planes = planes;
  P.bits = bits;
  hipError_t e = hipSuccess;
  if (!F.count) {
    float* dq = (float*)alloc(F.quant.size() * sizeof(float));
    if (!dq) return fail(QSMI_ERR_NOMEM, "path loop: out of device memory");
    e = hipMemcpy(dq, F.quant.data(), F.quant.size() * sizeof(float), hipMemcpyHostToDevice);
    P.quant = dq;
  }
  if (e == hipSuccess) e = hipMemsetAsync(P.ctl, 0, kCtlWords * sizeof(int), st);
  if (e == hipSuccess) e = hipMemsetAsync(P.stats, 0, kFlowStats * sizeof(unsigned long long), st);
  const long long words = (long long)SD * R.nVar;
  hipLaunchKernelGGL(k_flow_grid, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, st, R.dDi, P.work, words);
  if (F.count && e == hipSuccess)
    e = hipMemsetAsync(bits + (size_t)P.zeroPlane * P.planeWords, 0, (size_t)P.planeWords * sizeof(uint32_t), st);
  for (int v = 0; v < R.nVar; ++v) {
    if (F.count)
      hipLaunchKernelGGL(k_flow_bits, dim3((unsigned)((P.planeWords + 255) / 256)), dim3(256), 0, st, R.dTi, t->s[0],
                         rows, R.nVar, v, F.cat0[v], F.nCat[v], R.dCatvals, P.W0, P.planeWords, bits);
    else
      hipLaunchKernelGGL(k_flow_planes, dim3((unsigned)((t->S + 255) / 256)), dim3(256), 0, st, R.dTi, (int)t->S,
                         R.nVar, v, R.types[v] != 0 ? 1 : 0, F.cat0[v], F.nCat[v], R.dCatvals,
                         planes + (size_t)v * t->S);
  }
  if (e == hipSuccess) e = hipGetLastError();
  if (e != hipSuccess) return fail(QSMI_ERR_HIP, std::string("path loop set-up: ") + hipGetErrorString(e));
  int cus = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, t->gpu) != hipSuccess || cus <= 0) cus = 256;
  P.polls = t->tune.flowPolls > 0 ? t->tune.flowPolls : flow_polls(F, t->S, terms, P.G, cus);
  const int nv = R.n * R.nVar;
  const size_t lds = F.count ? (size_t)(2 * (((nv + 7) & ~7) + 8) + 2 * nv + 2 * R.n) * 4
                             : (size_t)(5 * (((nv + 7) & ~7) + 8) + R.nVar * kFlowQuant + 3 * nv + 2 * R.n) * 4;
  const bool timing = R.stageTiming > 0;
  hipEvent_t ev[2] = {nullptr, nullptr};
  if (timing)
    for (auto& x : ev)
      if (hipEventCreate(&x) != hipSuccess) x = nullptr;
  double ms = 0.0;
  const auto begun = std::chrono::steady_clock::now();
  auto told = begun;
  // Whether the waves may be the faster ones: not if the scan is ahead of them
  // with every step of every tile. Otherwise the first segments end after n
  // nodes (whose neighbour lists are still filling), four times that, ... and
  // are judged each; from 65536 nodes on, the 8192 after every 65536.
  bool slow = false;
  bool judge = F.waveNodeUs > 0.0;
  const double maxSteps = (terms + kStep - 1) / kStep;
  if (judge) {
    const double tiles = (double)((t->s[0] + kTileX * kPair - 1) / (kTileX * kPair)) * ((t->s[1] + kTileY - 1) / kTileY) *
                         t->s[2];
    judge = flow_path_us(F, R, 0, flow_cost(tiles, tiles * maxSteps, terms, R.nVar, P.K, P.G)) >
            kHandOver * wave_path_us(F, R, 0);
  }
  size_t countFrom = judge ? 0 : nPath, verdict = (size_t)std::max(64, R.n);  // nodes counted, then judged
  unsigned long long seen[kFlowStats] = {};
  size_t done = 0, judgedAt = 0;
  const size_t stop = t->tune.flowNodes > 0 && !F.alone ? std::min(nPath, (size_t)t->tune.flowNodes) : nPath;
  for (size_t b = 0; b < stop && e == hipSuccess && !slow; b = done) {
    P.node0 = (int)b;
    const bool counted = b >= countFrom;
    P.nNodes = (int)std::min({seg, stop - b, (counted ? verdict : countFrom) - b});
    if (b) hipLaunchKernelGGL(k_flow_next, dim3(1), dim3(1), 0, st, P.ctl);
    if (e == hipSuccess && slotWords) e = hipMemsetAsync(P.slots, 0xFF, slotWords * sizeof(unsigned long long), st);
    if (ev[0] && ev[1]) (void)hipEventRecord(ev[0], st);
    const int maxBlocks = (int)std::min<long long>((long long)P.nNodes * P.G, (long long)F.inFlight * P.G);
#define QSMI_COUNT(NP_, NV_, KT_) launch_persistent(k_flow_count<NP_, NV_, KT_>, P, lds, maxBlocks, cus, st)
#define QSMI_DIRECT(FORM_, NV_, KT_)                                                              \
  (counted ? launch_persistent(k_flow_direct<FORM_, NV_, KT_, true>, P, lds, maxBlocks, cus, st) \
           : launch_persistent(k_flow_direct<FORM_, NV_, KT_, false>, P, lds, maxBlocks, cus, st))
#define QSMI_FLOW(KT_)                                                                           \
  e = F.count ? (terms >= 128  ? QSMI_COUNT(10, 8, KT_)                                          \
                 : R.nVar == 1 ? QSMI_COUNT(7, 1, KT_)                                           \
                               : QSMI_COUNT(7, 8, KT_))                                          \
      : F.mixed    ? (R.nVar <= 2 ? QSMI_DIRECT(2, 2, KT_) : QSMI_DIRECT(2, 8, KT_))             \
      : R.nVar > 1 ? QSMI_DIRECT(1, 8, KT_)                                                      \
      : F.unitW    ? QSMI_DIRECT(0, 1, KT_)                                                      \
                   : QSMI_DIRECT(1, 1, KT_)
    if (e != hipSuccess) break;
    if (P.K <= 2) QSMI_FLOW(2);
    else if (P.K <= 4) QSMI_FLOW(4);
    else QSMI_FLOW(16);
#undef QSMI_FLOW
#undef QSMI_DIRECT
#undef QSMI_COUNT
    if (ev[0] && ev[1]) {
      (void)hipEventRecord(ev[1], st);
      float one = 0.f;
      if (hipEventSynchronize(ev[1]) == hipSuccess && hipEventElapsedTime(&one, ev[0], ev[1]) == hipSuccess) ms += one;
    }
    done = b + (size_t)P.nNodes;
    if (counted && done == verdict && done < nPath) {
      unsigned long long sv[kFlowStats];
      e = hipStreamSynchronize(st);
      if (e == hipSuccess) e = hipMemcpy(sv, P.stats, sizeof(sv), hipMemcpyDeviceToHost);
      if (e != hipSuccess) break;
      const double nodes = (double)(done - countFrom);
      const double tiles = (double)(sv[4] - seen[4]) / nodes, full = (double)(sv[6] - seen[6]) / nodes;
      double steps = (double)(sv[5] - seen[5]) / nodes;
      // the first lists are short: what comes after the first step grows with them
      if (countFrom == 0 && full > tiles)
        steps = tiles + (steps - tiles) * std::max(1.0, tiles * (maxSteps - 1.0) / (full - tiles));
      // An image of ties (zeros, plateaus) fills the scan's lists before their
      // end. The wave loop's lists overflow there too and it rescores whole
      // boxes, some 200 us a node, which its cost does not hold: no hand-over
      // where a node flushes more than one list. 1000 x 1000, 80 neighbours,
      // correlation length 20, us a node, direct / waves: 40 % zeros 11 / 41 (10
      // best 35 / 102), 70 % 12 / 44 (67 / 86), 95 % 46 / 155 (258 / 227); they
      // flush 10 to 3000 lists, noise none.
      const bool ties = sv[3] - seen[3] > done - judgedAt;
      const FlowCost cost = flow_cost(tiles, steps, terms, R.nVar, P.K, P.G);
      slow = !ties && flow_path_us(F, R, done, cost) > kHandOver * wave_path_us(F, R, done);
      judgedAt = done;
      memcpy(seen, sv, sizeof(sv));
      countFrom = done < 65536 ? done : done + 65536;
      verdict = done < 65536 ? 4 * done : countFrom + 8192;
    }
    if (R.progressSec > 0 && hipStreamSynchronize(st) == hipSuccess) {
      const auto now = std::chrono::steady_clock::now();
      if (std::chrono::duration<double>(now - told).count() >= R.progressSec) {
        told = now;
        std::fprintf(stderr, "[qsmi] path loop: %zu of %zu nodes done, %.0f s\n", done, nPath,
                     std::chrono::duration<double>(now - begun).count());
        std::fflush(stderr);
      }
    }
  }
  for (auto& x : ev)
    if (x) (void)hipEventDestroy(x);
  hipLaunchKernelGGL(k_flow_finish, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, st, R.dDi, P.work, words);
  if (e == hipSuccess) e = hipGetLastError();
  int gone = 0;
  unsigned long long sv[kFlowStats] = {};
  const hipError_t es = hipStreamSynchronize(st);
  if (e == hipSuccess) e = es;
  if (e == hipSuccess) e = hipMemcpy(&gone, P.ctl + kGaveUp, sizeof(gone), hipMemcpyDeviceToHost);
  if (e == hipSuccess) e = hipMemcpy(sv, P.stats, sizeof(sv), hipMemcpyDeviceToHost);
  if (e != hipSuccess) return fail(QSMI_ERR_HIP, std::string("path loop: ") + hipGetErrorString(e));
  *gaveUp = gone != 0;
  *doneOut = done;
  *kernelMs = ms;
  for (int q = 0; q < 4; ++q) stats[q] = (long long)sv[q];
  return QSMI_OK;
}

}  // namespace qsmi
