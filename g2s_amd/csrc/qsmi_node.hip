// One node at a time (the per-node API): the mismatch map summed directly in
// FP64, and the K best of it in one pass (gfx950).
//
// A single node leaves the chip idle, so the call is bound by its launches,
// copies and the latency of the longest serial chain, not by arithmetic. The
// transforms need a fill, a neighbour sort, a tap list, the column and the
// row kernel plus three copies of the neighbours; the direct sum is one
// launch whose neighbours travel in the kernel arguments:
//
//   E(p) = delta0 + sum_j sum_a v_ja Y_a(p + d_j)   in FP64, the order and
//   the rounding of the exact selection (qsmi_band.hip),
//
// kept twice: rounded to FP32 (the map that callers read and edit) and in
// FP64. The selection then needs no FP32 band and no second scoring: the
// device rule on the FP64 values of all positions that are finite in the
// FP32 map (exclusions are -inf there) is the exact selection.
//
// Candidate and search of one node, before -> now: 400 x 300 with 40
// neighbours 175 -> 50 us (two launches' and two waits' latency), 1000 x 1000
// with 80 neighbours 207 -> 92 us, of which the sum takes 45 (640 MB of
// cached reads, 14 TB/s: address and FP64 issue, then L1).
#include <hip/hip_runtime.h>

#include "qsmi_internal.hpp"
#include "qsmi_select.hpp"

namespace qsmi {
namespace {

constexpr int kBatch = 8;  // neighbours whose loads are in flight together

// 256 threads, P positions a thread 64 apart. A position outside the valid
// box reads as the box's first corner (every load stays inside the TI) and
// writes -inf. VV: sub-images, 0 for any number.
template <int VV, int P>
__global__ void __launch_bounds__(256) k_node_map(ScanGeom g, NodeArgs a, const float* __restrict__ Y, int S,
                                                  double nscale, float* __restrict__ map, double* __restrict__ mapD,
                                                  NodeInfo* __restrict__ info, int* __restrict__ off,
                                                  float* __restrict__ val) {
  __shared__ int sd[kNodeWords + kBatch];
  __shared__ double sv[kNodeWords];
  const int tid = threadIdx.x, nb = a.ni.nb, D = g.D, V = VV ? VV : g.V;
  for (int j = tid; j < nb + kBatch; j += 256) {
    int t = 0, mul = 1;
    for (int d = 0; d < D; ++d) {
      t += a.w[min(j, nb - 1) * D + d] * mul;
      mul *= g.s[d];
    }
    sd[j] = t;
  }
  for (int i = tid; i < nb * V; i += 256) sv[i] = (double)__int_as_float(a.w[nb * D + i]);
  if (blockIdx.x == 0) {  // what the other selections of this node read
    for (int i = tid; i < nb * D; i += 256) off[i] = a.w[i];
    for (int i = tid; i < nb * V; i += 256) val[i] = __int_as_float(a.w[nb * D + i]);
    if (tid == 0) *info = a.ni;
  }
  const int n0 = a.ni.hi[0] - a.ni.lo[0], n1 = a.ni.hi[1] - a.ni.lo[1], n2 = a.ni.hi[2] - a.ni.lo[2];
  const bool box = n0 >= 0 && n1 >= 0 && n2 >= 0;
  const int corner = a.ni.lo[0] + g.s[0] * (a.ni.lo[1] + g.s[1] * a.ni.lo[2]);
  const long long first = ((long long)blockIdx.x * 4 + (tid >> 6)) * (64 * P) + (tid & 63);
  int p[P];
  bool ok[P], any = false;
  double acc[P];
#pragma unroll
  for (int q = 0; q < P; ++q) {
    const long long i = first + 64 * q;
    const int c = (int)min(i, (long long)S - 1);
    const int c0 = c % g.s[0], r = c / g.s[0], c1 = r % g.s[1], c2 = r / g.s[1];
    ok[q] = box && i < S && (unsigned)(c0 - a.ni.lo[0]) <= (unsigned)n0 && (unsigned)(c1 - a.ni.lo[1]) <= (unsigned)n1 &&
            (unsigned)(c2 - a.ni.lo[2]) <= (unsigned)n2;
    p[q] = ok[q] ? c : corner;
    any |= ok[q];
    acc[q] = (double)a.ni.delta0;
  }
  __syncthreads();
  if (__any(any)) {
    for (int j0 = 0; j0 < nb; j0 += kBatch) {
      if (VV) {
        float y[kBatch][VV ? VV : 1][P];
#pragma unroll
        for (int u = 0; u < kBatch; ++u)
#pragma unroll
          for (int v = 0; v < VV; ++v)
#pragma unroll
            for (int q = 0; q < P; ++q) y[u][v][q] = Y[(long long)g.A[v] * S + (p[q] + sd[j0 + u])];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
          if (j0 + u < nb) {
#pragma unroll
            for (int v = 0; v < VV; ++v)
#pragma unroll
              for (int q = 0; q < P; ++q)
                acc[q] = __dadd_rn(acc[q], __dmul_rn(sv[(j0 + u) * VV + v], (double)y[u][v][q]));
          }
        }
      } else {
        for (int u = 0; u < kBatch && j0 + u < nb; ++u)
#pragma unroll 4
          for (int v = 0; v < V; ++v)
#pragma unroll
            for (int q = 0; q < P; ++q)
              acc[q] = __dadd_rn(acc[q], __dmul_rn(sv[(j0 + u) * V + v],
                                                   (double)Y[(long long)g.A[v] * S + (p[q] + sd[j0 + u])]));
      }
    }
  }
#pragma unroll
  for (int q = 0; q < P; ++q) {
    const long long i = first + 64 * q;
    if (i >= S) continue;
    const double e = ok[q] ? (nscale == 1.0 ? acc[q] : acc[q] * nscale) : -INFINITY;
    map[i] = (float)e;
    mapD[i] = e;
  }
}

// The K best of a chunk of the map; grid.x chunks, part [chunk][K].
template <int KT>
__global__ void __launch_bounds__(256) k_node_select(const float* __restrict__ map, const double* __restrict__ mapD,
                                                     int S, int chunk, int K, uint32_t seedbits,
                                                     Cand64* __restrict__ part) {
  __shared__ Cand64 red[4];
  const int beg = blockIdx.x * chunk, end = min(S, beg + chunk);
  TopK64<KT> tk;
  tk.init();
  for (int i = beg + (int)threadIdx.x; i < end; i += 256) {
    if (!isfinite(map[i])) continue;
    Cand64 c;
    c.val = mapD[i];
    c.h = tie_hash(seedbits, (uint32_t)i);
    c.pos = (uint32_t)i;
    tk.push(c);
  }
  block_topk64<KT>(tk, K, part + (long long)blockIdx.x * K, red);
}

// The K best of the chunks, into host memory: K values, then K positions.
template <int KT>
__global__ void __launch_bounds__(256) k_node_merge(const Cand64* __restrict__ part, int n, int K,
                                                    uint32_t* __restrict__ out) {
  __shared__ Cand64 red[4];
  __shared__ Cand64 best[kMaxK];
  TopK64<KT> tk;
  tk.init();
  for (int i = threadIdx.x; i < n; i += 256) tk.push(part[i]);
  block_topk64<KT>(tk, K, best, red);
  if (threadIdx.x < (unsigned)K) {
    out[threadIdx.x] = __float_as_uint((float)best[threadIdx.x].val);
    out[K + threadIdx.x] = best[threadIdx.x].pos;
  }
}

}  // namespace

void launch_node_map(const ScanGeom& g, const NodeArgs& a, const float* Y, long long S, double nscale, float* map,
                     double* mapD, NodeInfo* info, int* off, float* val, hipStream_t st) {
  // four positions a thread share the neighbours' reads; below 2^19 positions
  // that would leave fewer than two wavefronts a SIMD
  const bool wide = S >= (1 << 19);
  const unsigned blocks = (unsigned)((S + (wide ? 1023 : 255)) / (wide ? 1024 : 256));
#define QSMI_NODE(VV_, P_)                                                                                       \
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_node_map<VV_, P_>), dim3(blocks), dim3(256), 0, st, g, a, Y, (int)S,     \
                     nscale, map, mapD, info, off, val)
  if (wide) {
    if (g.V == 2) QSMI_NODE(2, 4);
    else if (g.V == 1) QSMI_NODE(1, 4);
    else QSMI_NODE(0, 4);
  } else {
    if (g.V == 2) QSMI_NODE(2, 1);
    else if (g.V == 1) QSMI_NODE(1, 1);
    else QSMI_NODE(0, 1);
  }
#undef QSMI_NODE
}

// part: kNodeChunks * K entries.
void launch_node_select(const float* map, const double* mapD, long long S, int K, uint32_t seedbits, Cand64* part,
                        uint32_t* out, hipStream_t st) {
  const int chunk = (int)std::max<long long>(1024, (S + kNodeChunks - 1) / kNodeChunks);
  const int blocks = (int)((S + chunk - 1) / chunk);
#define QSMI_NODE(KT_)                                                                                           \
  hipLaunchKernelGGL(k_node_select<KT_>, dim3(blocks), dim3(256), 0, st, map, mapD, (int)S, chunk, K, seedbits,  \
                     part);                                                                                      \
  hipLaunchKernelGGL(k_node_merge<KT_>, dim3(1), dim3(256), 0, st, part, blocks * K, K, out)
  if (K <= 2) {
    QSMI_NODE(2);
  } else if (K <= 4) {
    QSMI_NODE(4);
  } else if (K <= 8) {
    QSMI_NODE(8);
  } else {
    QSMI_NODE(16);
  }
#undef QSMI_NODE
}

}  // namespace qsmi
