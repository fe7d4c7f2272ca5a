// Small device utilities: fills, fixed-point conversion
// and the final fixed-order energy/virial reduction (self energy included).
#include <algorithm>
#include <cmath>
#include <set>
#include <type_traits>

#include "apocharmm_amd.h"
#include "system.hpp"

namespace apo {

// Fills (kernels instead of hipMemsetAsync so the step stays graph-safe).
__global__ void k_fill_i64(int64_t *p, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    p[i] = 0;
}
static int fill_blocks(size_t n) { return (int)std::min<size_t>((n + 255) / 256, 4096); }
__global__ void k_fill_f64(double *p, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    p[i] = 0.0;
}

__global__ void k_fill_i32(int *p, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    p[i] = 0;
}
void launch_fill_i32(int *p, size_t n, hipStream_t s) {
  if (!n) return;
  int nb = (int)std::min<size_t>((n + 255) / 256, 4096);
  k_fill_i32<<<nb, 256, 0, s>>>(p, n);
  APO_LAUNCH_CHECK();
}

void launch_fill_i64(int64_t *p, size_t n, hipStream_t s) {
  if (!n) return;
  int nb = (int)std::min<size_t>((n + 255) / 256, 4096);
  k_fill_i64<<<nb, 256, 0, s>>>(p, n);
  APO_LAUNCH_CHECK();
}
void launch_fill_f64(double *p, size_t n, hipStream_t s) {
  if (!n) return;
  int nb = (int)std::min<size_t>((n + 255) / 256, 4096);
  k_fill_f64<<<nb, 256, 0, s>>>(p, n);
  APO_LAUNCH_CHECK();
}

// Force<long long> -> double (src/reduce.cu:132-143).
__global__ void k_force_to_double(const int64_t *f, int natom, int stride, double *out) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= natom) return;
  for (int c = 0; c < 3; c++)
    out[(size_t)c * stride + i] = (double)f[(size_t)c * stride + i] * kInvForceScale;
}

void launch_force_to_double(const int64_t *f, int natom, int stride, double *out,
                            hipStream_t s) {
  k_force_to_double<<<(natom + 255) / 256, 256, 0, s>>>(f, natom, stride, out);
  APO_LAUNCH_CHECK();
}

// Plugin gradient into the total (add_force, src/reduce.cu:177-189).
__global__ void k_add_force(const int64_t *src, int natom, int stride, int64_t *dst) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= natom) return;
  for (int c = 0; c < 3; c++) dst[(size_t)c * stride + i] += src[(size_t)c * stride + i];
}
void launch_add_force(const int64_t *src, int natom, int stride, int64_t *dst, hipStream_t s) {
  k_add_force<<<(natom + 255) / 256, 256, 0, s>>>(src, natom, stride, dst);
  APO_LAUNCH_CHECK();
}
// Plugin energy term 0 into the potential (src/ForceManager.cu:774-778).
__global__ void k_add_energy(const double *src, double *energy) {
  if (threadIdx.x == 0) energy[APO_E_EPOT] += src[0];
}
void launch_add_energy(const double *src, double *energy, hipStream_t s) {
  k_add_energy<<<1, 64, 0, s>>>(src, energy);
  APO_LAUNCH_CHECK();
}

// Final reduction of the energy and virial partials, two launches: k_reduce_parts
// sums kReduceRows rows of one region's partials per block (all components of
// a row together), and k_reduce_final, one block, adds the blocks' sums and
// writes the energies and the virial.  Both sum in a fixed order, so the bits
// do not change from run to run.  The Ewald self energy's sum of q^2
// (include/cuda_pme_selfe.h:14-53) is one more region, read from xyzq.
// Latency bounds both: the partials are at most a few hundred KB.  A block per
// 1,024 rows gives each thread four rows in flight and 13 to 35 blocks; one
// block reading component after component, with the self energy's own launch
// before it, took 73 us at 2,529 atoms and 92 us at 93,984, the two launches
// take 8 and 11 us (energy and virial calls 240 -> 179 us and 1,172 -> 1,094).
constexpr int kReduceThreads = 256, kReduceRows = 1024, kReduceAtoms = 4096;
constexpr int kReduceWidth = 11;  // widest region (bonded)
enum { RED_PAIR = 0, RED_P14, RED_BOND, RED_RECIP, RED_SELF, RED_NUM };
struct ReduceRegion {
  int off, n, width;  // offset in the partials, rows (atoms for RED_SELF), components per row
  int start;          // first chunk
};
struct ReduceArgs {
  ReduceRegion r[RED_NUM];
  int nchunk;
  int E, V;
  int acc;  // add into energy / virial instead of overwriting
  double self_fac;
};

static_assert(kPairPart <= kReduceWidth && kP14Part <= kReduceWidth &&
                  kBondPart <= kReduceWidth && kRecipPart <= kReduceWidth,
              "reduction width");

template <int W, typename Load>
__device__ __forceinline__ void reduce_chunk(int r0, int r1, Load &&load, double *out) {
  __shared__ double sh[kReduceThreads / 64][W];
  double v[W];
#pragma unroll
  for (int k = 0; k < W; k++) v[k] = 0.0;
  for (int r = r0 + threadIdx.x; r < r1; r += kReduceThreads)
#pragma unroll
    for (int k = 0; k < W; k++) v[k] += load(r, k);
#pragma unroll
  for (int k = 0; k < W; k++) {
    for (int off = 32; off > 0; off >>= 1) v[k] += __shfl_xor(v[k], off);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6][k] = v[k];
  }
  __syncthreads();
  if (threadIdx.x < W) {
    double s = 0.0;
    for (int w = 0; w < kReduceThreads / 64; w++) s += sh[w][threadIdx.x];
    out[threadIdx.x] = s;
  }
}

__global__ __launch_bounds__(kReduceThreads) void k_reduce_parts(const double *__restrict__ parts,
                                                                 const float4 *__restrict__ xyzq,
                                                                 ReduceArgs a,
                                                                 double *__restrict__ sums) {
  const int c = blockIdx.x;
  int g = 0;
  while (g + 1 < RED_NUM && a.r[g + 1].start <= c) g++;
  const ReduceRegion R = a.r[g];
  double *out = sums + (size_t)c * kReduceWidth;
  const int per = g == RED_SELF ? kReduceAtoms : kReduceRows;
  const int r0 = (c - R.start) * per, r1 = min(r0 + per, R.n);
  const double *p = parts + R.off;
  auto row = [&](auto w) {
    constexpr int W = decltype(w)::value;
    reduce_chunk<W>(r0, r1, [&](int r, int k) { return p[(size_t)r * W + k]; }, out);
  };
  if (g == RED_PAIR) row(std::integral_constant<int, kPairPart>{});
  else if (g == RED_P14) row(std::integral_constant<int, kP14Part>{});
  else if (g == RED_BOND) row(std::integral_constant<int, kBondPart>{});
  else if (g == RED_RECIP) row(std::integral_constant<int, kRecipPart>{});
  else
    reduce_chunk<1>(r0, r1, [&](int r, int) {
      const double q = (double)xyzq[r].w;
      return q * q;
    }, out);
}

// Four lanes per (region, component) add that component's chunk sums.
__global__ __launch_bounds__(256) void k_reduce_final(const double *__restrict__ sums, ReduceArgs a,
                                                      double *__restrict__ energy,
                                                      double *__restrict__ virial) {
  static_assert(4 * RED_NUM * kReduceWidth <= 256, "one thread group per component");
  __shared__ double t[RED_NUM][kReduceWidth];
  const int id = threadIdx.x >> 2, sub = threadIdx.x & 3;
  const int g = id / kReduceWidth, k = id % kReduceWidth;
  double s = 0.0;
  if (g < RED_NUM && k < a.r[g].width) {
    const int c1 = g + 1 < RED_NUM ? a.r[g + 1].start : a.nchunk;
    for (int c = a.r[g].start + sub; c < c1; c += 4) s += sums[(size_t)c * kReduceWidth + k];
  }
  s += __shfl_xor(s, 1);
  s += __shfl_xor(s, 2);
  if (g < RED_NUM && sub == 0) t[g][k] = s;
  __syncthreads();
  if (threadIdx.x != 0) return;
  if (a.E) {
    double e[APO_NUM_ENERGY] = {0};
    for (int c = 0; c < 5; c++) e[c] = t[RED_BOND][c];
    e[APO_E_EWKS] = t[RED_RECIP][0];
    e[APO_E_EWSE] = a.self_fac * t[RED_SELF][0];
    e[APO_E_EWEX] = t[RED_P14][2];
    e[APO_E_ELEC] = t[RED_PAIR][0] + t[RED_P14][0];
    e[APO_E_VDW] = t[RED_PAIR][1] + t[RED_P14][1];
    double tot = 0;
    for (int c = 0; c < APO_E_EPOT; c++) tot += e[c];
    e[APO_E_EPOT] = tot;
    for (int c = 0; c < APO_NUM_ENERGY; c++) energy[c] = a.acc ? energy[c] + e[c] : e[c];
  }
  if (a.V) {
    double v6[6];
    for (int c = 0; c < 6; c++)
      v6[c] = t[RED_PAIR][2 + c] + t[RED_P14][3 + c] + t[RED_BOND][5 + c] + t[RED_RECIP][1 + c];
    const double w[9] = {v6[0], v6[1], v6[2], v6[1], v6[3], v6[4], v6[2], v6[4], v6[5]};
    for (int c = 0; c < 9; c++) virial[c] = a.acc ? virial[c] + w[c] : w[c];
  }
}

// chunk sums of the largest reduction this system can ask for
size_t reduce_sums_size(const PartLayout &L, int natom) {
  auto chunks = [](int n, int per) { return (size_t)((n + per - 1) / per); };
  return kReduceWidth * (chunks(L.pair_n, kReduceRows) + chunks(L.p14_n, kReduceRows) +
                         chunks(L.bond_n, kReduceRows) + chunks(L.recip_n, kReduceRows) +
                         chunks(natom, kReduceAtoms));
}

void reduce_energy_launch(NbSystem &S, const float4 *x, int terms, bool E, bool V, double *energy,
                          double *virial, hipStream_t s, bool accumulate) {
  const PartLayout &L = S.part;
  const bool bonded = S.nbond + S.nub + S.nangle + S.ndihe + S.nimdihe > 0;
  ReduceArgs a;
  a.nchunk = 0;
  auto region = [&](int g, bool on, int off, int n, int width, int per) {
    a.r[g] = ReduceRegion{off, on ? n : 0, width, a.nchunk};
    a.nchunk += (a.r[g].n + per - 1) / per;
  };
  // rows the kernels of this call wrote; a term that is off or empty has none
  region(RED_PAIR, terms & APO_TERM_DIRECT, L.pair_off, L.pair_n, kPairPart, kReduceRows);
  region(RED_P14, (terms & APO_TERM_PAIRS14) && S.nin14 + S.nex14 > 0, L.p14_off, L.p14_n,
         kP14Part, kReduceRows);
  region(RED_BOND, (terms & APO_TERM_BONDED) && bonded, L.bond_off, L.bond_n, kBondPart,
         kReduceRows);
  region(RED_RECIP, terms & APO_TERM_RECIP, L.recip_off, L.recip_used, kRecipPart, kReduceRows);
  region(RED_SELF, (terms & APO_TERM_SELF) && E, 0, S.natom, 1, kReduceAtoms);
  a.E = E;
  a.V = V;
  a.acc = accumulate ? 1 : 0;
  a.self_fac = -S.kappa * kCcelec / std::sqrt(kPi);
  if (a.nchunk) {
    k_reduce_parts<<<a.nchunk, kReduceThreads, 0, s>>>(S.parts_ptr(), x, a, S.red_sums.get());
    APO_LAUNCH_CHECK();
  }
  k_reduce_final<<<1, 256, 0, s>>>(S.red_sums.get(), a, energy, virial);
  APO_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------
// Topology: 1-2/1-3/1-4 sets from the bond graph and the exclusion CSR /
// in14 / ex14 lists (CharmmPSF::buildTopologicalExclusions and
// getInclusionExclusionLists, src/CharmmPSF.cu:235-385).
// ---------------------------------------------------------------------------
void build_exclusions(int natom, int nbond, const int32_t *bonds,
                      std::vector<int32_t> &excl_ptr, std::vector<int32_t> &excl_idx,
                      std::vector<int32_t> &in14, std::vector<int32_t> &ex14) {
  std::vector<std::set<int>> c12(natom), c13(natom), c14(natom);
  for (int b = 0; b < nbond; b++) {
    int i = bonds[2 * b], j = bonds[2 * b + 1];
    c12[i].insert(j);
    c12[j].insert(i);
  }
  for (int b = 0; b < nbond; b++) {
    int i = bonds[2 * b], j = bonds[2 * b + 1];
    for (int a : c12[j])
      if (a != i) c13[i].insert(a);
    for (int a : c12[i])
      if (a != j) c13[j].insert(a);
  }
  for (int i = 0; i < natom; i++)
    for (int j : c13[i])
      for (int k : c12[j])
        if (!c12[i].count(k)) c14[i].insert(k);
  excl_ptr.assign(1, 0);
  excl_idx.clear();
  in14.clear();
  ex14.clear();
  for (int i = 0; i < natom; i++) {
    std::set<int> all;
    all.insert(c12[i].begin(), c12[i].end());
    all.insert(c13[i].begin(), c13[i].end());
    all.insert(c14[i].begin(), c14[i].end());
    all.erase(i);
    for (int j : all) excl_idx.push_back(j);
    excl_ptr.push_back((int32_t)excl_idx.size());
    for (int j : c14[i])
      if (j > i && !c12[i].count(j) && !c13[i].count(j)) {
        in14.push_back(i);
        in14.push_back(j);
      }
    std::set<int> ex(c12[i].begin(), c12[i].end());
    ex.insert(c13[i].begin(), c13[i].end());
    for (int j : ex)
      if (j > i) {
        ex14.push_back(i);
        ex14.push_back(j);
      }
  }
}

}  // namespace apo
