// Neighbor list: xy-column binning, deterministic z sort per column in LDS,
// 32-atom cells with bounding boxes, cell-pair tiles inside the list cutoff,
// per-tile 32x32 exclusion/prune masks, per 16-slot i-group the packed
// j slots that have a live pair, and the pair-kernel work items.
//
// Reference behaviour (re-designed, not translated):
//   CudaNeighborListSort   src/CudaNeighborListSort.cu:31-716 (columns of edge
//                          (V*32/N)^(1/3), z-sorted 32-atom cells, bbox)
//   CudaNeighborListBuild  src/CudaNeighborListBuild.cu:336-969 (cell pairs
//                          within the list cutoff, 32x32 exclusion masks,
//                          diagonal tile keeps i<j only)
// Differences by design: coordinates are 32-bit fixed point per box edge, so
// every pair uses its minimum image through integer wrap-around and a tile is
// one cell pair (no 27 image shifts); the column sort orders (z, atom index)
// so what the list holds -- and every result -- is bitwise reproducible (only
// the places of the cells' entry runs in their buffer vary).
#include <algorithm>
#include <cmath>

#include "system.hpp"
#include "thermo.hpp"

namespace apo {

__device__ __forceinline__ uint32_t to_fixed(double x, double inv_len) {
  double f = x * inv_len;
  f -= floor(f);
  // [0,1) -> [0, 2^32); 2^32 wraps to 0 which is the same periodic point
  return (uint32_t)(int64_t)llrint(f * 4294967296.0);
}

// 0. zeroes the build's counts and flags and the column counters.
__global__ void k_list_clear(int *__restrict__ meta, int *__restrict__ col_count, int ncol) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < 16) meta[i] = 0;
  if (i <= ncol) col_count[i] = 0;
}

// 1. column of each atom (wrapped xy) and its slot in the column.  Atoms
// that are neighbours in index order usually share a column, so the lanes of
// a wave that hit the same column take their slots with one atomic (the
// first such lane adds the group's size, the others take consecutive slots).
// The lanes are grouped first and every group's atomic is in flight at once:
// with a round trip inside the grouping loop the kernel took 26.8 us at 94k
// atoms and 12.6 at 12k, so 12.0 and 4.2.
// The coordinates the list is built from are kept (xref) for the integrator's
// displacement check.
__global__ void k_assign(const float4 *__restrict__ xyzq, int n, double3 inv_len, double3 len,
                         int ncx, int ncy, int *__restrict__ col_count, int *__restrict__ atom_col,
                         int *__restrict__ atom_slot, float *__restrict__ zkey,
                         int *__restrict__ meta, float4 *__restrict__ xref) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float4 p = xyzq[i];
  xref[i] = p;
  double fx = (double)p.x * inv_len.x, fy = (double)p.y * inv_len.y, fz = (double)p.z * inv_len.z;
  fx -= floor(fx);
  fy -= floor(fy);
  fz -= floor(fz);
  // non-finite input: flag it (the host raises) and keep every index in range
  if (!(fx >= 0.0 && fx <= 1.0 && fy >= 0.0 && fy <= 1.0 && fz >= 0.0 && fz <= 1.0)) {
    atomicOr(&meta[6], 1);
    fx = fy = fz = 0.0;
  }
  int cx = max(0, min((int)(fx * ncx), ncx - 1)), cy = max(0, min((int)(fy * ncy), ncy - 1));
  int col = cx + ncx * cy;
  atom_col[i] = col;
  zkey[i] = (float)(fz * len.z);
  const int lane = threadIdx.x & 63;
  const unsigned long long below = (1ull << lane) - 1ull;
  unsigned long long todo = __ballot(true);
  int lead = 0, rank = 0, size = 0;
  while (todo) {
    const int leader = __ffsll((long long)todo) - 1;
    const bool mine = col == __builtin_amdgcn_readlane(col, leader);
    const unsigned long long peers = __ballot(mine);
    if (mine) {
      lead = leader;
      rank = __popcll(peers & below);
      size = __popcll(peers);
    }
    todo &= ~peers;
  }
  int base = 0;
  if (lane == lead) base = atomicAdd(&col_count[col], size);
  atom_slot[i] = __shfl(base, lead, 64) + rank;
}

// 2. starts of the columns: block 0 scans the atom counts (and notes the
// largest column), block 1 the 32-atom cells; the cell total is meta[0].
// Eight columns per thread, chunks of 8192 follow each other with a carry.
constexpr int kScanThreads = 1024, kScanPer = 8;
__global__ __launch_bounds__(kScanThreads) void k_col_scan(const int *__restrict__ col_count,
                                                           int ncol, int *__restrict__ col_start,
                                                           int *__restrict__ col_cellstart,
                                                           int *__restrict__ meta) {
  constexpr int kW = kScanThreads / 64;
  __shared__ int wsum[kW];
  const bool cells = blockIdx.x == 1;
  int *out = cells ? col_cellstart : col_start;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int carry = 0, mx = 0;
  for (int base = 0; base < ncol; base += kScanThreads * kScanPer) {
    const int i0 = base + tid * kScanPer;
    int v[kScanPer];
    int sum = 0;
#pragma unroll
    for (int k = 0; k < kScanPer; k++) {
      v[k] = i0 + k < ncol ? col_count[i0 + k] : 0;
      mx = max(mx, v[k]);
      if (cells) v[k] = (v[k] + kCell - 1) / kCell;
      sum += v[k];
    }
    int x = sum;  // inclusive scan of the thread sums within the wave
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int y = __shfl_up(x, off, 64);
      if (lane >= off) x += y;
    }
    if (lane == 63) wsum[wave] = x;
    __syncthreads();
    int e = carry + x - sum;
    for (int w = 0; w < kW; w++) {
      if (w < wave) e += wsum[w];
      carry += wsum[w];
    }
#pragma unroll
    for (int k = 0; k < kScanPer; k++) {
      if (i0 + k < ncol) out[i0 + k] = e;
      e += v[k];
    }
    __syncthreads();  // wsum is rewritten by the next chunk
  }
  if (tid == 0) {
    out[ncol] = carry;
    if (cells) meta[0] = carry;
  }
  if (!cells) {
    for (int off = 32; off > 0; off >>= 1) mx = max(mx, __shfl_xor(mx, off, 64));
    if (lane == 0 && mx > 0) atomicMax(&meta[4], mx);
  }
}

// 3. scatter atoms into column order (slot order is arbitrary here; step 4
// makes it deterministic).
__global__ void k_scatter(int n, const int *__restrict__ atom_col, const int *__restrict__ atom_slot,
                          const int *__restrict__ col_start, const float *__restrict__ zkey,
                          unsigned long long *__restrict__ keys) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int pos = col_start[atom_col[i]] + atom_slot[i];
  // (z, atom) packed so that an unsigned compare orders by z then index;
  // z >= 0, so its float bits are monotone as unsigned.
  keys[pos] = ((unsigned long long)__float_as_uint(zkey[i]) << 32) | (unsigned)i;
}

// 4. per-column sort in LDS, then cell layout.  A key's place is the start of
// its z bin plus the number of smaller keys in the bin: atoms spread nearly
// evenly in z, so a bin of a column of 500 holds about two and each key meets
// only those; clustered atoms cost more compares, never a different order.
// Five barriers, 5.7 us for 196 columns of about 480 keys; a bitonic sort,
// 45 barriers, took 31.
constexpr int kSortBins = 256;
__global__ __launch_bounds__(kSortBins) void k_colsort(
    const unsigned long long *__restrict__ keys, const int *__restrict__ col_count,
    const int *__restrict__ col_start, const int *__restrict__ col_cellstart, float bins_per_len,
    int *__restrict__ loc2glo, int *__restrict__ glo2loc, int *__restrict__ meta) {
  constexpr int kPer = kMaxColumn / kSortBins;
  __shared__ unsigned long long sh[kMaxColumn];
  __shared__ int bin_cnt[kSortBins], bin_start[kSortBins + 1];
  __shared__ int wsum[kSortBins / 64];
  const int c = blockIdx.x;
  const int cnt = col_count[c], st = col_start[c];
  const int cs = col_cellstart[c], ncl = (cnt + kCell - 1) / kCell;
  if (cnt > kMaxColumn) {
    // leave the column's slots empty (the host raises after the build)
    if (threadIdx.x == 0) atomicOr(&meta[5], 1);
    for (int k = threadIdx.x; k < ncl * kCell; k += blockDim.x) loc2glo[cs * kCell + k] = -1;
    return;
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // monotone in the key: z >= 0 is its high word
  auto bin_of = [&](unsigned long long key) {
    const float z = __uint_as_float((uint32_t)(key >> 32));
    return max(0, min((int)(z * bins_per_len), kSortBins - 1));
  };
  bin_cnt[tid] = 0;
  __syncthreads();
  unsigned long long key[kPer];
  int slot[kPer];
#pragma unroll
  for (int m = 0; m < kPer; m++) {
    const int k = tid + m * kSortBins;
    if (k < cnt) {
      key[m] = keys[st + k];
      slot[m] = atomicAdd(&bin_cnt[bin_of(key[m])], 1);
    }
  }
  __syncthreads();
  const int n = bin_cnt[tid];
  int x = n;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(x, off, 64);
    if (lane >= off) x += y;
  }
  if (lane == 63) wsum[wave] = x;
  __syncthreads();
  for (int w = 0; w < wave; w++) x += wsum[w];
  bin_start[tid] = x - n;
  if (tid == kSortBins - 1) bin_start[kSortBins] = x;
  __syncthreads();
#pragma unroll
  for (int m = 0; m < kPer; m++)
    if (tid + m * kSortBins < cnt) sh[bin_start[bin_of(key[m])] + slot[m]] = key[m];
  __syncthreads();
#pragma unroll
  for (int m = 0; m < kPer; m++)
    if (tid + m * kSortBins < cnt) {
      const int b = bin_of(key[m]), b0 = bin_start[b], b1 = bin_start[b + 1];
      int r = b0;
      for (int k = b0; k < b1; k++) r += sh[k] < key[m] ? 1 : 0;
      const int a = (int)(unsigned)(key[m] & 0xffffffffull), loc = cs * kCell + r;
      loc2glo[loc] = a;
      glo2loc[a] = loc;
    }
  for (int k = cnt + tid; k < ncl * kCell; k += kSortBins) loc2glo[cs * kCell + k] = -1;
}

// Per-step gather of xyzq into cell order as 32-bit fixed-point coordinates
// (setSortedCoords, src/CudaPMEDirectForce.cu:1389-1400), fused with the
// clear of the sorted force buffer and the cell bounding boxes (centre and
// half extent in A of the fixed-point coordinates, and the cell's atoms in the
// centre's w; the list build and the spread read them).  A block of 256 slots covers 8 whole cells, so each
// cell's box is a reduction over one half wave.
__device__ __forceinline__ void sort_coords_body(int bid, const float4 *__restrict__ xyzq,
                                                 const int *__restrict__ vdwtype,
                                                 const int *__restrict__ loc2glo,
                                                 const int *__restrict__ meta, double3 inv_len,
                                                 float qscale, float3 unit,
                                                 int4 *__restrict__ posq,
                                                 int *__restrict__ type_s,
                                                 int64_t *__restrict__ fsort, int ss,
                                                 float4 *__restrict__ bb,
                                                 int64_t *__restrict__ force, size_t nforce,
                                                 int nb) {
  const int loc = bid * 256 + threadIdx.x;
  // the step's gradient starts from zero (every term adds into it after the sort)
  if (force)
    for (size_t k = loc; k < nforce; k += (size_t)nb * 256) force[k] = 0;
  const int ncell = meta[0];
  const bool in = loc < ncell * kCell;
  const int g = in ? loc2glo[loc] : -1;
  int4 o = make_int4(0, 0, 0, 0);
  int ty = 0;
  if (g >= 0) {
    float4 p = xyzq[g];
    o.x = (int)to_fixed((double)p.x, inv_len.x);
    o.y = (int)to_fixed((double)p.y, inv_len.y);
    o.z = (int)to_fixed((double)p.z, inv_len.z);
    o.w = __float_as_int(p.w * qscale);
    ty = vdwtype[g];
  }
  if (in) {
    posq[loc] = o;
    type_s[loc] = ty;
    fsort[loc] = 0;
    fsort[ss + loc] = 0;
    fsort[2 * (size_t)ss + loc] = 0;
  }
  const bool valid = g >= 0;
  const float x = (float)(uint32_t)o.x * unit.x, y = (float)(uint32_t)o.y * unit.y,
              z = (float)(uint32_t)o.z * unit.z;
  float mnx = valid ? x : 3e38f, mny = valid ? y : 3e38f, mnz = valid ? z : 3e38f;
  float mxx = valid ? x : -3e38f, mxy = valid ? y : -3e38f, mxz = valid ? z : -3e38f;
  for (int off = 16; off > 0; off >>= 1) {
    mnx = fminf(mnx, __shfl_xor(mnx, off));
    mny = fminf(mny, __shfl_xor(mny, off));
    mnz = fminf(mnz, __shfl_xor(mnz, off));
    mxx = fmaxf(mxx, __shfl_xor(mxx, off));
    mxy = fmaxf(mxy, __shfl_xor(mxy, off));
    mxz = fmaxf(mxz, __shfl_xor(mxz, off));
  }
  const int cell = loc >> 5;
  const int filled = __popc((uint32_t)(__ballot(valid) >> (threadIdx.x & 32)));
  if (cell < ncell && (loc & 31) == 0) {
    bb[2 * cell] = make_float4(0.5f * (mnx + mxx), 0.5f * (mny + mxy), 0.5f * (mnz + mxz),
                               (float)filled);
    bb[2 * cell + 1] = make_float4(0.5f * (mxx - mnx), 0.5f * (mxy - mny), 0.5f * (mxz - mnz), 0.f);
  }
}
// with_fin: the last block runs an integrator's pending kinetic-energy
// reduction instead (thermo.hpp)
__global__ __launch_bounds__(256) void k_sort_coords(const float4 *__restrict__ xyzq,
                                                     const int *__restrict__ vdwtype,
                                                     const int *__restrict__ loc2glo,
                                                     const int *__restrict__ meta, double3 inv_len,
                                                     float qscale, float3 unit,
                                                     int4 *__restrict__ posq,
                                                     int *__restrict__ type_s,
                                                     int64_t *__restrict__ fsort, int ss,
                                                     float4 *__restrict__ bb,
                                                     int64_t *__restrict__ force, size_t nforce,
                                                     LtFinArgs fin, int with_fin) {
  const int nsort = gridDim.x - with_fin;
  if ((int)blockIdx.x >= nsort) {
    lt_finalize_body(fin.part, fin.npart, fin.ndof, fin.thermo, fin.counters, fin.dpart, fin.meta,
                     fin.hdisp, fin.pend);
    return;
  }
  sort_coords_body(blockIdx.x, xyzq, vdwtype, loc2glo, meta, inv_len, qscale, unit, posq, type_s,
                   fsort, ss, bb, force, nforce, nsort);
}
__global__ __launch_bounds__(256) void kb_sort_coords(const SortArgs *__restrict__ tab,
                                                      const int *__restrict__ bstart, int nsys) {
  const int s = batch_system(bstart, nsys);
  const SortArgs a = tab[s];
  sort_coords_body(blockIdx.x - bstart[s], a.xyzq, a.vdwtype, a.loc2glo, a.meta, a.inv_len, 1.0f,
                   a.unit, a.posq, a.type_s, a.fsort, a.ss, a.bb, a.force, a.nforce,
                   bstart[s + 1] - bstart[s]);
}

// Squared gap of two boxes (centre, half extent) in their closest images.
__device__ __forceinline__ float bb_gap2(float4 ci, float4 hi, float4 cj, float4 hj, float3 L,
                                         float3 inv_L) {
  float d2 = 0.f;
  float d, g;
  d = ci.x - cj.x; d -= L.x * rintf(d * inv_L.x); g = fmaxf(fabsf(d) - hi.x - hj.x, 0.f); d2 += g * g;
  d = ci.y - cj.y; d -= L.y * rintf(d * inv_L.y); g = fmaxf(fabsf(d) - hi.y - hj.y, 0.f); d2 += g * g;
  d = ci.z - cj.z; d -= L.z * rintf(d * inv_L.z); g = fmaxf(fabsf(d) - hi.z - hj.z, 0.f); d2 += g * g;
  return d2;
}

// 6. Tiles, masks and entries of one i-cell per block:
//   a. candidate tiles: cells j >= i whose boxes are within the list cutoff,
//      in j order.
//   b. per tile the 32x32 mask: bit t of lane l's word set <=> the pair (i-cell
//      atom t, j-cell atom l) is skipped: padding, diagonal i >= j, topological
//      exclusion (1-2/1-3/1-4), or farther than the list cutoff at build time.
//   c. per i-group (kGroup consecutive slots) the j slots with at least one
//      live pair, packed in tile and slot order with their skip bits, and null
//      entries (full skip mask on the first tile) up to whole 64-lane steps.
// The cell takes its places in cand_j and ent with two atomics, so no count
// pass and no scan come between a, b and c, and the masks stay in LDS
// (cand_mask holds those of a cell with more than kLdsTiles tiles).  Where a
// cell's places lie differs from run to run; what stands there does not.
// The distance test is the work (1024 pairs per tile, 90 tiles per cell in
// water with a 14 A list): r^2 - rl^2 = |i|^2 - 2 i.j + |j|^2 - rl^2 relative
// to the cell's centre comes from two FP32 32x32x2 matrix instructions per
// tile, and the sign bits are the mask; 16 sign and 8 min instructions per
// lane instead of 12 per pair.  A tile with a pair whose value is within the
// rounding of these sums (eps) is tested pair by pair instead, so the mask is
// that of the pairwise test, bit for bit; so is every tile of a box too small
// for one image per cell (list cutoff + half the cell > half the box).
// The exclusions of the cell's atoms stand in an LDS table by partner cell
// (read per j atom and tile from memory they were a chain of four loads).
// One block of eight waves per cell, tiles split evenly; up to 80 registers,
// so three cells per CU hide each other's chains of loads and atomics (about
// half of a cell's 20 us).  89 us at 94k atoms, 24 at 12k; as separate count,
// emit, mask, count and emit passes with two scans between them 173 and 83.
constexpr int kTileWaves = 8;
constexpr int kScanWords = 64 * kTileWaves;  // 64-cell words per sweep of step a
constexpr int kLdsTiles = 192;
constexpr int kExclSlots = 64;  // partner cells of one cell's exclusions (power of two)
// a tile in LDS: j cell (26 bits: 2^31 slots), its atoms - 1, exclusions with it
constexpr uint32_t kTileCell = (1u << 26) - 1u, kTileExcl = 1u << 31;
using f32x16 = __attribute__((ext_vector_type(16))) float;

struct TileArgs {
  const float4 *bb;
  const int4 *posq;
  const int *loc2glo, *glo2loc, *excl_ptr, *excl_idx;
  float3 L, inv_L, unit, inv_unit;
  float rl, rl2, rl2u;  // list cutoff, its square, its square in fixed-point units
  int iso;              // cubic box: the pairwise test compares in fixed-point units
  int *cand_j, *icell_start, *grp_cnt, *grp_start;
  uint32_t *cand_mask, *ent;
  int cand_cap, ent_cap;
};

// Slot of cell jc in the table of exclusion partners, or -1.
__device__ __forceinline__ int excl_slot(const int *ex_cell, int jc) {
  int s = jc & (kExclSlots - 1);
#pragma unroll 1
  for (int probe = 0; probe < kExclSlots; probe++, s = (s + 1) & (kExclSlots - 1)) {
    const int c = ex_cell[s];
    if (c == jc) return s;
    if (c == -1) return -1;
  }
  return -1;
}

__global__ __launch_bounds__(64 * kTileWaves, 6) void k_tiles(int *__restrict__ meta,
                                                           const TileArgs A) {
  constexpr uint32_t kFull = (1u << kGroup) - 1u;
  __shared__ uint32_t sh_tile[kMaxCellTiles];
  union Work {
    struct {
      unsigned long long word[kScanWords];
      int off[kScanWords];
    } s;
    uint32_t mask[kLdsTiles * kCell];
  };
  __shared__ Work sh;
  __shared__ int ex_cell[kExclSlots];
  __shared__ uint32_t ex_mask[kExclSlots][kCell];
  __shared__ int4 sh_pi[kCell];
  __shared__ int sh_cnt[kTileWaves][kGroupsPerCell], sh_base[1 + kGroupsPerCell];
  __shared__ int ex_any, ex_over;

  const int ic = blockIdx.x;
  const int ncell = meta[0];
  if (ic >= ncell) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l = lane & (kCell - 1), half = lane / kCell;
  const unsigned long long below = (1ull << lane) - 1ull;
  const float4 ci = A.bb[2 * ic], hi = A.bb[2 * ic + 1];

  if (tid == 0) ex_any = ex_over = 0;
  if (tid < kExclSlots) ex_cell[tid] = -1;
  for (int k = tid; k < kExclSlots * kCell; k += 64 * kTileWaves) (&ex_mask[0][0])[k] = 0;
  const int4 pi = A.posq[ic * kCell + l];
  const int gi = A.loc2glo[ic * kCell + l];
  if (tid < kCell) sh_pi[tid] = pi;
  __syncthreads();

  // excluded partners: sixteen threads per atom
  if (gi >= 0) {
    const int e1 = A.excl_ptr[gi + 1];
    for (int x = A.excl_ptr[gi] + tid / kCell; x < e1; x += 2 * kTileWaves) {
      const int lp = A.glo2loc[A.excl_idx[x]];
      const int jc = lp / kCell;
      if (jc < ic) continue;  // the partner's cell holds that pair
      ex_any = 1;
      int s = jc & (kExclSlots - 1), probe = 0;
#pragma unroll 1
      for (; probe < kExclSlots; probe++, s = (s + 1) & (kExclSlots - 1)) {
        const int old = atomicCAS(&ex_cell[s], -1, jc);
        if (old == -1 || old == jc) break;
      }
      if (probe < kExclSlots) atomicOr(&ex_mask[s][lp & (kCell - 1)], 1u << l);
      else ex_over = 1;
    }
  }

  // a. candidate tiles
  int n = 0;
  for (int seg = ic; seg < ncell; seg += 64 * kScanWords) {
    const int nw = min(kScanWords, (ncell - seg + 63) / 64);
#pragma unroll 4
    for (int w = wave; w < nw; w += kTileWaves) {
      const int j = seg + 64 * w + lane, jr = min(j, ncell - 1);
      const bool hit = bb_gap2(ci, hi, A.bb[2 * jr], A.bb[2 * jr + 1], A.L, A.inv_L) < A.rl2;
      const unsigned long long b = __ballot(hit && j < ncell);
      if (lane == 0) sh.s.word[w] = b;
    }
    __syncthreads();
    const int c = tid < nw ? __popcll(sh.s.word[tid]) : 0;
    int x = c;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int y = __shfl_up(x, off, 64);
      if (lane >= off) x += y;
    }
    if (lane == 63) sh_cnt[wave][0] = x;
    __syncthreads();
    int before = n;
    for (int w = 0; w < kTileWaves; w++) {
      if (w < wave) before += sh_cnt[w][0];
      n += sh_cnt[w][0];
    }
    sh.s.off[tid] = before + x - c;
    __syncthreads();
    for (int w = wave; w < nw; w += kTileWaves) {
      const unsigned long long b = sh.s.word[w];
      const int pos = sh.s.off[w] + __popcll(b & below);
      if (((b >> lane) & 1ull) && pos < kMaxCellTiles) {
        const int j = seg + 64 * w + lane;
        bool ex = ex_over != 0;
        if (ex_any && !ex) ex = excl_slot(ex_cell, j) >= 0;
        sh_tile[pos] = (uint32_t)j | ((uint32_t)max((int)A.bb[2 * j].w - 1, 0) << 26) |
                       (ex ? kTileExcl : 0u);
      }
    }
    __syncthreads();
  }
  const int g0 = ic * kGroupsPerCell;
  if (n > kMaxCellTiles) {
    // the entry format indexes at most kMaxCellTiles tiles per cell: the list
    // is emptied and the host raises
    if (tid == 0) {
      atomicOr(&meta[7], 1);
      atomicAdd(&meta[1], n);
      A.icell_start[ic] = 0;
    }
    if (tid < kGroupsPerCell) A.grp_cnt[g0 + tid] = A.grp_start[g0 + tid] = 0;
    return;
  }
  // the place among the candidates is asked for here and needed after b
  // (before it by a cell whose masks go to memory)
  int got = 0;
  if (tid == 0) got = atomicAdd(&meta[1], n);
  const bool lds = n <= kLdsTiles;
  bool keep = true;
  uint16_t *mbuf = reinterpret_cast<uint16_t *>(sh.mask);
  if (!lds) {
    if (tid == 0) sh_base[0] = got;
    __syncthreads();
    keep = sh_base[0] + n <= A.cand_cap;
    mbuf = reinterpret_cast<uint16_t *>(A.cand_mask + (size_t)sh_base[0] * kCell);
  }

  // b. masks; lane (half h, l) forms the 16 bits of group h and j slot l
  const unsigned cx = (unsigned)(ci.x * A.inv_unit.x), cy = (unsigned)(ci.y * A.inv_unit.y),
                 cz = (unsigned)(ci.z * A.inv_unit.z);
  // one image of every j serves the whole cell (margins far above rounding)
  const bool one_image = A.rl + hi.x + 0.01f < 0.5f * A.L.x && A.rl + hi.y + 0.01f < 0.5f * A.L.y &&
                         A.rl + hi.z + 0.01f < 0.5f * A.L.z;
  // |D - exact| < 16 roundings of the sum of its terms' sizes, (|i| + |j|)^2 +
  // rl^2 with |j| <= rl + |i| for a pair near the cutoff; twice that is used
  const float di = sqrtf(hi.x * hi.x + hi.y * hi.y + hi.z * hi.z) + 0.01f;
  const float eps = 2e-6f * ((2.f * di + A.rl) * (2.f * di + A.rl) + A.rl2);
  float a1, a2;
  f32x16 C;
  {
    const float x = (float)(int)((unsigned)pi.x - cx) * A.unit.x,
                y = (float)(int)((unsigned)pi.y - cy) * A.unit.y,
                z = (float)(int)((unsigned)pi.z - cz) * A.unit.z;
    a1 = -2.f * (half ? y : x);
    a2 = half ? 1.f : -2.f * z;
    const float c = x * x + y * y + z * z - A.rl2;
#pragma unroll
    for (int r = 0; r < 16; r++) C[r] = __shfl(c, 8 * (r / 4) + 4 * half + (r & 3), 64);
  }
  const uint32_t ipad = (uint32_t)__ballot(gi < 0);  // bit t: i slot t is padding
  const bool excl_mem = ex_over != 0;
  const int per = (n + kTileWaves - 1) / kTileWaves;
  const int k0 = min(wave * per, n), k1 = min(k0 + per, n);
  int cnt0 = 0, cnt1 = 0;
  // the next tile's coordinates load while this one is tested; the tile is the
  // same for the whole wave, so its address and flags are scalar
  uint32_t t_n = 0;
  int4 pj_n = make_int4(0, 0, 0, 0);
  auto load = [&](int k) {
    t_n = (uint32_t)__builtin_amdgcn_readfirstlane((int)sh_tile[k]);
    pj_n = (A.posq + (size_t)(t_n & kTileCell) * kCell)[l];
  };
  if (k0 < k1) load(k0);
  for (int k = k0; k < k1; k++) {
    const uint32_t t = t_n;
    const int jc = (int)(t & kTileCell);
    const int4 pj = pj_n;
    if (k + 1 < k1) load(k + 1);
    uint32_t m = 0;
    bool pairwise = !one_image;
    if (one_image) {
      const float x = (float)(int)((unsigned)pj.x - cx) * A.unit.x,
                  y = (float)(int)((unsigned)pj.y - cy) * A.unit.y,
                  z = (float)(int)((unsigned)pj.z - cz) * A.unit.z;
      f32x16 D = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, half ? y : x, C, 0, 0, 0);
      D = __builtin_amdgcn_mfma_f32_32x32x2f32(a2, half ? x * x + y * y + z * z : z, D, 0, 0, 0);
      // D[r] is i slot 8 (r / 4) + 4 half + r % 4
      float near = 3e38f;
      uint32_t in = 0;
#pragma unroll
      for (int r = 15; r >= 0; r--) {
        in = __builtin_amdgcn_alignbit(in, __float_as_uint(D[r]), 31);
        near = fminf(near, fabsf(D[r]));
      }
      in = (in | (in << 8)) & 0x00ff00ffu;
      in = ((in | (in << 4)) & 0x0f0f0f0fu) << (4 * half);
      in |= (uint32_t)__shfl_xor((int)in, 32, 64);
      m = ~in >> (kGroup * half);
      pairwise = __any(near < eps);
    }
    if (pairwise) {
      m = 0;
#pragma unroll 4
      for (int t = 0; t < kGroup; t++) {
        const int4 p = sh_pi[kGroup * half + t];
        const int ix = p.x - pj.x, iy = p.y - pj.y, iz = p.z - pj.z;
        const float ux = A.iso ? 1.f : A.unit.x, uy = A.iso ? 1.f : A.unit.y,
                    uz = A.iso ? 1.f : A.unit.z;
        const float dx = (float)ix * ux, dy = (float)iy * uy, dz = (float)iz * uz;
        if (dx * dx + dy * dy + dz * dz > (A.iso ? A.rl2u : A.rl2)) m |= 1u << t;
      }
    }
    m |= ipad >> (kGroup * half);
    if (jc == ic) m |= ~((1u << l) - 1u) >> (kGroup * half);
    if (t & kTileExcl) {
      uint32_t skip = 0;
      if (!excl_mem) {
        skip = ex_mask[excl_slot(ex_cell, jc)][l];
      } else {
        const int gj = A.loc2glo[jc * kCell + l];
        if (gj >= 0)
          for (int x = A.excl_ptr[gj]; x < A.excl_ptr[gj + 1]; x++) {
            const int lp = A.glo2loc[A.excl_idx[x]];
            if (lp / kCell == ic) skip |= 1u << (lp & (kCell - 1));
          }
      }
      m |= skip >> (kGroup * half);
    }
    // the cell's empty slots are its last
    m = l > (int)((t >> 26) & 31u) ? kFull : m & kFull;
    const unsigned long long b = __ballot(m != kFull);
    cnt0 += __popc((uint32_t)b);
    cnt1 += __popc((uint32_t)(b >> 32));
    if (keep) mbuf[((size_t)k * kCell + l) * 2 + half] = (uint16_t)m;
  }
  if (lane == 0) {
    sh_cnt[wave][0] = cnt0;
    sh_cnt[wave][1] = cnt1;
  }
  if (tid == 0) sh_base[0] = got;
  __syncthreads();

  // c. candidates and entries; what does not fit is counted, not written
  const int base = sh_base[0];
  const bool cand_ok = base + n <= A.cand_cap;
  if (cand_ok)
    for (int k = tid; k < n; k += 64 * kTileWaves) A.cand_j[base + k] = sh_tile[k] & kTileCell;
  int total[kGroupsPerCell] = {0, 0}, first[kGroupsPerCell] = {0, 0};
  for (int w = 0; w < kTileWaves; w++)
    for (int h = 0; h < kGroupsPerCell; h++) {
      if (w < wave) first[h] += sh_cnt[w][h];
      total[h] += sh_cnt[w][h];
    }
  const int pad0 = (total[0] + 63) / 64 * 64, pad1 = (total[1] + 63) / 64 * 64;
  if (tid == 0) {
    const int e = atomicAdd(&meta[2], pad0 + pad1);
    sh_base[1] = e;
    A.icell_start[ic] = base;
    A.grp_start[g0] = e;
    A.grp_start[g0 + 1] = e + pad0;
    A.grp_cnt[g0] = pad0;
    A.grp_cnt[g0 + 1] = pad1;
  }
  __syncthreads();
  const int ebase = sh_base[1];
  if (!cand_ok || ebase + pad0 + pad1 > A.ent_cap) return;
  const int start = half ? ebase + pad0 : ebase;
  int pos = start + (half ? first[1] : first[0]);
  const uint32_t below_l = (1u << l) - 1u;
#pragma unroll 2
  for (int k = k0; k < k1; k++) {
    const uint32_t m = mbuf[((size_t)k * kCell + l) * 2 + half];
    const bool live = m != kFull;
    const unsigned long long b = __ballot(live);
    const uint32_t bh = half ? (uint32_t)(b >> 32) : (uint32_t)b;
    if (live) A.ent[pos + __popc(bh & below_l)] = (uint32_t)(k << 5 | l) | (m << 16);
    pos += __popc(bh);
  }
  if (wave < kGroupsPerCell) {
    const int s = wave ? ebase + pad0 : ebase;
    const int p = s + (wave ? total[1] : total[0]) + lane;
    if (p < s + (wave ? pad1 : pad0)) A.ent[p] = kFull << 16;
  }
}

// List pruning (no counterpart in the reference; the idea of GROMACS's
// dynamic pruning).  Between builds, every K steps, each group's entries of
// the build's list are tested against the current coordinates with the
// radius r_p = r_off + (cutnb - r_off) K / nbfreq, which assumes the same
// largest relative motion per step as the build's own buffer; pairs beyond
// r_p gain their skip bit, entries left with no live pair are dropped, the
// rest are packed to the front of the group's region of ent_p (same region
// as in ent, null padding after them) and the group's items are shortened.
// Every index stays inside the group's region, so an item that becomes
// empty still points at valid entries.  One wave per group.
__global__ __launch_bounds__(64 * kGroupsPerCell) void k_prune(
    const int *__restrict__ meta, const int *__restrict__ icell_start,
    const int *__restrict__ grp_start, const int *__restrict__ grp_cnt,
    const int *__restrict__ grp_itemstart, const int *__restrict__ cand_j,
    const int4 *__restrict__ posq, const uint32_t *__restrict__ ent, const int4 *__restrict__ items, float3 unit, float rp2,
    uint32_t *__restrict__ ent_p, int4 *__restrict__ items_p) {
  constexpr uint32_t kFull = (1u << kGroup) - 1u;
  const int icell = blockIdx.x;
  if (icell >= meta[0] || meta[8]) return;
  const int lane = threadIdx.x & 63, h = threadIdx.x >> 6;
  const int g = icell * kGroupsPerCell + h;
  const int st = grp_start[g], en = st + grp_cnt[g];
  const int *tiles = cand_j + icell_start[icell];
  const int4 pil = posq[g * kGroup + (lane & (kGroup - 1))];
  unsigned pix[kGroup], piy[kGroup], piz[kGroup];
#pragma unroll
  for (int k = 0; k < kGroup; k++) {
    pix[k] = (unsigned)__builtin_amdgcn_readlane(pil.x, k);
    piy[k] = (unsigned)__builtin_amdgcn_readlane(pil.y, k);
    piz[k] = (unsigned)__builtin_amdgcn_readlane(pil.z, k);
  }
  const unsigned long long below = (1ull << lane) - 1ull;
  int run = 0;
  // the next chunk's entry and j coordinates load while this one is tested
  auto jpos = [&](uint32_t e) { return posq[tiles[(e & 0xffffu) >> 5] * kCell + (int)(e & 31u)]; };
  uint32_t e_n = st < en ? ent[st + lane] : 0u;
  int4 pj_n = st < en ? jpos(e_n) : make_int4(0, 0, 0, 0);
  for (int p0 = st; p0 < en; p0 += 64) {  // en - st is a multiple of 64
    const uint32_t e = e_n;
    const int4 pj = pj_n;
    if (p0 + 64 < en) {
      e_n = ent[p0 + 64 + lane];
      pj_n = jpos(e_n);
    }
    uint32_t m = e >> 16;
#pragma unroll
    for (int k = 0; k < kGroup; k++) {
      const float dx = (float)(int)(pix[k] - (unsigned)pj.x) * unit.x;
      const float dy = (float)(int)(piy[k] - (unsigned)pj.y) * unit.y;
      const float dz = (float)(int)(piz[k] - (unsigned)pj.z) * unit.z;
      if (!(dx * dx + dy * dy + dz * dz < rp2)) m |= 1u << k;
    }
    const bool live = m != kFull;
    const unsigned long long b = __ballot(live);
    if (live) ent_p[st + run + __popcll(b & below)] = (e & 0xffffu) | (m << 16);
    run += __popcll(b);
  }
  for (int p = st + run + lane; p < en; p += 64) ent_p[p] = kFull << 16;
  const int end = st + (run + 63) / 64 * 64;
  for (int it = grp_itemstart[g] + lane; it < grp_itemstart[g + 1]; it += 64) {
    int4 q = items[it];
    q.z = max(q.y, min(q.z, end));
    items_p[it] = q;
  }
}

void nblist_prune(NbSystem &S, hipStream_t s) {
  const float3 unit = make_float3((float)(S.box[0] / 4294967296.0), (float)(S.box[1] / 4294967296.0),
                                  (float)(S.box[2] / 4294967296.0));
  k_prune<<<S.ncell_cap, 64 * kGroupsPerCell, 0, s>>>(
      S.meta.get(), S.icell_start.get(), S.grp_start.get(), S.grp_cnt.get(),
      S.grp_itemstart.get(), S.cand_j.get(), S.posq.get(), S.ent.get(), S.items.get(), unit, S.prune_r2, S.ent_p.get(),
      S.items_p.get());
  APO_LAUNCH_CHECK();
}

// 7. Work items of <= isteps 64-entry steps, their processing order, and the
// build's counts (one block).  A group's items are full ones and one shorter
// remainder, in group order.  The order for the pair kernel is by step count,
// longest first, items of one length in index order: its blocks take items in
// this order, so the items still running when the launch drains are short
// ones (list scheduling, longest processing time first).  order[p] = item
// index.  Each wave counts the lengths of its own contiguous groups; with the
// other waves' counts it then knows the place of each of its items, so the
// block meets only once: 15 us at 94k atoms and 9 at 12k, after 33 and 21 for
// two scans, the export and a pass over the items in three barriers per 1024.
// Any capacity overflow or input error leaves the list empty (no pair kernel
// work, no out-of-range write) and sets meta[8]; the build's counts and flags
// go to pinned host memory with the running build number in slot 15
// (meta[16] survives the per-build clear), where the host learns of errors
// and growth.
constexpr int kItemThreads = 1024;
__global__ __launch_bounds__(kItemThreads) void k_list_guard_export(
    int *__restrict__ meta, int cand_cap, int ent_cap, int item_cap, int *__restrict__ host,
    const int *__restrict__ grp_cnt, const int *__restrict__ grp_start,
    const int *__restrict__ icell_start, int *__restrict__ grp_itemstart,
    int4 *__restrict__ items, int *__restrict__ order, int isteps) {
  constexpr int kW = kItemThreads / 64;
  static_assert(kItemSteps < 64 && (kItemSteps & (kItemSteps - 1)) == 0,
                "one lane per item length from 0 to kItemSteps, lengths compared bit by bit");
  __shared__ int sh_hist[kW][64];  // [wave][length]; length isteps: the full items
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const unsigned long long below = (1ull << lane) - 1ull;
  const int ngrp = meta[0] * kGroupsPerCell;
  const int per = (ngrp + kItemThreads - 1) / kItemThreads * 64;
  const int gb = min(wave * per, ngrp), ge = min(gb + per, ngrp);
  sh_hist[wave][lane] = 0;
  int full = 0;  // full items of the lane's groups
#pragma unroll 4
  for (int g = gb + lane; g - lane < ge; g += 64) {
    const int c = grp_cnt[min(g, ge - 1)], steps = g < ge ? c / 64 : 0;
    full += steps / isteps;
    atomicAdd(&sh_hist[wave][steps % isteps], 1);
  }
  for (int off = 32; off > 0; off >>= 1) full += __shfl_xor(full, off, 64);
  if (lane == 0) {
    sh_hist[wave][0] = 0;
    sh_hist[wave][isteps] = full;
  }
  __syncthreads();
  // lane L: items of length L in all waves and in the waves before this one
  int all = 0, prev = 0;
  for (int w = 0; w < kW; w++) {
    const int h = sh_hist[w][lane];
    if (w < wave) prev += h;
    all += h;
  }
  int longer = all, item0 = prev;  // sums over the lanes: from L up; every length
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_down(longer, off, 64);
    if (lane + off < 64) longer += y;
    item0 += __shfl_xor(item0, off, 64);
  }
  const int nitem = __shfl(longer, 0, 64);
  __shared__ int sh_run[kW][64];  // next place in the order for length L
  sh_run[wave][lane] = longer - all + prev;
  int run_full = __shfl(longer - all + prev, isteps, 64);
  const bool over = meta[1] > cand_cap || meta[2] > ent_cap || nitem > item_cap;
  const bool bad = over || meta[5] || meta[6] || meta[7];
  if (!bad)
#pragma unroll 2
    for (int g = gb + lane; g - lane < ge; g += 64) {
      const int gr = min(g, ge - 1);
      const int c = grp_cnt[gr], a = grp_start[gr], tile0 = icell_start[gr / kGroupsPerCell];
      const int steps = g < ge ? c / 64 : 0;
      const int nf = steps / isteps, rem = steps % isteps;
      int x = nf;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
      }
      const unsigned long long tails = __ballot(rem > 0);
      const int item = item0 + x - nf + __popcll(tails & below);
      // the wave's 64 groups with the same remainder (isteps: power of two)
      unsigned long long peers = ~0ull;
      for (int bit = 1; bit < isteps; bit <<= 1) {
        const unsigned long long b = __ballot(rem & bit);
        peers &= rem & bit ? b : ~b;
      }
      const int nfull = __shfl(x, 63, 64);
      const int place_f = run_full + x - nf;
      const int next = sh_run[wave][rem], place = next + __popcll(peers & below);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if (!(peers & below)) sh_run[wave][rem] = next + __popcll(peers);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if (g < ge) {
        grp_itemstart[g] = item;
        for (int m = 0; m < nf; m++) {
          items[item + m] = make_int4(g, a + m * 64 * isteps, a + (m + 1) * 64 * isteps, tile0);
          order[place_f + m] = item + m;
        }
        if (rem) {
          items[item + nf] = make_int4(g, a + nf * 64 * isteps, a + steps * 64, tile0);
          order[place] = item + nf;
        }
      }
      run_full += nfull;
      item0 += nfull + __popcll(tails);
    }
  if (tid != kItemThreads - 64) return;  // the last wave has the fewest groups
  grp_itemstart[ngrp] = nitem;
  meta[3] = nitem;
  int m[15];
  for (int k = 0; k < 15; k++) m[k] = meta[k];
  if (bad) {
    m[8] = meta[8] = over ? 1 : 2;
    m[3] = meta[3] = 0;
  }
  const int seq = meta[16] + 1;
  meta[16] = seq;
  for (int k = 0; k < 15; k++) host[k] = m[k];
  __threadfence_system();
  host[15] = seq;
  __threadfence_system();
}

static inline int nblk(long n, int b) { return (int)((n + b - 1) / b); }

// Host side of the exported counts: errors of a finished build raise here;
// with allow_growth (only right before a rebuild, whose lists replace the
// current ones) capacities that the last finished build used above 85 % grow:
// the device is drained first and captured step graphs see the new
// generation.  Without it a pending growth stays pending for the next check.
void list_export_check(NbSystem &S, hipStream_t s, bool allow_growth) {
  const volatile int *h = S.h_meta;
  if (!h || h[15] == 0) return;
  int m[16];
  for (int k = 0; k < 16; k++) m[k] = h[k];
  if (m[15] == S.meta_checked) return;
  const bool grow = m[1] > 0.85 * S.cand_cap || m[2] > 0.85 * S.ent_cap || m[3] > 0.85 * S.item_cap;
  const bool error = m[5] || m[6] || m[7] || m[8] == 1;
  if (!error && grow && !allow_growth) return;
  S.meta_checked = m[15];
  if (m[6]) throw RuntimeError("non-finite coordinates in xyzq at a neighbor-list rebuild");
  if (m[5]) throw RuntimeError("neighbor list: an xy column exceeds the LDS sort capacity");
  if (m[7]) throw RuntimeError("neighbor list: a cell has more than 2048 candidate tiles");
  if (m[8] == 1)
    throw RuntimeError("neighbor list: a rebuild exceeded the list capacity; the forces of the "
                       "steps after it are invalid (capacity was sized from earlier builds)");
  if (grow) {
    APO_HIP(hipStreamSynchronize(s));
    APO_HIP(hipDeviceSynchronize());
    list_reserve(S, m[1], m[2], m[3]);
  }
}

void list_reserve(NbSystem &S, int ncand, int nent, int nitem) {
  if ((size_t)ncand > S.cand_cap * 0.85 || S.cand_cap == 0) {
    S.cand_cap = (size_t)(ncand * 1.5) + 64;
    S.cand_j.reserve(S.cand_cap);
    S.cand_mask.reserve(S.cand_cap * kCell);
    S.generation++;
  }
  if ((size_t)nent > S.ent_cap * 0.85 || S.ent_cap == 0) {
    S.ent_cap = (size_t)(nent * 1.5) + 64 * kItemSteps;
    S.ent.reserve(S.ent_cap);
    S.ent_p.reserve(S.ent_cap);
    S.generation++;
  }
  if ((size_t)nitem > S.item_cap * 0.85 || S.item_cap == 0) {
    S.item_cap = (size_t)(nitem * 1.5) + 64;
    S.items.reserve(S.item_cap);
    S.items_p.reserve(S.item_cap);
    S.item_order.reserve(S.item_cap);
    S.generation++;
  }
}

// Builds the list from xyzq.  sizing = true synchronises to size the
// buffers exactly and raises input errors at once (the first build and
// apo_nb_reset_list); otherwise the build is host-sync free, guarded by the
// capacities, and its errors surface at the next check of the exported
// counts (so a rebuild can be part of a captured step graph).
// force/nforce go to the coordinate sort; true if that sort, which a sizing
// build leaves to the caller, is the step's own.
bool nblist_build(NbSystem &S, const float4 *x, hipStream_t s, bool sizing, int64_t *force,
                  size_t nforce) {
  const int n = S.natom;
  const double3 inv = make_double3(1.0 / S.box[0], 1.0 / S.box[1], 1.0 / S.box[2]);
  const double3 len = make_double3(S.box[0], S.box[1], S.box[2]);
  int *meta = S.meta.get();
  sizing = sizing || S.cand_cap == 0 || S.ent_cap == 0 || S.item_cap == 0;
  if (sizing && !S.may_allocate)
    throw InvalidArgument("the neighbor list has no capacity yet: build it once with an "
                          "allocating call (apo_nb_reset_list or apo_nb_calc_force)");
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  APO_HIP(hipStreamIsCapturing(s, &cap));
  if (sizing && cap != hipStreamCaptureStatusNone)
    throw RuntimeError("the first neighbor-list build cannot be captured in a graph");
  if (!sizing && cap == hipStreamCaptureStatusNone) list_export_check(S, s, S.may_allocate);

  k_list_clear<<<nblk(std::max(S.ncol + 1, 16), 256), 256, 0, s>>>(meta, S.col_count.get(),
                                                                   S.ncol);
  APO_LAUNCH_CHECK();
  k_assign<<<nblk(n, 256), 256, 0, s>>>(x, n, inv, len, S.ncx, S.ncy, S.col_count.get(),
                                         S.atom_col.get(), S.atom_slot.get(), S.zkey.get(), meta,
                                         S.xref.get());
  APO_LAUNCH_CHECK();
  k_col_scan<<<2, kScanThreads, 0, s>>>(S.col_count.get(), S.ncol, S.col_start.get(),
                                        S.col_cellstart.get(), meta);
  APO_LAUNCH_CHECK();
  unsigned long long *kb = S.colkeys.get();
  k_scatter<<<nblk(n, 256), 256, 0, s>>>(n, S.atom_col.get(), S.atom_slot.get(), S.col_start.get(),
                                          S.zkey.get(), kb);
  APO_LAUNCH_CHECK();
  k_colsort<<<S.ncol, kSortBins, 0, s>>>(kb, S.col_count.get(), S.col_start.get(),
                                         S.col_cellstart.get(), (float)(kSortBins / S.box[2]),
                                         S.loc2glo.get(), S.glo2loc.get(), meta);
  APO_LAUNCH_CHECK();
  // also the cell boxes
  nblist_sort_coords(S, x, s, sizing ? nullptr : force, sizing ? 0 : nforce);
  const double u[3] = {S.box[0] / 4294967296.0, S.box[1] / 4294967296.0, S.box[2] / 4294967296.0};
  TileArgs A;
  A.bb = S.cell_bb.get();
  A.posq = S.posq.get();
  A.loc2glo = S.loc2glo.get();
  A.glo2loc = S.glo2loc.get();
  A.excl_ptr = S.excl_ptr.get();
  A.excl_idx = S.excl_idx.get();
  A.L = make_float3((float)S.box[0], (float)S.box[1], (float)S.box[2]);
  A.inv_L = make_float3((float)inv.x, (float)inv.y, (float)inv.z);
  A.unit = make_float3((float)u[0], (float)u[1], (float)u[2]);
  A.inv_unit = make_float3((float)(1.0 / u[0]), (float)(1.0 / u[1]), (float)(1.0 / u[2]));
  A.rl = (float)S.cutnb;
  A.rl2 = (float)(S.cutnb * S.cutnb);
  A.rl2u = (float)(S.cutnb * S.cutnb / (u[0] * u[0]));
  A.iso = S.box[0] == S.box[1] && S.box[1] == S.box[2];
  A.icell_start = S.icell_start.get();
  A.grp_cnt = S.grp_cnt.get();
  A.grp_start = S.grp_start.get();
  auto tiles = [&] {
    A.cand_j = S.cand_j.get();
    A.cand_mask = S.cand_mask.get();
    A.ent = S.ent.get();
    A.cand_cap = (int)S.cand_cap;
    A.ent_cap = (int)S.ent_cap;
    k_tiles<<<S.ncell_cap, 64 * kTileWaves, 0, s>>>(meta, A);
    APO_LAUNCH_CHECK();
  };
  tiles();
  if (sizing) {
    int hmeta[8];
    std::vector<int> cnt((size_t)S.ncell_cap * kGroupsPerCell);
    APO_HIP(hipMemcpyAsync(hmeta, meta, sizeof(hmeta), hipMemcpyDeviceToHost, s));
    APO_HIP(hipMemcpyAsync(cnt.data(), S.grp_cnt.get(), cnt.size() * sizeof(int),
                           hipMemcpyDeviceToHost, s));
    APO_HIP(hipStreamSynchronize(s));
    if (hmeta[6]) {
      S.list_valid = false;
      throw RuntimeError("non-finite coordinates in xyzq");
    }
    if (hmeta[5]) {
      S.list_valid = false;
      throw RuntimeError("neighbor list: an xy column exceeds the LDS sort capacity");
    }
    if (hmeta[7]) {
      S.list_valid = false;
      throw RuntimeError("neighbor list: a cell has more than 2048 candidate tiles");
    }
    S.host_ncell = hmeta[0];
    S.host_ncand = hmeta[1];
    S.host_nent = hmeta[2];
    if (S.item_steps == 0) {
      // the longest items that still give every other pair-kernel wave one
      // (measured: 98,304 atoms keep 16 steps, 23,558 atoms run faster on 4);
      // a candidate tile holds ~32 live entries, half a 64-entry step
      const double steps = 0.5 * hmeta[1];
      int k = kItemSteps;
      while (k > 2 && steps / k < 0.5 * S.pair_blocks) k /= 2;
      S.item_steps = k;
    }
    S.host_nitem = 0;
    for (int g = 0; g < hmeta[0] * kGroupsPerCell; g++)
      S.host_nitem += (cnt[g] + 64 * S.item_steps - 1) / (64 * S.item_steps);
    const auto gen = S.generation;
    list_reserve(S, hmeta[1], hmeta[2], S.host_nitem);
    if (S.generation != gen) {  // a buffer is new: the counts stand, the list does not
      launch_fill_i32(meta + 1, 2, s);
      tiles();
    }
  }
  if (S.item_steps == 0) S.item_steps = kItemSteps;
  k_list_guard_export<<<1, kItemThreads, 0, s>>>(
      meta, (int)S.cand_cap, (int)S.ent_cap, (int)S.item_cap, S.h_meta, S.grp_cnt.get(),
      S.grp_start.get(), S.icell_start.get(), S.grp_itemstart.get(), S.items.get(),
      S.item_order.get(), S.item_steps);
  APO_LAUNCH_CHECK();
  S.builds_queued++;
  S.list_valid = true;
  return !sizing;
}

void nblist_sort_coords(NbSystem &S, const float4 *x, hipStream_t s, int64_t *force,
                        size_t nforce) {
  const double3 inv = make_double3(1.0 / S.box[0], 1.0 / S.box[1], 1.0 / S.box[2]);
  const float qscale = 1.0f;  // raw charge; ccelec is applied per tile in the pair kernel
  const float3 unit = make_float3((float)(S.box[0] / 4294967296.0), (float)(S.box[1] / 4294967296.0),
                                  (float)(S.box[2] / 4294967296.0));
  const int with_fin = S.sort_fin ? 1 : 0;
  const LtFinArgs fin = S.sort_fin ? *S.sort_fin : LtFinArgs{};
  k_sort_coords<<<nblk(S.ssort, 256) + with_fin, 256, 0, s>>>(
      x, S.vdwtype.get(), S.loc2glo.get(), S.meta.get(), inv, qscale, unit, S.posq.get(),
      S.type_s.get(), S.fsort.get(), S.ssort, S.cell_bb.get(), force, nforce, fin, with_fin);
  APO_LAUNCH_CHECK();
}

// Pairs inside the list cutoff covered by the list (clear skip-mask bits).
__global__ void k_count_pairs(const uint32_t *__restrict__ ent, int nent,
                              unsigned long long *__restrict__ out) {
  size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  unsigned c = 0;
  if (k < (size_t)nent) c = __popc(~(ent[k] >> 16) & ((1u << kGroup) - 1u));
  for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off);
  if ((threadIdx.x & 63) == 0 && c) atomicAdd(out, (unsigned long long)c);
}

void nblist_stats(NbSystem &S, int64_t *out6, hipStream_t s) {
  int hmeta[16];
  APO_HIP(hipMemcpyAsync(hmeta, S.meta.get(), sizeof(hmeta), hipMemcpyDeviceToHost, s));
  APO_HIP(hipStreamSynchronize(s));
  list_export_check(S, s, false);
  const int nent = hmeta[8] ? 0 : std::min(hmeta[2], (int)S.ent_cap);
  DevBuf<unsigned long long> cnt;
  cnt.reserve(1);
  APO_HIP(hipMemsetAsync(cnt.get(), 0, sizeof(unsigned long long), s));
  if (S.list_valid && nent > 0)
    k_count_pairs<<<nblk((long)nent, 256), 256, 0, s>>>(S.ent.get(), nent, cnt.get());
  APO_LAUNCH_CHECK();
  unsigned long long pairs = 0;
  APO_HIP(hipMemcpyAsync(&pairs, cnt.get(), sizeof(pairs), hipMemcpyDeviceToHost, s));
  APO_HIP(hipStreamSynchronize(s));
  out6[0] = hmeta[0];
  out6[1] = hmeta[2];
  out6[2] = hmeta[3];
  out6[3] = (int64_t)pairs;
  out6[4] = S.ncol;
  out6[5] = hmeta[4];
}

// ---- fused launches over several systems ------------------------------------
void batch_add_sort(BatchLaunch<SortArgs> &b, NbSystem &S, const float4 *x, int64_t *force,
                    size_t nforce) {
  SortArgs a{x, S.vdwtype.get(), S.loc2glo.get(), S.meta.get(),
             make_double3(1.0 / S.box[0], 1.0 / S.box[1], 1.0 / S.box[2]),
             make_float3((float)(S.box[0] / 4294967296.0), (float)(S.box[1] / 4294967296.0),
                         (float)(S.box[2] / 4294967296.0)),
             S.posq.get(), S.type_s.get(), S.fsort.get(), S.ssort, S.cell_bb.get(), force,
             nforce};
  b.add(a, nblk(S.ssort, 256));
}
void batch_sort(BatchLaunch<SortArgs> &b, hipStream_t s) {
  if (!b.blocks()) return;
  kb_sort_coords<<<b.blocks(), 256, 0, s>>>(b.d_args.get(), b.d_start.get(), b.nsys());
  APO_LAUNCH_CHECK();
}

}  // namespace apo
