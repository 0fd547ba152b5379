// wf_tiles.hip — LDS-staged neighbour tiles.
//
// A tile is kTileP consecutive particles of the Morton order (one workgroup
// of the pair kernels).  At each rebuild the tile gets:
//   - the sorted set of occupied grid cells adjacent to any of its particles
//     (tile_keys); the particles of those cells (in cell order, ascending
//     particle index within a cell) that are a neighbour of at least one of
//     the tile's particles form the tile's staged set (tile_j, tile_uc
//     entries) — on a cubic lattice with h = 1.2 dx about 740 of the ~1,230
//     particles of the adjacent cells;
//   - for each of its particles, the neighbour list in ascending staged
//     order as 16-bit positions in the staged set, four per 8-byte word,
//     interleaved [(k/4)*npad + i] so a wavefront reads contiguous words (the
//     particle indices are tile_j of those positions).
// The pair kernels write the staged set to LDS (position + index per slot)
// and read a neighbour's position from LDS through its slot.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>

#include "wf_device.hpp"
#include "wf_tiles.hpp"

namespace wf {

constexpr int kSortN = 4096;  // >= kTileP * 27, power of two
static_assert(kTileP * 27 <= kSortN, "sort buffer too small");

// The cell coordinates of a cell key (the inverse of cell_key).
__device__ __forceinline__ void key_cell(const GridDesc& g, int key, int& cx, int& cy, int& cz) {
  const int meta = key >> 9, m = key & 511;
  int x = 0, y = 0, z = 0;
#pragma unroll
  for (int b = 0; b < 3; b++) {
    x |= ((m >> (3 * b)) & 1) << b;
    y |= ((m >> (3 * b + 1)) & 1) << b;
    z |= ((m >> (3 * b + 2)) & 1) << b;
  }
  const int mx = meta % g.mdim[0], myz = meta / g.mdim[0];
  cx = 8 * mx + x;
  cy = 8 * (myz % g.mdim[1]) + y;
  cz = 8 * (myz / g.mdim[1]) + z;
}

// Exclusive prefix of v over the NT threads of the block (wave prefixes by
// shuffles, then the wave totals through LDS); `total` receives the block
// sum.  Every thread of the block must call it.
template <int NT>
__device__ __forceinline__ int block_excl_scan(int v, int* wsum, int& total) {
  constexpr int NW = NT / 64;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int incl = v;
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(incl, d);
    if (lane >= d) incl += o;
  }
  if (lane == 63) wsum[w] = incl;
  __syncthreads();
  int off = 0;
  total = 0;
  for (int u = 0; u < NW; u++) {
    const int t = wsum[u];
    off += u < w ? t : 0;
    total += t;
  }
  __syncthreads();  // wsum may be written again
  return off + incl - v;
}

// Per tile: sorted unique occupied neighbour cells and the staged count.
// After a reorder the tile's particles are in cell order, so its own cells
// are the runs of equal keys; a tile re-listed without a reorder
// (SORT_OWN) first sorts its particles' keys.  Only the tile's few distinct
// cells (typically 10-20) are expanded to their 27 neighbours.
// tiles: the tiles to build (null: block b builds tile b).
template <bool SORT_OWN>
__global__ __launch_bounds__(kTileP) void k_tile_cells(const float* __restrict__ p0,
                                                       const float* __restrict__ p1,
                                                       const float* __restrict__ p2, int n,
                                                       GridDesc g,
                                                       const int* __restrict__ cell_start,
                                                       const int* __restrict__ tiles,
                                                       int* tile_keys, int* tile_nc,
                                                       int* tile_ucnt, int* overflow) {
  __shared__ int keys[kSortN];
  __shared__ int own[kTileP];   // the key of each particle's cell
  __shared__ int ukey[kTileMaxCells];
  __shared__ int blo[3], bdim[3];
  __shared__ int wcnt[kTileP / 64 + 1];
  const int t = tiles ? tiles[blockIdx.x] : blockIdx.x;
  const int tid = threadIdx.x;
  const int i = t * kTileP + tid;
  int cx = 0, cy = 0, cz = 0, kown = INT_MAX;
  if (i < n) {
    cell_of(g, p0[i], p1[i], p2[i], cx, cy, cz);
    kown = cell_key(g, cx, cy, cz);
  }
  own[tid] = kown;
  __syncthreads();
  if constexpr (SORT_OWN) {
    for (int size = 2; size <= kTileP; size <<= 1) {
      for (int stride = size >> 1; stride > 0; stride >>= 1) {
        if (tid < kTileP / 2) {
          const int lo = 2 * tid - (tid & (stride - 1));
          const int hi = lo + stride;
          const bool up = (lo & size) == 0;
          const int a = own[lo], b = own[hi];
          if ((a > b) == up) {
            own[lo] = b;
            own[hi] = a;
          }
        }
        __syncthreads();
      }
    }
    kown = own[tid];
    if (kown != INT_MAX) key_cell(g, kown, cx, cy, cz);
  }
  // first particle of each run of equal cells (keys ascend along the tile)
  const bool first = kown != INT_MAX && (tid == 0 || own[tid - 1] != kown);
  const unsigned long long bal = __ballot(first);
  const int lane = lane_id(), w = tid >> 6;
  if (lane == 0) wcnt[w] = __popcll(bal);
  __syncthreads();
  int wbase = 0;
  for (int u = 0; u < w; u++) wbase += wcnt[u];
  int nown = 0;
  for (int u = 0; u < kTileP / 64; u++) nown += wcnt[u];
  const int rank = wbase + __popcll(bal & ((1ull << lane) - 1ull));
  // the coordinates of the tile's unique cells, in key order
  __shared__ int ocx[kTileP], ocy[kTileP], ocz[kTileP];
  if (first) {
    ocx[rank] = cx;
    ocy[rank] = cy;
    ocz[rank] = cz;
  }
  __syncthreads();
  const int total = 27 * nown;
  int* out = tile_keys + (int64_t)t * kTileMaxCells;
  // the box of cells around the tile's own, one cell wider
  if (tid < 3) {
    const int* oc = tid == 0 ? ocx : tid == 1 ? ocy : ocz;
    int lo = oc[0], hi = oc[0];
    for (int o = 1; o < nown; o++) {
      lo = min(lo, oc[o]);
      hi = max(hi, oc[o]);
    }
    blo[tid] = lo - 1;
    bdim[tid] = hi - lo + 3;
  }
  if (tid == 0) wcnt[kTileP / 64] = 0;
  __syncthreads();
  const int bx = bdim[0], by = bdim[1], bz = bdim[2];
  int run, cnt = 0;
  if ((int64_t)bx * by * bz <= kSortN) {
    // a flag a box cell; the occupied ones' keys in any order; each key's rank
    // among them by counting (they are some hundred, and distinct).  Sorting
    // the candidates, 45 or 55 barriers and two serial sums, took 20 us for 17
    // tiles and 78 us for 5,931, this 7 and 41
    const int vol = bx * by * bz;
    for (int q = tid; q < vol; q += kTileP) keys[q] = 0;
    __syncthreads();
    for (int q = tid; q < total; q += kTileP) {
      const int o = q / 27, r = q - 27 * o;
      const int x = ocx[o] + (r % 3) - 1 - blo[0], y = ocy[o] + ((r / 3) % 3) - 1 - blo[1];
      const int z = ocz[o] + r / 9 - 1 - blo[2];
      keys[(z * by + y) * bx + x] = 1;
    }
    __syncthreads();
    for (int q = tid; q < vol; q += kTileP) {
      if (!keys[q]) continue;
      const int x = blo[0] + q % bx, y = blo[1] + q / bx % by, z = blo[2] + q / (bx * by);
      if (x < 0 || y < 0 || z < 0 || x >= g.dim[0] || y >= g.dim[1] || z >= g.dim[2]) continue;
      const int kk = cell_key(g, x, y, z);
      const int n_in = cell_start[kk + 1] - cell_start[kk];
      if (n_in <= 0) continue;
      const int pos = atomicAdd(&wcnt[kTileP / 64], 1);
      if (pos < kTileMaxCells) ukey[pos] = kk;
      cnt += n_in;
    }
    __syncthreads();
    run = wcnt[kTileP / 64];
    const int m = min(run, kTileMaxCells);
    for (int q = tid; q < m; q += kTileP) {
      const int k = ukey[q];
      int r = 0;
      for (int u = 0; u < m; u++) r += ukey[u] < k;
      out[r] = k;
    }
    __syncthreads();
  } else {
    // a tile whose cells lie far apart: the candidate keys, sorted
    int S = 2;
    while (S < total) S <<= 1;
    for (int q = tid; q < S; q += kTileP) {
      int k = INT_MAX;
      if (q < total) {
        const int o = q / 27, r = q - 27 * o;
        const int x = ocx[o] + (r % 3) - 1, y = ocy[o] + ((r / 3) % 3) - 1, z = ocz[o] + r / 9 - 1;
        if (x >= 0 && y >= 0 && z >= 0 && x < g.dim[0] && y < g.dim[1] && z < g.dim[2]) {
          const int kk = cell_key(g, x, y, z);
          if (cell_start[kk + 1] > cell_start[kk]) k = kk;
        }
      }
      keys[q] = k;
    }
    __syncthreads();
    // bitonic sort of the S candidate keys
    for (int size = 2; size <= S; size <<= 1) {
      for (int stride = size >> 1; stride > 0; stride >>= 1) {
        for (int s2 = tid; s2 < S / 2; s2 += kTileP) {
          int lo = 2 * s2 - (s2 & (stride - 1));
          int hi = lo + stride;
          bool up = ((lo & size) == 0);
          int a = keys[lo], b = keys[hi];
          if ((a > b) == up) {
            keys[lo] = b;
            keys[hi] = a;
          }
        }
        __syncthreads();
      }
    }
    // unique: each thread owns a segment of ceil(S/kTileP) entries
    const int seg = (S + kTileP - 1) / kTileP;
    const int sb0 = min(tid * seg, S), sb1 = min(sb0 + seg, S);
    int c = 0;
    for (int s = sb0; s < sb1; s++) {
      int k = keys[s];
      if (k != INT_MAX && (s == 0 || keys[s - 1] != k)) c++;
    }
    int pos = block_excl_scan<kTileP>(c, wcnt, run);
    for (int s = sb0; s < sb1; s++) {
      int k = keys[s];
      if (k != INT_MAX && (s == 0 || keys[s - 1] != k)) {
        if (pos < kTileMaxCells) {
          out[pos] = k;
          cnt += cell_start[k + 1] - cell_start[k];
        }
        pos++;
      }
    }
  }
  int tot;
  block_excl_scan<kTileP>(cnt, wcnt, tot);
  if (tid == 0) {
    tile_nc[t] = run;
    if (run > kTileMaxCells) atomicAdd(overflow, 1);
    tile_ucnt[t] = tot;
    if (tot > 65535) atomicAdd(overflow, 1);
  }
}

// adjacent-cell sets up to compact_max (at most this, the LDS flag array)
// are compacted to the particles that some list references (larger ones are
// staged whole)
constexpr int kCompactMax = 4096;
// candidate positions held in LDS at a time by the list builder (50 KB with
// the lists, three workgroups a CU)
constexpr int kListStage = 256;

// Neighbour lists in staged order (16-bit slots), and the staged set
// tile_j / tile_uc.  Same float criterion as the reference
// search: 0 < d2 < r2, d2 = dx*dx + dy*dy + dz*dz without contraction, at
// most cap entries (70 as in the reference, 96 with a list skin).  A candidate
// outside the cells around the particle's own cell is more than the 1.01 r
// cell width away, so it never passes the test, and the lists are those of a
// scan over the 27 cells around each particle.  The compaction keeps the order
// of the set, so every list stays in ascending staged order.
//
// The vector ALU bounds it: a tile has ~1,230 candidates for each of its 128
// particles, and 56 pass.  So each wavefront (16 particles, four threads each)
// first keeps the candidates within r of the box around its particles, in
// order, and only those are tested, all lanes of a quarter reading the same
// one (an LDS broadcast).  Lists are built in LDS and written once, whole quads;
// appending to them in memory cost a scattered 2-byte store a neighbour and a
// second pass.  Two threads a particle (32 to a box, two workgroups fewer a
// CU) took 916 us where four take 395.  us a build, before -> now: 17 tiles
// 73 -> 34, 147 tiles 126 -> 51, 1,875 tiles 241 -> 157, 5,931 tiles 578 -> 395.
constexpr int kListLanes = 4;  // threads per particle
constexpr int kListThreads = kListLanes * kTileP;
// 16-bit entries from one particle's list to the next while it is built in LDS:
// the longest list, a multiple of four, and an odd number of 8-byte words so
// that the lanes' entries spread over the banks
constexpr int kRowStride = 100;
static_assert(kListCap <= kRowStride && kRowStride % 4 == 0, "a list fits its row");

// The cell holding staged position q: the last p with spre[p] <= q (an empty
// cell shares its prefix with the next one, so the cell found is never empty).
__device__ __forceinline__ int staged_cell(const int* spre, int nc, int q) {
  int lo = 0, hi = nc - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (spre[mid] <= q) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// p0..p2: the positions of the cell-sorted order (candidates); o0..o2: the
// positions of the tiles' own particles by storage index, and map[s] the
// storage index at sorted position s (both null right after a reorder,
// where the two orders are one).  tiles: the tiles to build (null: all).
// With map, each tile's staged set must fit the region it was given at the
// last reorder; a tile whose set does not raises *overflow.
__global__ __launch_bounds__(kListThreads) void k_tile_lists(
    const float* __restrict__ p0, const float* __restrict__ p1, const float* __restrict__ p2,
    const float* __restrict__ o0, const float* __restrict__ o1, const float* __restrict__ o2,
    const int* __restrict__ map, const int* __restrict__ tiles,
    int n, GridDesc g, const int* __restrict__ cell_start, const int* __restrict__ tile_keys,
    const int* __restrict__ tile_nc, const int* __restrict__ tile_uoff, float r2, int cap,
    int rcap, int64_t npad, int* __restrict__ count, unsigned short* __restrict__ slot,
    int* __restrict__ tile_j, int* __restrict__ tile_uc, int* __restrict__ tile_over,
    int* overflow, int compact_max) {
#pragma clang fp contract(off)
  constexpr int NT = kListThreads;
  __shared__ int sb[kTileMaxCells], spre[kTileMaxCells];
  __shared__ float4 spos[kListStage + 1];  // candidate positions; the last: near nothing
  __shared__ short sidx[kCompactMax];  // referenced flag, then compacted position (or -1)
  __shared__ __align__(16) unsigned short near[NT / 64][kListStage + 8 * kListLanes];
  __shared__ __align__(8) unsigned short row[kTileP * kRowStride];
  __shared__ int wsum[NT / 64];
  const int t = tiles ? tiles[blockIdx.x] : blockIdx.x;
  const int tid = threadIdx.x;
  const int sub = tid & (kListLanes - 1);  // lanes 4p .. 4p+3 hold particle p
  const int nc = min(tile_nc[t], kTileMaxCells);
  const int* keys = tile_keys + (int64_t)t * kTileMaxCells;
  // cell ranges and their prefix: thread tid takes cells [tid*K, tid*K+K)
  const int K = (nc + NT - 1) / NT;  // at most kTileMaxCells / NT
  const int p0c = min(tid * K, nc), p1c = min(p0c + K, nc);
  int mine = 0;
  for (int p = p0c; p < p1c; p++) {
    const int k = keys[p];
    const int b = cell_start[k];
    sb[p] = b;
    spre[p] = cell_start[k + 1] - b;
    mine += spre[p];
  }
  int U;
  int run0 = block_excl_scan<NT>(mine, wsum, U);
  for (int p = p0c; p < p1c; p++) {
    const int c = spre[p];
    spre[p] = run0;
    run0 += c;
  }
  const bool compact = U <= compact_max;
  if (compact)
    for (int s = tid; s < U; s += NT) sidx[s] = 0;
  __syncthreads();
  const int uoff = tile_uoff[t];
  const int i = t * kTileP + tid / kListLanes;
  const bool act = i < n;
  int c = 0;  // the particle's list length so far (the same in its lanes)
  // a lane without a particle is near nothing (comparisons with NaN are false)
  float xi = NAN, yi = NAN, zi = NAN;
  if (act) {
    xi = o0 ? o0[i] : p0[i];
    yi = o1 ? o1[i] : p1[i];
    zi = o2 ? o2[i] : p2[i];
  }
  // the box around the wavefront's particles
  float bl[3] = {xi, yi, zi}, bh[3] = {xi, yi, zi};
#pragma unroll
  for (int a = 0; a < 3; a++)
    for (int d = kListLanes; d < 64; d <<= 1) {
      bl[a] = fminf(bl[a], __shfl_xor(bl[a], d));
      bh[a] = fmaxf(bh[a], __shfl_xor(bh[a], d));
    }
  const int lane = lane_id();
  const unsigned rbits = r2 > 0.f ? __float_as_uint(r2) - 1u : 0u;
  unsigned short* nr = near[tid >> 6];
  if (tid == 0) spos[kListStage] = make_float4(NAN, NAN, NAN, 0.f);
  unsigned short* rw = row + tid / kListLanes * kRowStride;
  for (int c0 = 0; c0 < U; c0 += kListStage) {
    const int m = min(kListStage, U - c0);
    __syncthreads();  // the previous chunk is consumed (and spre is complete)
    for (int q = tid; q < m; q += NT) {
      const int p = staged_cell(spre, nc, c0 + q);
      const int j = sb[p] + (c0 + q - spre[p]);
      spos[q] = make_float4(p0[j], p1[j], p2[j], 0.f);
    }
    __syncthreads();
    // the candidates within r of the box, in order: rounding is monotone, so
    // the distance to the box is at most the distance to a particle in it, and
    // a candidate left out here fails the test of every particle
    int nn = 0;
    for (int q0 = 0; q0 < m; q0 += 64) {
      const int q = q0 + lane;
      const float4 pj = spos[min(q, m - 1)];
      const float dx = fmaxf(fmaxf(bl[0] - pj.x, pj.x - bh[0]), 0.f);
      const float dy = fmaxf(fmaxf(bl[1] - pj.y, pj.y - bh[1]), 0.f);
      const float dz = fmaxf(fmaxf(bl[2] - pj.z, pj.z - bh[2]), 0.f);
      const float d2 = __fadd_rn(__fadd_rn(__fmul_rn(dx, dx), __fmul_rn(dy, dy)),
                                 __fmul_rn(dz, dz));
      const bool in = q < m && d2 < r2;
      const unsigned long long b = __ballot(in);
      if (in) nr[nn + __popcll(b & ((1ull << lane) - 1ull))] = (unsigned short)q;
      nn += __popcll(b);
    }
    if (lane < 8 * kListLanes) nr[nn + lane] = kListStage;  // to a whole round
    __syncthreads();
    // 32 candidates at a time: each of a particle's lanes tests eight into a
    // bit mask, the masks are joined, and each lane appends its own hits at the
    // positions the joined mask gives them, in candidate order
    uint4 e = *reinterpret_cast<const uint4*>(nr + 8 * sub);
    for (int q0 = 0; q0 < nn; q0 += 8 * kListLanes) {
      const int qb = q0 + 8 * sub;
      const unsigned ew[4] = {e.x, e.y, e.z, e.w};
      e = *reinterpret_cast<const uint4*>(nr + min(qb + 8 * kListLanes, kListStage + 8 * sub));
      unsigned mine = 0u;
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const float4 pj = spos[u & 1 ? ew[u >> 1] >> 16 : ew[u >> 1] & 0xFFFFu];
        float ddx = pj.x - xi, ddy = pj.y - yi, ddz = pj.z - zi;
        float d2 = __fadd_rn(__fadd_rn(__fmul_rn(ddx, ddx), __fmul_rn(ddy, ddy)),
                             __fmul_rn(ddz, ddz));
        // 0 < d2 < r2 in one comparison: non-negative floats order as their bits,
        // 0 goes to the top and NaN lies above every number
        if (__float_as_uint(d2) - 1u < rbits) mine |= 1u << u;
      }
      unsigned all = mine << (8 * sub);
      all |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)all, 0xB1, 0xF, 0xF, false);  // lane ^ 1
      all |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)all, 0x4E, 0xF, 0xF, false);  // lane ^ 2
      int k = c + __popc(all & ((1u << (8 * sub)) - 1u));
      unsigned h = mine;
      while (h) {
        const int u = __builtin_ctz(h);
        h &= h - 1u;
        const unsigned w2 = u & 4 ? (u & 2 ? ew[3] : ew[2]) : (u & 2 ? ew[1] : ew[0]);
        const int sl = c0 + (int)(u & 1 ? w2 >> 16 : w2 & 0xFFFFu);
        if (k < cap) {
          rw[k] = (unsigned short)sl;
          if (compact) sidx[sl] = 1;
        }
        k++;
      }
      c += __popc(all);
    }
  }
  if (act && sub == 0) count[i] = c < cap ? c : cap;
  __syncthreads();  // every row entry and flag is visible
  int used = U;
  if (compact) {
    // exclusive scan of the flags, one contiguous segment per thread
    const int seg = (U + NT - 1) / NT;
    const int s0 = min(tid * seg, U), s1 = min(s0 + seg, U);
    int sum = 0;
    for (int s = s0; s < s1; s++) sum += sidx[s];
    int run = block_excl_scan<NT>(sum, wsum, used);
    for (int s = s0; s < s1; s++) {
      const int fl = sidx[s];
      sidx[s] = fl ? run : -1;
      run += fl;
    }
    __syncthreads();
  }
  // the particle's list, its slots as positions in the compacted set, its
  // quads dealt out to its lanes
  const int m = act ? min(c, cap) : 0;
  const int nq = (m + 3) >> 2;
  uint2* qrow = reinterpret_cast<uint2*>(slot) + i;
  for (int q = sub; q < nq; q += kListLanes) {
    const uint2 w = *reinterpret_cast<const uint2*>(rw + 4 * q);
    unsigned v[4] = {w.x & 0xFFFFu, w.x >> 16, w.y & 0xFFFFu, w.y >> 16};
#pragma unroll
    for (int u = 0; u < 4; u++) {
      if (4 * q + u >= m) v[u] = v[0];  // the quad's first, which is in the list
      else if (compact) v[u] = (unsigned short)sidx[v[u]];
    }
    qrow[(int64_t)q * npad] = make_uint2(v[0] | v[1] << 16, v[2] | v[3] << 16);
  }
  // the region this tile was given at the last reorder
  const int room = map ? tile_uoff[t + 1] - uoff : INT_MAX;
  if (used > room) {
    if (tid == 0) atomicAdd(overflow, 1);
  } else {
    for (int s = tid; s < U; s += NT) {
      const int d = compact ? sidx[s] : s;
      if (d >= 0) {
        const int p = staged_cell(spre, nc, s);
        const int js = sb[p] + (s - spre[p]);
        tile_j[uoff + d] = map ? map[js] : js;
      }
    }
  }
  if (tid == 0) tile_uc[t] = used;
  // particles of the tile over the reported cap, one count each
  const int over = act && sub == 0 && c > rcap;
  const unsigned long long o = wave_sum_u64((unsigned long long)over);
  if (lane_id() == 0) wsum[threadIdx.x >> 6] = (int)o;
  __syncthreads();
  if (tid == 0) {
    int tot = 0;
    for (int u = 0; u < NT / 64; u++) tot += wsum[u];
    tile_over[t] = tot;
  }
}

void launch_tile_cells(hipStream_t s, const float* const pf[3], int n, const GridDesc& g,
                       const int* cell_start, const int* tiles, int ntiles, bool sort_own,
                       int* tile_keys, int* tile_nc, int* tile_ucnt, int* overflow) {
  if (ntiles <= 0) return;
  if (sort_own)
    hipLaunchKernelGGL(k_tile_cells<true>, dim3(ntiles), dim3(kTileP), 0, s, pf[0], pf[1], pf[2],
                       n, g, cell_start, tiles, tile_keys, tile_nc, tile_ucnt, overflow);
  else
    hipLaunchKernelGGL(k_tile_cells<false>, dim3(ntiles), dim3(kTileP), 0, s, pf[0], pf[1],
                       pf[2], n, g, cell_start, tiles, tile_keys, tile_nc, tile_ucnt, overflow);
}

void launch_tile_lists(hipStream_t s, const float* const pf[3], const float* const own[3],
                       const int* map, const int* tiles, int ntiles, int n, const GridDesc& g,
                       const int* cell_start, const int* tile_keys, const int* tile_nc,
                       const int* tile_uoff, float r2, int cap, int rcap, int64_t npad,
                       int* count, unsigned short* slot, int* tile_j, int* tile_uc,
                       int* tile_over, int* overflow, int compact_max) {
  if (ntiles <= 0) return;
  compact_max = compact_max > 0 ? std::min(compact_max, kCompactMax) : kCompactMax;
  const float* o0 = own ? own[0] : nullptr;
  const float* o1 = own ? own[1] : nullptr;
  const float* o2 = own ? own[2] : nullptr;
  hipLaunchKernelGGL(k_tile_lists, dim3(ntiles), dim3(kListThreads), 0, s, pf[0], pf[1], pf[2],
                     o0, o1, o2, map, tiles, n, g, cell_start, tile_keys, tile_nc, tile_uoff, r2,
                     cap, rcap, npad, count, slot, tile_j, tile_uc, tile_over, overflow,
                     compact_max);
}

}  // namespace wf
