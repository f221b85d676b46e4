// Neighbour lists for the BP+EE path.
//
// Replaces MolEmb.Make_NListNaive (C_API/MolEmb.cpp:1180-1247) and the Python
// pair/triple assembly of NeighborList.buildPairsAndTriples and
// NeighborListSet.buildPairsAndTriplesWithEleIndex
// (TensorMol/ForceModifiers/Neighbors.py:117-201, 344-423).
//
// Pair predicate: the reference keeps j when sqrt(dx*dx+dy*dy+dz*dz)+1e-13 < rc
// in float64.  With correctly rounded sqrt and add that predicate is monotone
// in s = (dx*dx+dy*dy)+dz*dz, so the host computes the first double s* that
// fails it and the kernel tests s < s* with s evaluated without contraction:
// the same set, bit for bit, and no dependence on the device sqrt.
//
// Output (ELL rows, one per centre atom, stride ldr):
//   nbr[i*ldr + n]   neighbour atom j (global packed index), sorted by
//                    (element index of j, j) = the (m,i,l,j) order of trpE
//   ncnt[i]          row length
//   rseg[i*(nele+1)+e] start of element e's segment in the row (last = ncnt)
//   ang[i*lda + a]   position (in row i) of the a-th neighbour closer than
//                    the angular cutoff; the sub-list keeps the row order
//   acnt[i], aseg[i*(nele+1)+e]  as above for the sub-list
//   rev[i*ldr + n]   slot (j*ldr + n') of the mirror entry j -> i
//
// Candidate atoms come either from the atom's molecule (batches of small
// molecules) or from a cell grid (one large open or periodic system).
#include "tm_cells.h"

namespace {

constexpr int NL_WAVES = 4;           // waves per block, one centre per wave
constexpr int NL_LDS_CAP = 256;       // candidate buffer per wave
constexpr int NL_RANGES = 192;        // finer grids than this many stencil ranges are refused
constexpr int NL_LIST = 256;          // candidate list per wave

__device__ __forceinline__ double sq_dist_nocontract(double xi, double yi, double zi, double xj,
                                                     double yj, double zj, double Lx, double Ly,
                                                     double Lz) {
#pragma clang fp contract(off)
  double dx = tm_min_image(xi - xj, Lx);
  double dy = tm_min_image(yi - yj, Ly);
  double dz = tm_min_image(zi - zj, Lz);
  double s = dx * dx + dy * dy;
  s = s + dz * dz;
  return s;
}

__device__ __forceinline__ double sq_dist_nocontract(double xi, double yi, double zi, double xj,
                                                     double yj, double zj) {
#pragma clang fp contract(off)
  const double dx = xi - xj, dy = yi - yj, dz = zi - zj;
  double s = dx * dx + dy * dy;
  s = s + dz * dz;
  return s;
}

// The same with the reciprocal edges (0 for open boundaries).  The image it
// picks differs only where a separation is half an edge to the last digit, for
// which the two images are equally far.
__device__ __forceinline__ double sq_dist_nocontract(double xi, double yi, double zi, double xj,
                                                     double yj, double zj, double Lx, double Ly,
                                                     double Lz, double iLx, double iLy, double iLz) {
#pragma clang fp contract(off)
  double dx = xi - xj, dy = yi - yj, dz = zi - zj;
  dx = dx - Lx * rint(dx * iLx);
  dy = dy - Ly * rint(dy * iLy);
  dz = dz - Lz * rint(dz * iLz);
  double s = dx * dx + dy * dy;
  s = s + dz * dz;
  return s;
}

// One wavefront per centre: candidates from the molecule, or from the cell list
// with their loads one chunk ahead; kept ones as (atom, near) until the sweep is
// over, then their elements in one round of loads, a rank sort and the segment
// counts.  What bounds it: a chain of five dependent loads and some 700 vector
// instructions per centre.  Elements read chunk by chunk behind the cell's
// atoms, divisions by the box edges, a search over ranges and block barriers
// made it 20.6 us for the 12,288-atom box; now 18.6, lists and descriptors
// 64.6 -> 61.0.
// BOX false (no boxes): the images' FP64 operations, half of a test, are left
// out.  A kernel of its own: a branch cost the periodic rows 0.8 us.
template <bool BOX>
__global__ void __launch_bounds__(NL_WAVES * 64)
nl_rows_kernel(int N, const double* __restrict__ pos, const int* __restrict__ elem,
               const int* __restrict__ mol, const int* __restrict__ mol_start,
               const double* __restrict__ box, CellGrid grid, int nele,
               double s_r, double s_a, int ldr, int lda,
               int* __restrict__ nbr, int* __restrict__ ncnt, int* __restrict__ rseg,
               int* __restrict__ ang, int* __restrict__ acnt, int* __restrict__ aseg,
               int* __restrict__ flags) {
  // key = element << 28 | j << 1 | (within the angular cutoff): the order of
  // keys is the order of (element, j) for distinct atoms (j < 2^27)
  __shared__ __align__(16) unsigned keys[NL_WAVES][NL_LDS_CAP + 4];
  __shared__ unsigned sorted[NL_WAVES][NL_LDS_CAP];
  __shared__ ListLds<NL_LIST> list[NL_WAVES];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int i = blockIdx.x * NL_WAVES + w;
  if (i >= N) return;   // wave-level synchronisation only below
  const int mi = mol[i];
  const double xi = pos[3 * (long)i], yi = pos[3 * (long)i + 1], zi = pos[3 * (long)i + 2];
  double Lx = 0, Ly = 0, Lz = 0, iLx = 0, iLy = 0, iLz = 0;
  if constexpr (BOX) {
    Lx = box[3 * mi]; Ly = box[3 * mi + 1]; Lz = box[3 * mi + 2];
    iLx = Lx > 0.0 ? 1.0 / Lx : 0.0;
    iLy = Ly > 0.0 ? 1.0 / Ly : 0.0;
    iLz = Lz > 0.0 ? 1.0 / Lz : 0.0;
  }
  int count = 0;   // wave-uniform
  // candidate j at (x, y, z); self and other molecules are not taken
  auto test = [&](double x, double y, double z, int j, bool take) {
    const double s = BOX ? sq_dist_nocontract(xi, yi, zi, x, y, z, Lx, Ly, Lz, iLx, iLy, iLz)
                         : sq_dist_nocontract(xi, yi, zi, x, y, z);
    const bool ok = take & (s < s_r);
    const unsigned long long bal = __ballot(ok);
    const int slot = count + tm_lanes_below(bal);
    if (ok && slot < NL_LDS_CAP) keys[w][slot] = ((unsigned)j << 1) | (s < s_a ? 1u : 0u);
    count += __popcll(bal);
  };
  if (grid.cell_atoms != nullptr) {
    struct Cand {
      double x, y, z;
      int j, m;
    };
    tm_sweep_list(
        grid, tm_centre(grid, grid.cell_of[i], xi, yi, zi), list[w], lane,
        [&](int p) {
          const double* c = grid.posc + 3 * (long)p;
          return Cand{c[0], c[1], c[2], grid.cell_atoms[p], grid.molc == nullptr ? mi : grid.molc[p]};
        },
        [&](int, bool valid, const Cand& c) {
          test(c.x, c.y, c.z, c.j, valid & (c.j != i) & (c.m == mi));
        });
  } else {
    const int lo = mol_start[mi], hi = mol_start[mi + 1];
    for (int base = lo; base < hi; base += 64) {
      // lanes past the end read the last atom, so the test is branch-free
      const int j = min(base + lane, hi - 1);
      test(pos[3 * (long)j], pos[3 * (long)j + 1], pos[3 * (long)j + 2], j,
           (base + lane < hi) & (j != i));
    }
  }
  if (count > NL_LDS_CAP || count > ldr) {
    if (lane == 0) atomicOr(&flags[TM_FLAG_NB_OVERFLOW], 1);
    count = min(count, min(NL_LDS_CAP, ldr));
  }
  __syncwarp();
  for (int a = lane; a < count; a += 64) {
    const unsigned k = keys[w][a];
    keys[w][a] = ((unsigned)elem[k >> 1] << 28) | k;
  }
  if (lane < 4) keys[w][count + lane] = ~0u;   // nothing sorts behind the padding
  __syncwarp();
  // rank sort by (element, atom index)
  for (int a = lane; a < count; a += 64) {
    const unsigned ka = keys[w][a];
    int rank = 0;
#pragma unroll 2
    for (int b = 0; b < count; b += 4) {
      const uint4 kb = *reinterpret_cast<const uint4*>(&keys[w][b]);
      rank += (kb.x < ka) + (kb.y < ka) + (kb.z < ka) + (kb.w < ka);
    }
    sorted[w][rank] = ka;
  }
  __syncwarp();
  long rowr = (long)i * ldr;
  long rowa = (long)i * lda;
  int acount = 0;
  int cr = 0, ca = 0;   // lane e <= nele: entries (all / angular) with element < e
  for (int base = 0; base < count; base += 64) {
    int a = base + lane;
    bool have = a < count;
    unsigned k = have ? sorted[w][a] : 0u;
    if (have) nbr[rowr + a] = (int)((k >> 1) & ((1u << 27) - 1u));
    bool isang = have && (k & 1u);
    unsigned long long bal = __ballot(isang);
    int before = tm_lanes_below(bal);
    if (isang) {
      int slot = acount + before;
      if (slot < lda) ang[rowa + slot] = a;
    }
    acount += __popcll(bal);
    const int el = (int)(k >> 28);
    for (int e = 1; e <= nele; ++e) {   // element segment starts of this chunk
      const unsigned long long br = __ballot(have && el < e);
      const unsigned long long ba = __ballot(isang && el < e);
      if (lane == e) { cr += __popcll(br); ca += __popcll(ba); }
    }
  }
  if (acount > lda) {
    if (lane == 0) atomicOr(&flags[TM_FLAG_ANG_OVERFLOW], 1);
    acount = lda;
  }
  if (lane == 0) { ncnt[i] = count; acnt[i] = acount; }
  if (lane <= nele) {
    if (ca > acount) ca = acount;
    rseg[(long)i * (nele + 1) + lane] = cr;
    aseg[(long)i * (nele + 1) + lane] = ca;
  }
}

// Mirror slot of every entry: rev[i*ldr+n] = j*ldr + position of i in row j.
__global__ void nl_rev_kernel(int N, int ldr, int nele, const int* __restrict__ elem,
                              const int* __restrict__ nbr, const int* __restrict__ ncnt,
                              const int* __restrict__ rseg, int* __restrict__ rev,
                              int* __restrict__ flags) {
  long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  int i = (int)(t / ldr);
  int n = (int)(t % ldr);
  if (i >= N || n >= ncnt[i]) return;
  int j = nbr[(long)i * ldr + n];
  int e = elem[i];
  int lo = rseg[(long)j * (nele + 1) + e];
  int hi = rseg[(long)j * (nele + 1) + e + 1];
  const int* row = nbr + (long)j * ldr;
  while (lo < hi) {
    int mid = (lo + hi) >> 1;
    if (row[mid] < i) lo = mid + 1; else hi = mid;
  }
  if (lo < ncnt[j] && row[lo] == i) {
    rev[(long)i * ldr + n] = (int)((long)j * ldr + lo);
  } else {
    rev[(long)i * ldr + n] = (int)((long)i * ldr + n);   // unmatched (truncated row)
    atomicOr(&flags[TM_FLAG_NB_OVERFLOW], 2);
  }
}

// ---------------------------------------------------------------- cell grid
// Cell of atom i; raises what is wrong with its coordinates in st (bit 0 not
// finite: taken as the origin; bit 1 outside an open grid: clamped).
struct CellGeom {
  double o[3], cs[3];
  int n[3], periodic;
};
__device__ __forceinline__ int cell_of_atom(const double* __restrict__ pos, int i,
                                            const CellGeom& g, int& st) {
  double p[3] = {pos[3 * i], pos[3 * i + 1], pos[3 * i + 2]};
  st = 0;
  if (!isfinite(p[0]) || !isfinite(p[1]) || !isfinite(p[2])) {
    st = 1;
    p[0] = p[1] = p[2] = 0.0;
  }
  int c[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    long q = (long)floor((p[d] - g.o[d]) / g.cs[d]);
    if (g.periodic) {
      q %= g.n[d];
      if (q < 0) q += g.n[d];
    } else if (q < 0 || q >= g.n[d]) {
      st |= 2;
      q = q < 0 ? 0 : g.n[d] - 1;
    }
    c[d] = (int)q;
  }
  return c[0] + g.n[0] * (c[1] + g.n[1] * c[2]);
}
__device__ __forceinline__ void raise_status(int st, int* flags) {
  if (st & 1) atomicOr(&flags[TM_FLAG_NONFINITE], 1);
  if (st & 2) atomicOr(&flags[TM_FLAG_CELL_OVERFLOW], 1);
}

// FRESH: the launch clears the flags instead of raising any, and the fill
// launch raises them (it finds the same from the positions again, under the
// latency of its other loads), so no launch goes before the build to clear them.
// Lists and descriptors of the 12,288-atom box 59.3 -> 58.0 us.
template <bool FRESH>
__global__ void cell_assign_kernel(int N, const double* __restrict__ pos, CellGeom g,
                                   int* __restrict__ cell_of, int* __restrict__ cell_count,
                                   int* __restrict__ flags) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if constexpr (FRESH)
    if (i < TM_NFLAGS) flags[i] = 0;
  if (i >= N) return;
  int st;
  const int cell = cell_of_atom(pos, i, g, st);
  if constexpr (!FRESH) raise_status(st, flags);
  cell_of[i] = cell;
  atomicAdd(&cell_count[cell], 1);
}

// Exclusive prefix sum of n ints (out[n] = total), zeroing the input as it is
// read (the per-cell counts become the fill counters).  A tile of 16384
// entries is scanned by a 1024-thread block: 16 consecutive entries per thread
// (four 16-byte loads; in and out are 16-byte aligned), a shuffle scan of the
// thread totals inside each wave, the 16 wave totals scanned through LDS.
// One block walks the tiles with a running carry when there are few; for
// more, a first launch writes the tile totals and a second scans every tile
// from the sum of the totals before it.
constexpr int SCAN_PT = 16;
constexpr int SCAN_TILE = 1024 * SCAN_PT;

__device__ __forceinline__ int scan_tile(int n, int* __restrict__ in, int* __restrict__ out,
                                         int base, int carry, int* wtot) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int i0 = base + SCAN_PT * tid;
  int v[SCAN_PT];
  if (i0 + SCAN_PT <= n) {
#pragma unroll
    for (int q = 0; q < SCAN_PT / 4; ++q) {
      const int4 x = reinterpret_cast<const int4*>(in + i0)[q];
      v[4 * q] = x.x; v[4 * q + 1] = x.y; v[4 * q + 2] = x.z; v[4 * q + 3] = x.w;
    }
#pragma unroll
    for (int q = 0; q < SCAN_PT / 4; ++q) reinterpret_cast<int4*>(in + i0)[q] = make_int4(0, 0, 0, 0);
  } else {
#pragma unroll
    for (int k = 0; k < SCAN_PT; ++k) v[k] = i0 + k < n ? in[i0 + k] : 0;
#pragma unroll
    for (int k = 0; k < SCAN_PT; ++k)
      if (i0 + k < n) in[i0 + k] = 0;
  }
  int t = 0;
#pragma unroll
  for (int k = 0; k < SCAN_PT; ++k) t += v[k];
  int incl = t;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    int u = __shfl_up(incl, o, 64);
    if (lane >= o) incl += u;
  }
  if (lane == 63) wtot[w] = incl;
  __syncthreads();
  if (w == 0) {
    int x = lane < 16 ? wtot[lane] : 0;
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) {
      int u = __shfl_up(x, o, 64);
      if (lane >= o) x += u;
    }
    if (lane < 16) wtot[lane] = x;   // inclusive over waves
  }
  __syncthreads();
  int run = carry + (w > 0 ? wtot[w - 1] : 0) + incl - t;
  int e[SCAN_PT];
#pragma unroll
  for (int k = 0; k < SCAN_PT; ++k) { e[k] = run; run += v[k]; }
  if (i0 + SCAN_PT <= n) {
#pragma unroll
    for (int q = 0; q < SCAN_PT / 4; ++q)
      reinterpret_cast<int4*>(out + i0)[q] = make_int4(e[4 * q], e[4 * q + 1], e[4 * q + 2], e[4 * q + 3]);
  } else {
#pragma unroll
    for (int k = 0; k < SCAN_PT; ++k)
      if (i0 + k < n) out[i0 + k] = e[k];
  }
  const int total = wtot[15];
  __syncthreads();   // wtot is reused by the next tile
  return total;
}

__global__ void __launch_bounds__(1024) scan_kernel(int n, int* __restrict__ in,
                                                    int* __restrict__ out) {
  __shared__ int wtot[16];
  int carry = 0;
  for (int base = 0; base < n; base += SCAN_TILE) carry += scan_tile(n, in, out, base, carry, wtot);
  if (threadIdx.x == 0) out[n] = carry;
}

// totals of the 16384-entry tiles (fixed-order block reduction)
__global__ void __launch_bounds__(1024) scan_sums_kernel(int n, const int* __restrict__ in,
                                                         int* __restrict__ sums) {
  __shared__ int wsum[16];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int i0 = blockIdx.x * SCAN_TILE + SCAN_PT * tid;
  int t = 0;
  if (i0 + SCAN_PT <= n) {
#pragma unroll
    for (int q = 0; q < SCAN_PT / 4; ++q) {
      const int4 x = reinterpret_cast<const int4*>(in + i0)[q];
      t += (x.x + x.y) + (x.z + x.w);
    }
  } else {
    for (int k = 0; k < SCAN_PT; ++k) t += i0 + k < n ? in[i0 + k] : 0;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
  if (lane == 0) wsum[w] = t;
  __syncthreads();
  if (tid == 0) {
    int x = 0;
    for (int q = 0; q < 16; ++q) x += wsum[q];
    sums[blockIdx.x] = x;
  }
}

// each block scans its tile from the sum of the totals of the tiles before it
__global__ void __launch_bounds__(1024) scan_apply_kernel(int n, int* __restrict__ in,
                                                          int* __restrict__ out,
                                                          const int* __restrict__ sums) {
  __shared__ int wtot[16];
  __shared__ int carry_s;
  const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  if (tid < 64) {
    int x = 0;
    for (int q = lane; q < b; q += 64) x += sums[q];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    if (tid == 0) carry_s = x;
  }
  __syncthreads();
  const int carry = carry_s;
  const int total = scan_tile(n, in, out, b * SCAN_TILE, carry, wtot);
  if (b == (int)gridDim.x - 1 && tid == 0) out[n] = carry + total;
}

// unsorted cell order into the staging array; the counters start at zero
template <bool FRESH>
__global__ void cell_fill_kernel(int N, const int* __restrict__ cell_of,
                                 const int* __restrict__ cell_start, int* __restrict__ counter,
                                 int* __restrict__ staging, const double* __restrict__ pos,
                                 CellGeom g, int* __restrict__ flags) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  int c = cell_of[i];
  if constexpr (FRESH) {
    int st;
    cell_of_atom(pos, i, g, st);
    raise_status(st, flags);
  }
  int slot = cell_start[c] + atomicAdd(&counter[c], 1);
  staging[slot] = i;
}

// order atoms inside each cell by index, so every later sweep is
// deterministic: one wavefront per cell ranks its entries (cells hold a few
// dozen atoms; larger cells are ranked in 64-entry rounds).  Each wave also
// clears its cell's counter, so the counters are zero for the next build.
__global__ void cell_sort_kernel(int ncell, const int* __restrict__ cell_start,
                                 const int* __restrict__ unsorted, int* __restrict__ cell_atoms,
                                 int* __restrict__ cell_pos, const double* __restrict__ pos,
                                 double* __restrict__ posc, const int* __restrict__ mol,
                                 int* __restrict__ molc, int* __restrict__ counter) {
  const int c = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (c >= ncell) return;
  if (lane == 0) counter[c] = 0;
  const int lo = cell_start[c], hi = cell_start[c + 1];
  for (int a = lo + lane; a < hi; a += 64) {
    int v = unsorted[a];
    int rank = 0;
    for (int b = lo; b < hi; ++b) rank += unsorted[b] < v;
    int q = lo + rank;
    cell_atoms[q] = v;
    cell_pos[v] = q;
    posc[3 * (long)q] = pos[3 * (long)v];
    posc[3 * (long)q + 1] = pos[3 * (long)v + 1];
    posc[3 * (long)q + 2] = pos[3 * (long)v + 2];
    if (molc != nullptr) molc[q] = mol[v];
  }
}

// Materialise the sorted triple list of one row set (API parity with
// buildPairsAndTriplesWithEleIndex): for each centre, triples grouped by
// element pair p, inside a group ordered by (k, j); rank = position in group.
// trip_start[i] is the exclusive prefix of per-centre triple counts.
__global__ void triples_kernel(int N, int ldr, int lda, int nele, const int* __restrict__ nbr,
                               const int* __restrict__ ang, const int* __restrict__ acnt,
                               const int* __restrict__ aseg, const long* __restrict__ trip_start,
                               int* __restrict__ out_jkpr) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  long o = trip_start[i];
  const int* seg = aseg + (long)i * (nele + 1);
  const int* arow = ang + (long)i * lda;
  const int* row = nbr + (long)i * ldr;
  int p = 0;
  for (int ea = 0; ea < nele; ++ea) {
    for (int eb = ea; eb < nele; ++eb, ++p) {
      int rank = 0;
      // order (k, j): k runs over the second element's segment ascending,
      // j over the first's ascending with j < k when the elements agree
      for (int kb = seg[eb]; kb < seg[eb + 1]; ++kb) {
        int jhi = (ea == eb) ? kb : seg[ea + 1];
        for (int ja = seg[ea]; ja < jhi; ++ja) {
          int j = row[arow[ja]], k = row[arow[kb]];
          out_jkpr[4 * o + 0] = j;
          out_jkpr[4 * o + 1] = k;
          out_jkpr[4 * o + 2] = p;
          out_jkpr[4 * o + 3] = rank++;
          ++o;
        }
      }
    }
  }
}

// Pair list for an arbitrary cutoff (the EE list of Neighbors.py:262-282 and
// Make_NListNaive with DoPerms 0/1): pass 1 counts, pass 2 writes each row in
// candidate order (ascending j for molecule sweeps, cell order otherwise).
// Centres i with local index >= nreal[m] get empty rows; with half = 1 only
// j > i is kept (pairs stored once under min(i, j)).
template <bool FILL>
__global__ void __launch_bounds__(NL_WAVES * 64)
pairs_kernel(int N, const double* __restrict__ pos, const int* __restrict__ mol,
             const int* __restrict__ mol_start, const int* __restrict__ nreal,
             const double* __restrict__ box, CellGrid grid, double s_c, int half,
             int* __restrict__ count, const long* __restrict__ start, int* __restrict__ out,
             int* __restrict__ flags) {
  __shared__ RangeLds<1024> rng[NL_WAVES];
  const int w = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int i = blockIdx.x * NL_WAVES + w;
  if (i >= N) return;   // wave-level synchronisation only
  const int mi = mol[i];
  if (nreal != nullptr && i - mol_start[mi] >= nreal[mi]) {
    if (!FILL && lane == 0) count[i] = 0;
    return;
  }
  double Lx = 0, Ly = 0, Lz = 0;
  if (box != nullptr) {
    Lx = box[3 * mi]; Ly = box[3 * mi + 1]; Lz = box[3 * mi + 2];
  }
  const double xi = pos[3 * i], yi = pos[3 * i + 1], zi = pos[3 * i + 2];
  const int cpi = grid.cell_pos != nullptr ? grid.cell_pos[i] : -1;
  long o = FILL ? start[i] : 0;
  int cnt = 0;
  auto visit = [&](int p, bool valid, int mapped) {
    bool ok = false;
    int j = -1;
    if (valid && (mapped ? p != cpi : p != i) &&
        (!mapped || grid.molc == nullptr || grid.molc[p] == mi)) {
      j = mapped ? grid.cell_atoms[p] : p;
      const double* q = mapped ? grid.posc + 3 * (long)p : pos + 3 * (long)p;
      ok = (!half || j > i) && sq_dist_nocontract(xi, yi, zi, q[0], q[1], q[2], Lx, Ly, Lz) < s_c;
    }
    unsigned long long bal = __ballot(ok);
    if (FILL && ok) out[o + cnt + tm_lanes_below(bal)] = j;
    cnt += __popcll(bal);
  };
  tm_sweep(i, mol, mol_start, grid, rng[w], lane, flags, xi, yi, zi, visit);
  if (!FILL && lane == 0) count[i] = cnt;
}

}  // namespace

template <bool FRESH>
static int cell_build(int N, const double* pos, const int* mol, double ox, double oy, double oz,
                  double cx, double cy, double cz, int nx, int ny, int nz, int periodic,
                  int* cell_of, int* cell_count, int* cell_start, int* cell_fill, int* cell_atoms,
                  int* cell_pos, double* posc, int* molc, int* flags, void* stream) {
  TM_REQUIRE(N >= 0 && nx > 0 && ny > 0 && nz > 0, "tm_cell_build: bad sizes");
  TM_REQUIRE((long)nx * ny * nz < (1l << 26), "tm_cell_build: %d x %d x %d cells is too many", nx, ny, nz);
  hipStream_t s = (hipStream_t)stream;
  long ncell = (long)nx * ny * nz;
  if (N == 0) return TM_OK;
  // cell_count is zero here: the previous call's sort cleared it (no memset
  // nodes when the caller captures a graph)
  const CellGeom g = {{ox, oy, oz}, {cx, cy, cz}, {nx, ny, nz}, periodic};
  cell_assign_kernel<FRESH><<<tm_div_up(N, 256), 256, 0, s>>>(N, pos, g, cell_of, cell_count,
                                                              flags);
  TM_LAUNCH_CHECK();
  const int ntile = (int)((ncell + SCAN_TILE - 1) / SCAN_TILE);
  if (ntile <= 2 || ntile > N) {
    scan_kernel<<<1, 1024, 0, s>>>((int)ncell, cell_count, cell_start);
    TM_LAUNCH_CHECK();
  } else {   // tile totals in cell_fill (not yet in use: the fill comes next)
    scan_sums_kernel<<<ntile, 1024, 0, s>>>((int)ncell, cell_count, cell_fill);
    TM_LAUNCH_CHECK();
    scan_apply_kernel<<<ntile, 1024, 0, s>>>((int)ncell, cell_count, cell_start, cell_fill);
    TM_LAUNCH_CHECK();
  }
  cell_fill_kernel<FRESH><<<tm_div_up(N, 256), 256, 0, s>>>(N, cell_of, cell_start, cell_count,
                                                            cell_fill, pos, g, flags);
  TM_LAUNCH_CHECK();
  cell_sort_kernel<<<tm_div_up(ncell, 4), 256, 0, s>>>((int)ncell, cell_start, cell_fill,
                                                       cell_atoms, cell_pos, pos, posc, mol, molc,
                                                       cell_count);
  TM_LAUNCH_CHECK();
  return TM_OK;
}

extern "C" {

static CellGrid make_grid(const int* cell_start, const int* cell_atoms, const int* cell_of,
                          const int* cell_pos, const double* posc, const int* molc, int nx, int ny,
                          int nz, double csx, double csy, double csz, double ox, double oy,
                          double oz, int periodic, double rc) {
  CellGrid g{};
  g.cell_start = cell_start; g.cell_atoms = cell_atoms; g.cell_of = cell_of;
  g.cell_pos = cell_pos; g.posc = posc; g.molc = molc;
  g.nc[0] = nx; g.nc[1] = ny; g.nc[2] = nz;
  g.cs[0] = (float)csx; g.cs[1] = (float)csy; g.cs[2] = (float)csz;
  g.org[0] = (float)ox; g.org[1] = (float)oy; g.org[2] = (float)oz;
  g.periodic = periodic;
  tm_set_stencil(g, (float)rc);
  return g;
}

// cell_count (ncell ints) must be zero on entry (zero-fill it once; every call
// leaves it zero); it holds the per-cell counts, then the fill counters.
// cell_fill (at least N ints) receives the unsorted staging copy of cell_atoms.
// Outputs cell_atoms (index order inside each cell), cell_pos (position of
// every atom in cell order), posc (positions in cell order) and molc
// (molecules in cell order; may be NULL for one system).
int tm_cell_build(int N, const double* pos, const int* mol, double ox, double oy, double oz,
                  double cx, double cy, double cz, int nx, int ny, int nz, int periodic,
                  int* cell_of, int* cell_count, int* cell_start, int* cell_fill, int* cell_atoms,
                  int* cell_pos, double* posc, int* molc, int* flags, void* stream) {
  return cell_build<false>(N, pos, mol, ox, oy, oz, cx, cy, cz, nx, ny, nz, periodic, cell_of, cell_count,
                           cell_start, cell_fill, cell_atoms, cell_pos, posc, molc, flags, stream);
}

int tm_zero_i32(int n, int* p, void* stream);

// tm_zero_i32 of the TM_NFLAGS flags, then tm_cell_build, without the launch
// that would clear them.
int tm_cell_build_fresh(int N, const double* pos, const int* mol, double ox, double oy, double oz,
                  double cx, double cy, double cz, int nx, int ny, int nz, int periodic,
                  int* cell_of, int* cell_count, int* cell_start, int* cell_fill, int* cell_atoms,
                  int* cell_pos, double* posc, int* molc, int* flags, void* stream) {
  if (N == 0) return tm_zero_i32(TM_NFLAGS, flags, stream);
  return cell_build<true>(N, pos, mol, ox, oy, oz, cx, cy, cz, nx, ny, nz, periodic, cell_of, cell_count,
                           cell_start, cell_fill, cell_atoms, cell_pos, posc, molc, flags, stream);
}

int tm_nl_build(int N, const double* pos, const int* elem, const int* mol, const int* mol_start,
                const double* box, const int* cell_start, const int* cell_atoms,
                const int* cell_of, const int* cell_pos, const double* posc, const int* molc,
                int nx, int ny, int nz, double csx, double csy, double csz, double ox, double oy, double oz, int periodic, int nele,
                double rc, double s_r, double s_a, int ldr, int lda, int* nbr, int* ncnt,
                int* rseg, int* ang, int* acnt, int* aseg, int* rev, int* flags, void* stream) {
  TM_REQUIRE(N >= 0 && nele > 0 && nele <= TM_MAX_ELE, "tm_nl_build: bad nele %d", nele);
  TM_REQUIRE(ldr > 0 && ldr <= 256 && lda > 0 && lda <= ldr, "tm_nl_build: bad strides %d %d", ldr,
             lda);
  TM_REQUIRE((long)N * ldr < (1l << 31), "tm_nl_build: N*ldr overflows int32 slots");
  TM_REQUIRE(N <= (1 << 27), "tm_nl_build: %d atoms above 2^27", N);
  if (cell_atoms != nullptr) {
    TM_REQUIRE(cell_start && cell_of && cell_pos && posc, "tm_nl_build: incomplete cell grid");
    int k = (int)ceil(rc / fmin(csx, fmin(csy, csz))) + 1;
    TM_REQUIRE((2 * k + 3) * (2 * k + 3) * 2 <= NL_RANGES,
               "tm_nl_build: cells of %.2f A are too small for rc %.2f", fmin(csx, fmin(csy, csz)), rc);
  }
  if (N == 0) return TM_OK;
  hipStream_t s = (hipStream_t)stream;
  CellGrid g = make_grid(cell_start, cell_atoms, cell_of, cell_pos, posc, molc, nx, ny, nz, csx, csy,
                         csz, ox, oy, oz, periodic, rc);
  const auto rows = box != nullptr ? nl_rows_kernel<true> : nl_rows_kernel<false>;
  rows<<<tm_div_up(N, NL_WAVES), NL_WAVES * 64, 0, s>>>(
      N, pos, elem, mol, mol_start, box, g, nele, s_r, s_a, ldr, lda, nbr, ncnt, rseg,
      ang, acnt, aseg, flags);
  TM_LAUNCH_CHECK();
  if (rev != nullptr) {   // else tm_sym_forward fills rev
    long total = (long)N * ldr;
    nl_rev_kernel<<<tm_div_up(total, 256), 256, 0, s>>>(N, ldr, nele, elem, nbr, ncnt, rseg, rev,
                                                        flags);
    TM_LAUNCH_CHECK();
  }
  return TM_OK;
}

int tm_triples(int N, int ldr, int lda, int nele, const int* nbr, const int* ang, const int* acnt,
               const int* aseg, const long* trip_start, int* out_jkpr, void* stream) {
  TM_REQUIRE(N >= 0 && nele > 0 && nele <= TM_MAX_ELE, "tm_triples: bad sizes");
  if (N == 0) return TM_OK;
  hipStream_t s = (hipStream_t)stream;
  triples_kernel<<<tm_div_up(N, 128), 128, 0, s>>>(N, ldr, lda, nele, nbr, ang, acnt, aseg,
                                                   trip_start, out_jkpr);
  TM_LAUNCH_CHECK();
  return TM_OK;
}


int tm_pairs(int N, const double* pos, const int* mol, const int* mol_start, const int* nreal,
             const double* box, const int* cell_start, const int* cell_atoms, const int* cell_of,
             const int* cell_pos, const double* posc, const int* molc, int nx, int ny, int nz,
             double csx, double csy, double csz, double ox, double oy, double oz, int periodic, double rc, double s_c, int half,
             int* count, const long* start, int* out, int* flags, void* stream) {
  TM_REQUIRE(N >= 0, "tm_pairs: bad sizes");
  TM_REQUIRE(start == nullptr || out != nullptr, "tm_pairs: fill pass needs an output array");
  if (cell_atoms != nullptr) {
    int k = (int)ceil(rc / fmin(csx, fmin(csy, csz))) + 1;
    TM_REQUIRE((2 * k + 3) * (2 * k + 3) * 2 <= 1024,
               "tm_pairs: cells of %.2f A are too small for rc %.2f", fmin(csx, fmin(csy, csz)), rc);
  }
  if (N == 0) return TM_OK;
  hipStream_t s = (hipStream_t)stream;
  CellGrid g = make_grid(cell_start, cell_atoms, cell_of, cell_pos, posc, molc, nx, ny, nz, csx, csy,
                         csz, ox, oy, oz, periodic, rc);
  if (start == nullptr)
    pairs_kernel<false><<<tm_div_up(N, NL_WAVES), NL_WAVES * 64, 0, s>>>(
        N, pos, mol, mol_start, nreal, box, g, s_c, half, count, nullptr, nullptr, flags);
  else
    pairs_kernel<true><<<tm_div_up(N, NL_WAVES), NL_WAVES * 64, 0, s>>>(
        N, pos, mol, mol_start, nreal, box, g, s_c, half, count, start, out, flags);
  TM_LAUNCH_CHECK();
  return TM_OK;
}

}  // extern "C"
