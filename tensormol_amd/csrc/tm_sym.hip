// ANI-style radial and angular symmetry functions and their adjoint.
//
// Forward restates TFSymRSet_Linear_WithEle (TensorMol/TFDescriptors/
// RawSymFunc.py:1696-1755), TFSymASet_Linear_WithEle (:868-962) and the
// concatenation of TFSymSet_Scattered_Linear_WithEle (:2223-2265):
//   G[i, l*NR + s]          = sum_j exp(-eta (r_ij - Rs_s)^2) fc_r(r_ij)
//   G[i, nele*NR + p*NA*NT + t*NA + s]
//        = sum_{j<k} 2^(1-zeta) (1 + cos(theta_ijk - theta_t))^zeta
//                     exp(-eta ((r_ij + r_ik)/2 - Rs_s)^2) fc_a(r_ij) fc_a(r_ik)
// with fc(r) = 0.5 (cos(3.14159265359 r / Rc) + 1) and the neighbour list as
// the only cutoff mask.  cos(theta - theta_t) is evaluated as
// c cos(theta_t) + s sin(theta_t) with c = cos(theta) and s = sin(theta) >= 0
// (taken from the cross product of the two bonds), which is the same function
// as the reference's acos-then-cos.
//
// One wavefront per centre atom.  Neighbour geometry is staged in LDS; the
// angular triples of a centre are enumerated on the fly from its short
// sub-list, grouped by element pair, so nothing per-triple is stored in HBM.
// Every output element is written exactly once; no atomics.
//
// The adjoint takes dE/dG per atom and returns, for every neighbour slot
// (i -> j), the vector w_ij = dE/d(x_j - x_i) of centre i's descriptor; a
// gather over mirror slots turns those into per-atom gradients without
// atomics, so forces are bitwise reproducible.
#include "tm_common.h"
#include "tm_sums.h"

namespace {

constexpr int SYM_WAVES = 4;
constexpr int MAX_ROW = 256;      // widest radial row (row stride) the kernels stage in LDS
constexpr int NR_MAX = 64;        // radial shells
constexpr int NA = 8;             // angular shells (fixed by the lane mapping)
constexpr int NT = 8;             // angular theta points

struct SymArgs {
  int nele, nelep, nr;            // elements, element pairs, radial shells
  int D;                          // descriptor length
  float eta, zeta, rr, ra;        // AN1 parameters and cutoffs (A)
  float two_1mz;                  // 2^(1-zeta)
  int zeta_int;                   // zeta when it is a small positive integer, else 0
  float kr, ka;                    // pi / Rc_r, pi / Rc_a (pi as the reference's literal)
  float rs_r[NR_MAX];
  float rs_a[NA];
  float cos_t[NT], sin_t[NT];
};

constexpr float PI_LIT = 3.14159265359f;

// b^zeta: ZI > 0 is zeta known at compile time (a few multiplies); ZI = 0 reads
// zeta from the arguments (square-and-multiply when it is a small integer).
template <int ZI>
__device__ __forceinline__ float powz(float b, const SymArgs& a) {
  const int zi = ZI > 0 ? ZI : a.zeta_int;
  if (zi > 0) {   // square-and-multiply over the 7 bits of zeta <= 64
    float r = 1.f, x = b;
#pragma unroll
    for (int k = 0; k < 7; ++k) {
      r = ((zi >> k) & 1) ? r * x : r;
      x *= x;
    }
    return r;
  }
  return b > 0.f ? __expf(a.zeta * __logf(b)) : 0.f;
}

// (1 + v)^zeta and zeta (1 + v)^(zeta - 1) for b = 1 + v >= 0, without a division
// when zeta is a small integer: r = b^(zeta - 1) by square-and-multiply.
template <int ZI>
__device__ __forceinline__ void powz_pair(float b, const SymArgs& a, float& Az, float& dAz) {
  const int zi = ZI > 0 ? ZI : a.zeta_int;
  if (zi > 0) {
    const int e = zi - 1;
    float r = 1.f, x = b;
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      r = ((e >> k) & 1) ? r * x : r;
      x *= x;
    }
    Az = r * b;
    dAz = (ZI > 0 ? (float)ZI : a.zeta) * r;
    return;
  }
  Az = b > 0.f ? __expf(a.zeta * __logf(b)) : 0.f;
  dAz = b > 0.f ? a.zeta * Az * __builtin_amdgcn_rcpf(b) : 0.f;
}

// A centre's row in LDS: x_j - x_i and r, and the radial cutoff where many
// lanes read it.  What one lane needs once (elements, the angular cutoff) is
// formed where it is used, which keeps the kernels at six to seven waves per
// SIMD.
template <int RC>
struct RowLdsFwd {
  static constexpr bool has_fc = true;
  float4 d[SYM_WAVES][RC];
  float fc[SYM_WAVES][RC];
};
template <int RC>
struct RowLdsAdj {
  static constexpr bool has_fc = false;
  float4 d[SYM_WAVES][RC];
};

__device__ __forceinline__ float cutoff_fc(float k, float r) { return 0.5f * (__cosf(k * r) + 1.0f); }

// sin of the angle between the bond vectors dj and dk (inv = 1 / (|dj| |dk|)),
// from the cross product: its relative error grows as eps / sin(theta) for
// nearly collinear bonds, where sqrt(1 - cos^2) loses every digit (eps / sin^2).
__device__ __forceinline__ float sin_between(const float4& dj, const float4& dk, float inv) {
  const float cx = dj.y * dk.z - dj.z * dk.y;
  const float cy = dj.z * dk.x - dj.x * dk.z;
  const float cz = dj.x * dk.y - dj.y * dk.x;
  return fminf(sqrtf(cx * cx + cy * cy + cz * cz) * inv, 1.0f);
}
__device__ __forceinline__ float cutoff_dfc(float k, float r) { return -0.5f * k * __sinf(k * r); }

// A lane's slots of row i; slots past the row's end hold anything.  Read
// before the row's length is known, so that the two loads overlap.
template <int RC>
__device__ __forceinline__ void row_slots(int (&jq)[RC / 64], const int* __restrict__ nbr, int i,
                                          int lane, int ldr) {
#pragma unroll
  for (int k = 0; k < RC / 64; ++k) {
    const int q = lane + 64 * k;
    jq[k] = q < ldr ? nbr[(long)i * ldr + q] : 0;
  }
}

// more(q, j, d): what else slot q needs
template <int RC, class LDS, class More>
__device__ __forceinline__ void load_row(int i, int w, int lane, const double* __restrict__ pos,
                                         const double* __restrict__ box, const int* __restrict__ mol,
                                         const int (&jq)[RC / 64], int n, const SymArgs& a, LDS& L,
                                         More more) {
  // minimum image with the reciprocal edge (iL = 0 for open boundaries): it
  // differs from d - L rint(d / L) only at |d| = L/2, far beyond the cutoff
  double Lx = 0, Ly = 0, Lz = 0, iLx = 0, iLy = 0, iLz = 0;
  if (box != nullptr) {
    int m = mol[i];
    Lx = box[3 * m]; Ly = box[3 * m + 1]; Lz = box[3 * m + 2];
    iLx = 1.0 / Lx; iLy = 1.0 / Ly; iLz = 1.0 / Lz;
  }
  const double xi = pos[3 * i], yi = pos[3 * i + 1], zi = pos[3 * i + 2];
#pragma unroll
  for (int k = 0; k < RC / 64; ++k) {
    const int q = lane + 64 * k, j = jq[k];
    if (q >= n) break;
    double ex = pos[3 * j] - xi, ey = pos[3 * j + 1] - yi, ez = pos[3 * j + 2] - zi;
    float dx = (float)(ex - Lx * rint(ex * iLx));
    float dy = (float)(ey - Ly * rint(ey * iLy));
    float dz = (float)(ez - Lz * rint(ez * iLz));
    float r = sqrtf(dx * dx + dy * dy + dz * dz + 1e-27f);
    L.d[w][q] = make_float4(dx, dy, dz, r);
    if constexpr (LDS::has_fc) L.fc[w][q] = cutoff_fc(a.kr, r);
    more(q, j, L.d[w][q]);
  }
}

// Segment boundary e of a lane register that holds boundary l in lane l.
__device__ __forceinline__ int seg_at(int v, int e) { return __builtin_amdgcn_readlane(v, e); }

template <int CTRL>
__device__ __forceinline__ float dpp_swap(float x) {   // another lane's x of the same quad
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL,
                                                               0xf, 0xf, true));
}
// x of lane ^ 4: lanes 0-3 and 8-11 of a row read four lanes up, the others down
__device__ __forceinline__ float dpp_swap4(float x) {
  const int v = __builtin_bit_cast(int, x);
  const int up = __builtin_amdgcn_update_dpp(0, v, 0x104, 0xf, 0x5, false);
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(up, v, 0x114, 0xf, 0xa, false));
}

// Sum of v[s] over the 8 lanes of a group, for s = the lane's own number g:
// ((0 + 1) + (2 + 3)) + ((4 + 5) + (6 + 7)).  Each step hands half of the
// shells that are left to the partner and keeps the other half.
__device__ __forceinline__ float group_sum8(const float (&v)[8], int g) {
  const bool b0 = g & 1, b1 = g & 2, b2 = g & 4;
  float x[4], y[2];
#pragma unroll
  for (int k = 0; k < 4; ++k)
    x[k] = (b0 ? v[2 * k + 1] : v[2 * k]) + dpp_swap<0xB1>(b0 ? v[2 * k] : v[2 * k + 1]);
#pragma unroll
  for (int k = 0; k < 2; ++k)
    y[k] = (b1 ? x[2 * k + 1] : x[2 * k]) + dpp_swap<0x4E>(b1 ? x[2 * k] : x[2 * k + 1]);
  return (b2 ? y[1] : y[0]) + dpp_swap4(b2 ? y[0] : y[1]);
}

// The angular functions of one centre, 64 triples at a time.  Triples are
// ordered by element pair (ea <= eb), inside a pair by (k, j), so each pair is
// a contiguous range of the enumeration.
// Phase A: lane = triple, stage(ja, kb) puts its geometry into LDS (ja, kb:
// places in the angular sub-list).  Phase B: lane = (theta point t, triple
// group g); it takes every 8th triple u of a pair's range, term(u, acc) adds it
// to one accumulator per shell.  When a pair ends, the 8 groups are summed and
// lane (t, g) writes shell s = g.
// av: boundary e of the sub-list's element segments in lane e.
//
// An atom of an organic molecule has some 50 triples in ten pairs, so what a
// pair costs besides its triples decides.  The walk over the pairs is
// wave-uniform (scalar registers) and keeps its place from chunk to chunk, an
// empty pair is one store, the 8 groups are summed with lane permutes of the
// vector unit (24 LDS permutes before), and members' places come from LDS, not
// from the list in memory.  Angular part of a wave, median cycles: 12,288-atom
// water box 10,400 -> 7,100, 24,000-atom C/H/N/O sphere 33,200 -> 16,300.
// Lists and descriptors of 37 chains (2,139 atoms) 38.5 -> 25.4 us, of the box
// 76 -> 64; descriptors of 10,398 chain atoms 61 -> 36 and their tangent
// 74 -> 47.  Reading the next pair's first triples ahead and keeping the pairs'
// ranges per lane gained nothing.
template <class Out, class Stage, class Term>
__device__ __forceinline__ void angular_pass(int lane, int nele, int nelep, int av, int ntrip,
                                             float scale, Out put, Stage stage, Term term) {
  const int g = lane & 7;
  float acc[NA];
#pragma unroll
  for (int s = 0; s < NA; ++s) acc[s] = 0.f;
  int p = 0, ea = 0, eb = 0, T = 0;   // pair in progress and its first triple
  auto pairs = [&](int x, int y) {
    const int la = seg_at(av, x + 1) - seg_at(av, x);
    return x == y ? la * (la - 1) / 2 : la * (seg_at(av, y + 1) - seg_at(av, y));
  };
  for (int base = 0; base < ntrip; base += 64) {
    const int cnt = min(64, ntrip - base), t = base + lane;
    {
      // place of triple t: walk over the pairs that this chunk touches
      int sa = 0, sb = 0, la = 0, tl = 0;
      int xa = ea, xb = eb, X = T;
      while (X < base + cnt && xa < nele) {
        const int s0 = seg_at(av, xa), l0 = seg_at(av, xa + 1) - s0, s1 = seg_at(av, xb);
        const bool in = t >= X;
        sa = in ? s0 : sa;
        sb = in ? s1 : sb;
        la = in ? (xa == xb ? 0 : l0) : la;
        tl = in ? t - X : tl;
        X += pairs(xa, xb);
        if (++xb == nele) xb = ++xa;
      }
      int ja, kb;
      if (la == 0) {   // k-major triangle: tl = k (k - 1) / 2 + j, j < k
        int k = (int)((1.0f + sqrtf(1.0f + 8.0f * (float)tl)) * 0.5f);
        k -= k * (k - 1) / 2 > tl ? 1 : 0;
        k += (k + 1) * k / 2 <= tl ? 1 : 0;
        kb = sb + k;
        ja = sa + (tl - k * (k - 1) / 2);
      } else {         // (tl + 1/2) / la is at least 1 / (2 la) away from an integer
        const int k = (int)(((float)tl + 0.5f) * __builtin_amdgcn_rcpf((float)la));
        kb = sb + k;
        ja = sa + (tl - k * la);
      }
      if (t < ntrip) stage(ja, kb);
    }
    __syncwarp();
    while (p < nelep) {
      const int n = pairs(ea, eb), Te = T + n;
      const int lo = max(T - base, 0), hi = min(Te - base, cnt);   // chunk-local part
      for (int u = lo + ((g - lo) & 7); u < hi; u += 8) term(u, acc);
      if (Te > base + cnt) break;   // goes on in the next chunk
      float x = 0.f;
      if (n > 0) {
        x = group_sum8(acc, g);
#pragma unroll
        for (int s = 0; s < NA; ++s) acc[s] = 0.f;
      }
      put(p * 64 + lane, scale * x);
      T = Te;
      ++p;
      if (++eb == nele) eb = ++ea;
    }
    __syncwarp();
  }
  for (; p < nelep; ++p) put(p * 64 + lane, 0.f);
}

// A training step's GEMMs read descriptors and tangents as BF16 rows in element
// order.  With ROWS the kernels below write those rows themselves (rounded to
// nearest even): places[4 i ..] = addresses of atom i's descriptor row, its
// tangent row, its float and its BF16 slot of dLoss/dy.
// Copying them from FP32 arrays afterwards took launches of 15 and 11 us on
// 10,398 atoms with 768 descriptors, bound by memory, where these kernels are
// bound by instructions and have the bandwidth to spare: training step 600 ->
// 576 us.  The descriptors are written in FP32 as well, for whoever reads them.
__device__ __forceinline__ unsigned short bf16_of(float x) {
  return __builtin_bit_cast(unsigned short, (__bf16)x);
}


template <int ZI, int RC, bool ROWS>
__global__ void __launch_bounds__(SYM_WAVES * 64)
sym_fwd_kernel(int N, const double* __restrict__ pos, const double* __restrict__ box,
               const int* __restrict__ mol, const int* __restrict__ elem,
               const int* __restrict__ nbr, const int* __restrict__ ncnt,
               const int* __restrict__ rseg, const int* __restrict__ ang,
               const int* __restrict__ acnt, const int* __restrict__ aseg, int ldr, int lda,
               SymArgs a, float* __restrict__ G, int ldg, int* __restrict__ rev,
               int* __restrict__ flags, const long* __restrict__ places) {
  __shared__ RowLdsFwd<RC> L;
  __shared__ float4 tq[SYM_WAVES][64];        // per triple: (cos theta, sin theta, fc_j fc_k, -)
  __shared__ float4 tR[SYM_WAVES][64][NA / 4];   // per triple: exp(-eta (ravg - Rs_s)^2), s = 0..7
  __shared__ unsigned char apos[SYM_WAVES][RC];   // row position of each sub-list member
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int i = blockIdx.x * SYM_WAVES + w;
  if (i >= N) return;   // only wave-level synchronisation below
  int jq[RC / 64];
  row_slots<RC>(jq, nbr, i, lane, ldr);
  const int n = min(ncnt[i], RC), m = min(acnt[i], lda);
  // element segments of the row and of the sub-list, boundary e in lane e
  const int le = min(lane, a.nele);
  const int rv = min(rseg[(long)i * (a.nele + 1) + le], n);
  const int av = min(aseg[(long)i * (a.nele + 1) + le], m);
  for (int x = lane; x < m; x += 64) apos[w][x] = (unsigned char)ang[(long)i * lda + x];
  load_row<RC>(i, w, lane, pos, box, mol, jq, n, a, L, [](int, int, const float4&) {});
  __syncwarp();
  float* Gi = G + (long)i * ldg;
  unsigned short* Xi = nullptr;
  if constexpr (ROWS) Xi = reinterpret_cast<unsigned short*>(places[4l * i]);
  auto put = [&](int f, float v) {
    Gi[f] = v;
    if constexpr (ROWS) Xi[f] = bf16_of(v);
  };
  // ---------------- radial: lane = (half h, shell s)
  {
    const int h = lane >> 5, s = lane & 31;
    for (int e = 0; e < a.nele; ++e) {
      const int lo = seg_at(rv, e), hi = seg_at(rv, e + 1);
      for (int s0 = 0; s0 < a.nr; s0 += 32) {
        int ss = s0 + s;
        float rs = ss < a.nr ? a.rs_r[ss] : 0.f;
        float acc = 0.f;
#pragma unroll 4
        for (int q = lo + h; q < hi; q += 2) {
          float r = L.d[w][q].w;
          float x = r - rs;
          acc += __expf(-a.eta * x * x) * L.fc[w][q];
        }
        acc += __shfl_xor(acc, 32, 64);
        if (h == 0 && ss < a.nr) put(e * a.nr + ss, acc);
      }
    }
  }
  // ---------------- angular
  // Phase B forms (1 + cos(theta - theta_t))^zeta fc_j fc_k once per triple and
  // theta point and adds it times R_s to the shells.
  const float ct = a.cos_t[lane >> 3], st = a.sin_t[lane >> 3];
  angular_pass(
      lane, a.nele, a.nelep, av, m * (m - 1) / 2, a.two_1mz,
      [&](int f, float v) { put(a.nele * a.nr + f, v); },
      [&](int ja, int kb) {
        const int qj = apos[w][ja], qk = apos[w][kb];
        float4 dj = L.d[w][qj], dk = L.d[w][qk];
        const float inv = __builtin_amdgcn_rcpf(dj.w * dk.w);
        float c = (dj.x * dk.x + dj.y * dk.y + dj.z * dk.z) * inv;
        c = fminf(fmaxf(c, -1.0f), 1.0f);
        float sn = sin_between(dj, dk, inv);
        float ravg = 0.5f * (dj.w + dk.w);
        tq[w][lane] = make_float4(c, sn, cutoff_fc(a.ka, dj.w) * cutoff_fc(a.ka, dk.w), 0.f);
        float R[NA];
#pragma unroll
        for (int s = 0; s < NA; ++s) {
          float x = ravg - a.rs_a[s];
          R[s] = __expf(-a.eta * x * x);
        }
        tR[w][lane][0] = make_float4(R[0], R[1], R[2], R[3]);
        tR[w][lane][1] = make_float4(R[4], R[5], R[6], R[7]);
      },
      [&](int u, float (&acc)[NA]) {
        const float4 q = tq[w][u];
        const float4 r0 = tR[w][u][0], r1 = tR[w][u][1];
        const float AF = powz<ZI>(1.0f + (q.x * ct + q.y * st), a) * q.z;
        acc[0] += AF * r0.x; acc[1] += AF * r0.y; acc[2] += AF * r0.z; acc[3] += AF * r0.w;
        acc[4] += AF * r1.x; acc[5] += AF * r1.y; acc[6] += AF * r1.z; acc[7] += AF * r1.w;
      });
  if (rev == nullptr) return;
  // Mirror slots (the rev output of the neighbour build): rev[i*ldr+q] =
  // j*ldr + position of i in row j, found by binary search in the element
  // segment of row j that holds i (rows are sorted by (element, index)).
  const int ei = elem[i];
#pragma unroll
  for (int k = 0; k < RC / 64; ++k) {
    const int q = lane + 64 * k, j = jq[k];
    if (q >= n) break;
    int lo = rseg[(long)j * (a.nele + 1) + ei];
    int hi = rseg[(long)j * (a.nele + 1) + ei + 1];
    const int* row = nbr + (long)j * ldr;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (row[mid] < i) lo = mid + 1; else hi = mid;
    }
    if (lo < ncnt[j] && row[lo] == i) {
      rev[(long)i * ldr + q] = (int)((long)j * ldr + lo);
    } else {
      rev[(long)i * ldr + q] = (int)((long)i * ldr + q);   // unmatched (truncated row)
      atomicOr(&flags[TM_FLAG_NB_OVERFLOW], 2);
    }
  }
}

// dE/dG (two contributions combined: gE + u_i * gQ) -> w slots.
//
// Angular part: triples (a, b) of sub-list members a < b, numbered t =
// b (b - 1) / 2 + a.  A window of ADJ_TC triples is evaluated, lane = triple,
// its contributions to a and to b left in LDS; then lane = member adds its own.
// Numbered like this, a member's triples come in ascending order of the
// partner, so "add over partners" is a plain loop whose LDS reads do not
// depend on each other.  (Numbered by element pair, as in the forward, a
// member had to search its triples block by block: 7,000 of a wave's 26,000
// cycles on the water box, 15,000 of 43,000 on the C/H/N/O sphere.)
//
// What bounds it now: the instructions of the triples (some 450 per 64) and of
// the 32 radial shells per neighbour, and the dE/dG rows (1 to 6 KB per
// centre), which are on their way while the neighbour row is staged.
// Adjoint and force gather: 12,288-atom box 54 -> 38 us, 24,000-atom sphere
// 175 -> 81 us, 2,139 chain atoms 41 -> 21 us.
constexpr int ADJ_TC = 128;   // triples per window, two per lane

template <int ZI, int RC>
__global__ void __launch_bounds__(SYM_WAVES * 64) __attribute__((amdgpu_waves_per_eu(RC == 128 ? 6 : 4)))
sym_adj_kernel(int N, const double* __restrict__ pos, const double* __restrict__ box,
               const int* __restrict__ mol, const int* __restrict__ elem,
               const int* __restrict__ nbr, const int* __restrict__ ncnt,
               const int* __restrict__ ang, const int* __restrict__ acnt, int ldr, int lda,
               SymArgs a, const float* __restrict__ gE, const float* __restrict__ gQ,
               const float* __restrict__ u, const double* __restrict__ phi,
               const double* __restrict__ phimean, int ldg, int vec4,
               float4* __restrict__ wslot) {
  constexpr int NQ = RC / 64;   // neighbours (and members) per lane
  constexpr int TU = ZI > 0 ? NT : 1;
  __shared__ RowLdsAdj<RC> L;
  // window: contributions of each triple to b (planes 0-2) and to a (3-5), x y z;
  // afterwards the members' sums by neighbour slot
  __shared__ float cw[SYM_WAVES][6 * ADJ_TC];
  static_assert(3 * RC <= 6 * ADJ_TC, "the members' sums reuse the window");
  __shared__ int mem[SYM_WAVES][RC];   // member: position in the row | element << 16
  extern __shared__ float4 gdyn[];     // dE/dG of each wave's centre, D rounded up to 4 floats
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int i = blockIdx.x * SYM_WAVES + w;
  if (i >= N) return;   // only wave-level synchronisation below
  // the radial part as it is, the angular part from a 16-byte boundary
  const int off = a.nele * a.nr, offa = (off + 3) & ~3, D4 = (a.D + offa - off + 3) >> 2;
  float* gw = reinterpret_cast<float*>(gdyn + w * D4);
  int jq[NQ];
  row_slots<RC>(jq, nbr, i, lane, ldr);
  const int n = min(ncnt[i], RC), m = min(min(acnt[i], lda), RC);
  // charge upstream u_i = phi_i - mean_m(phi) (as tm_charge_upstream) unless given
  const float ui = gQ == nullptr ? 0.f
                   : (u != nullptr ? u[i] : (float)(phi[i] - phimean[mol[i]]));
  const float* gEi = gE + (long)i * ldg;
  const float* gQi = gQ + (long)i * ldg;
  if (vec4) {   // D <= 1024: at most four float4 per lane, all on their way before the row
    float4 v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int f = 4 * (lane + 64 * k);
      if (f < a.D) {
        v[k] = *reinterpret_cast<const float4*>(gEi + f);
        if (gQ != nullptr) {
          const float4 z = *reinterpret_cast<const float4*>(gQi + f);
          v[k].x += ui * z.x; v[k].y += ui * z.y; v[k].z += ui * z.z; v[k].w += ui * z.w;
        }
      }
    }
    load_row<RC>(i, w, lane, pos, box, mol, jq, n, a, L, [](int, int, const float4&) {});
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int f = 4 * (lane + 64 * k);
      if (f < a.D) *reinterpret_cast<float4*>(gw + f) = v[k];   // off % 4 == 0 here
    }
  } else {
    for (int f = lane; f < a.D; f += 64) {
      float v = gEi[f];
      if (gQ != nullptr) v += ui * gQi[f];
      gw[f < off ? f : f + offa - off] = v;
    }
    load_row<RC>(i, w, lane, pos, box, mol, jq, n, a, L, [](int, int, const float4&) {});
  }
  for (int x = lane; x < m; x += 64) {
    const int q = ang[(long)i * lda + x];
    mem[w][x] = q | (elem[nbr[(long)i * ldr + q]] << 16);
  }
  __syncwarp();
  // ---------------- radial: lane = neighbour
  const float kr = a.kr;
  float wx[NQ], wy[NQ], wz[NQ];
#pragma unroll
  for (int k = 0; k < NQ; ++k) {
    const int q = lane + 64 * k;
    wx[k] = wy[k] = wz[k] = 0.f;
    if (q < n) {
      float4 d = L.d[w][q];
      float r = d.w;
      int e = elem[nbr[(long)i * ldr + q]];
      float fc = cutoff_fc(kr, r);
      float dfc = cutoff_dfc(kr, r);
      float dEdr = 0.f;
      const float* gr = gw + e * a.nr;
      auto shell = [&](float gs, int s) {
        float x = r - a.rs_r[s];
        float ex = __expf(-a.eta * x * x);
        dEdr += gs * ex * (dfc - 2.0f * a.eta * x * fc);
      };
      if ((a.nr & 3) == 0) {
        for (int s = 0; s < a.nr; s += 4) {
          const float4 g4 = *reinterpret_cast<const float4*>(gr + s);
          shell(g4.x, s); shell(g4.y, s + 1); shell(g4.z, s + 2); shell(g4.w, s + 3);
        }
      } else {
        for (int s = 0; s < a.nr; ++s) shell(gr[s], s);
      }
      float sc = dEdr * __builtin_amdgcn_rcpf(r);
      wx[k] = sc * d.x;
      wy[k] = sc * d.y;
      wz[k] = sc * d.z;
    }
  }
  // ---------------- angular
  const int ntrip = m * (m - 1) / 2;
  float ax[NQ], ay[NQ], az[NQ];   // sums of members lane, lane + 64, ...
#pragma unroll
  for (int k = 0; k < NQ; ++k) ax[k] = ay[k] = az[k] = 0.f;
  float* cwv = cw[w];
  for (int T0 = 0; T0 < ntrip; T0 += ADJ_TC) {
    const int len = min(ADJ_TC, ntrip - T0);
    for (int uu = lane; uu < len; uu += 64) {
      const int t = T0 + uu;
      // b: the largest with b (b - 1) / 2 <= t
      int kb = (int)((1.0f + __builtin_amdgcn_sqrtf(1.0f + 8.0f * (float)t)) * 0.5f);
      if (kb * (kb - 1) / 2 > t) --kb;
      if ((kb + 1) * kb / 2 <= t) ++kb;
      const int ja = t - kb * (kb - 1) / 2;
      const int mj = mem[w][ja], mk = mem[w][kb];
      const int ej = mj >> 16, ek = mk >> 16;   // ej <= ek: the sub-list is sorted
      const int p = ej * a.nele - ej * (ej - 1) / 2 + (ek - ej);
      float4 dj = L.d[w][mj & 0xffff], dk = L.d[w][mk & 0xffff];
      float rj = dj.w, rk = dk.w;
      const float irj = __builtin_amdgcn_rcpf(rj), irk = __builtin_amdgcn_rcpf(rk);
      float inv = irj * irk;
      float c = (dj.x * dk.x + dj.y * dk.y + dj.z * dk.z) * inv;
      c = fminf(fmaxf(c, -1.0f), 1.0f);
      float sn = sin_between(dj, dk, inv);
      float cos_over_sin = sn > 1e-6f ? c * __builtin_amdgcn_rcpf(sn) : 0.f;
      float ravg = 0.5f * (rj + rk);
      float fj = cutoff_fc(a.ka, rj), fk = cutoff_fc(a.ka, rk);
      float dfj = cutoff_dfc(a.ka, rj), dfk = cutoff_dfc(a.ka, rk);
      float F = fj * fk;
      float R[NA], Rp[NA];
#pragma unroll
      for (int s = 0; s < NA; ++s) {
        float x = ravg - a.rs_a[s];
        R[s] = __expf(-a.eta * x * x);
        Rp[s] = -2.0f * a.eta * x * R[s];
      }
      const float4* gp = reinterpret_cast<const float4*>(gw + offa + p * 64);
      float dEdc = 0.f, dEdrav = 0.f, dEdF = 0.f;
#pragma unroll TU
      for (int tt = 0; tt < NT; ++tt) {
        const float4 g0 = gp[2 * tt], g1 = gp[2 * tt + 1];
        const float gv[NA] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
        float S = 0.f, Sp = 0.f;
#pragma unroll
        for (int s = 0; s < NA; ++s) {
          S += gv[s] * R[s];
          Sp += gv[s] * Rp[s];
        }
        float v = c * a.cos_t[tt] + sn * a.sin_t[tt];
        float b = 1.0f + v;
        float Az, dAz;                             // (1+v)^zeta, zeta (1+v)^(zeta-1)
        powz_pair<ZI>(b, a, Az, dAz);
        float dv = a.cos_t[tt] - cos_over_sin * a.sin_t[tt];
        dEdc += dAz * dv * S;
        dEdrav += Az * Sp;
        dEdF += Az * S;
        __builtin_amdgcn_sched_barrier(0);   // one theta point's row in registers at a time
      }
      // the common factor 2^(1 - zeta) of every term, applied once
      dEdc *= a.two_1mz * F;
      dEdrav *= a.two_1mz * F;
      dEdF *= a.two_1mz;
      // chain rule into d_j, d_k
      float cj = (dEdrav * 0.5f + dEdF * dfj * fk - dEdc * c * irj) * irj;
      float ck = (dEdrav * 0.5f + dEdF * fj * dfk - dEdc * c * irk) * irk;
      float x = dEdc * inv;
      cwv[uu] = ck * dk.x + x * dj.x;
      cwv[ADJ_TC + uu] = ck * dk.y + x * dj.y;
      cwv[2 * ADJ_TC + uu] = ck * dk.z + x * dj.z;
      cwv[3 * ADJ_TC + uu] = cj * dj.x + x * dk.x;
      cwv[4 * ADJ_TC + uu] = cj * dj.y + x * dk.y;
      cwv[5 * ADJ_TC + uu] = cj * dj.z + x * dk.z;
    }
    __syncwarp();
    // members add their triples of the window in ascending order of the partner
    // y: below the member its number is x (x - 1) / 2 + y, above it y (y - 1) / 2 + x
    const int last = T0 + len - 1;
    int bh = (int)((1.0f + __builtin_amdgcn_sqrtf(1.0f + 8.0f * (float)last)) * 0.5f);
    if (bh * (bh - 1) / 2 > last) --bh;
    if ((bh + 1) * bh / 2 <= last) ++bh;   // the window's last b
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
      const int x = lane + 64 * k;
      if (64 * k > bh) break;
      const int tx = x * (x - 1) / 2 - T0;
      int ty = -T0;   // y (y - 1) / 2 - T0
#pragma unroll 4
      for (int y = 0; y <= bh; ++y) {
        const bool below = y < x;
        const int t = below ? tx + y : ty + x;
        const bool ok = (unsigned)t < (unsigned)len && y != x && x <= bh;
        const float* c = cwv + (ok ? t : 0) + (below ? 0 : 3 * ADJ_TC);
        const float cx = c[0], cy = c[ADJ_TC], cz = c[2 * ADJ_TC];
        ax[k] += ok ? cx : 0.f;
        ay[k] += ok ? cy : 0.f;
        az[k] += ok ? cz : 0.f;
        ty += y;
      }
    }
    __syncwarp();
  }
  if (m > 1) {   // the members' sums, by neighbour slot
    for (int q = lane; q < n; q += 64) cwv[q] = cwv[RC + q] = cwv[2 * RC + q] = 0.f;
    __syncwarp();
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
      const int x = lane + 64 * k;
      if (x < m) {
        const int q = mem[w][x] & 0xffff;
        cwv[q] = ax[k];
        cwv[RC + q] = ay[k];
        cwv[2 * RC + q] = az[k];
      }
    }
    __syncwarp();
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
      const int q = lane + 64 * k;
      if (q < n) {
        wx[k] += cwv[q];
        wy[k] += cwv[RC + q];
        wz[k] += cwv[2 * RC + q];
      }
    }
  }
#pragma unroll
  for (int k = 0; k < NQ; ++k) {
    const int q = lane + 64 * k;
    if (q < n) wslot[(long)i * ldr + q] = make_float4(wx[k], wy[k], wz[k], 0.f);
  }
}

// Velocity Verlet state advanced by the force gather (VV = true): the kick of
// the step with the gathered force, then the drift of the next step, with the
// operations of vv_kick_kernel and vv_drift_kernel.
struct VVState {
  double dt;
  const double* m;
  double *v, *a, *ke, *x;
};

// grad_a = sum_n (w[rev(a,n)] - w[(a,n)]) + extra_a ; optional force output
// force = -scale * grad (J/mol/A when scale = JOULEPERHARTREE).  16 lanes per
// atom, each summing every 16th slot, then a fixed butterfly over the 16.
template <bool VV>
__device__ __forceinline__ void force_gather(int block, int N, int ldr, const int* __restrict__ ncnt,
                                             const int* __restrict__ rev,
                                             const float4* __restrict__ wslot,
                                             const double* __restrict__ extra, double scale,
                                             double* __restrict__ grad, double* __restrict__ force,
                                             const VVState& vv) {
  const long t = (long)block * 256 + threadIdx.x;
  const int a = (int)(t >> 4);
  const int sub = threadIdx.x & 15;
  double gx = 0, gy = 0, gz = 0;
  if (a < N) {
    const int n = ncnt[a];
    for (int q = sub; q < n; q += 16) {
      long sl = (long)a * ldr + q;
      float4 wo = wslot[sl];
      float4 wi = wslot[rev[sl]];
      gx += (double)wi.x - (double)wo.x;
      gy += (double)wi.y - (double)wo.y;
      gz += (double)wi.z - (double)wo.z;
    }
  }
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) {
    gx += __shfl_xor(gx, o, 16);
    gy += __shfl_xor(gy, o, 16);
    gz += __shfl_xor(gz, o, 16);
  }
  if (a >= N || sub != 0) return;
  if (extra != nullptr) {
    gx += extra[3 * a]; gy += extra[3 * a + 1]; gz += extra[3 * a + 2];
  }
  if (grad != nullptr) {
    grad[3 * a] = gx; grad[3 * a + 1] = gy; grad[3 * a + 2] = gz;
  }
  const double f[3] = {-scale * gx, -scale * gy, -scale * gz};
  if (force != nullptr) {
    force[3 * a] = f[0]; force[3 * a + 1] = f[1]; force[3 * a + 2] = f[2];
  }
  if (VV) {
    const double mi = vv.m[a], dt = vv.dt;
    double s = 0.0;
    for (int d = 0; d < 3; ++d) {
      double an = 1e-10 * f[d] / mi;
      double vn = vv.v[3 * a + d] + 0.5 * (vv.a[3 * a + d] + an) * dt;
      vv.v[3 * a + d] = vn;
      vv.a[3 * a + d] = an;
      s += vn * vn;
      vv.x[3 * a + d] = vv.x[3 * a + d] + vn * dt + 0.5 * an * dt * dt;
    }
    if (vv.ke) vv.ke[a] = 0.5 * mi * s;
  }
}

template <bool VV>
__global__ void __launch_bounds__(256)
force_gather_kernel(int N, int ldr, const int* __restrict__ ncnt, const int* __restrict__ rev,
                    const float4* __restrict__ wslot, const double* __restrict__ extra, double scale,
                    double* __restrict__ grad, double* __restrict__ force, VVState vv) {
  force_gather<VV>(blockIdx.x, N, ldr, ncnt, rev, wslot, extra, scale, grad, force, vv);
}

// The gather and the evaluation's closing sums, which read nothing it writes:
// the first nsum blocks sum (ONE: one system by blocks of atoms, else a block
// per molecule), the others gather.  Either alone is latency: 7.6 and 9.9 us
// for the 12,288-atom box, 3.9 and 5.6 us for 192 atoms.
template <bool ONE>
__global__ void __launch_bounds__(256)
force_gather_sums_kernel(int nsum, const int* __restrict__ mol_start, SumCols S, double* work, int N,
                         int ldr, const int* __restrict__ ncnt, const int* __restrict__ rev,
                         const float4* __restrict__ wslot, const double* __restrict__ extra,
                         double scale, double* __restrict__ grad, double* __restrict__ force) {
  __shared__ SumsLds L;
  const int b = blockIdx.x;
  if (b >= nsum) {
    force_gather<false>(b - nsum, N, ldr, ncnt, rev, wslot, extra, scale, grad, force, VVState{});
  } else if (ONE) {
    sums_by_blocks(S, N, b, nsum, work, L);
  } else {
    sums_of_molecule<256>(S, mol_start, b, L);
  }
}

// Tangent (forward-mode derivative) of the descriptor along per-atom
// displacements du: V[i, f] = sum_j dG[i, f]/d(x_j - x_i) . (du_j - du_i).
// It is the transpose of the adjoint above (same partial derivatives, the
// same guard where sin(theta) vanishes), contracted over neighbours instead
// of features; the lane layout and the write-once order are the forward's.
// Used for the weight gradient of a force loss: with u = dLoss/dF,
// dLoss/dW = -d/dW sum_i (dE_i/dG_i)(W) . V_i.
template <int RC>
struct JvpLds {
  float4 t[SYM_WAVES][RC];     // (du_j - du_i, dr_j = d_j . (du_j - du_i) / r_j)
  float dfc[SYM_WAVES][RC];    // d fc_r / dr
};

template <int ZI, int RC, bool ROWS>
__global__ void __launch_bounds__(SYM_WAVES * 64)
sym_jvp_kernel(int N, const double* __restrict__ pos, const double* __restrict__ box,
               const int* __restrict__ mol, const int* __restrict__ elem,
               const int* __restrict__ nbr, const int* __restrict__ ncnt,
               const int* __restrict__ rseg, const int* __restrict__ ang,
               const int* __restrict__ acnt, const int* __restrict__ aseg, int ldr, int lda,
               SymArgs a, const double* __restrict__ du, float* __restrict__ V, int ldg,
               const float* __restrict__ ybar, const long* __restrict__ places) {
  // the forward's row (the angular cutoff and its derivative are formed per
  // triple), which with the per-triple staging below fits 4 waves per SIMD
  __shared__ RowLdsFwd<RC> L;
  __shared__ JvpLds<RC> T;
  // per triple: (cos theta, sin theta, cos/sin guarded, fc_j fc_k), (d(fc_j fc_k),
  // d cos theta, d ravg, ravg), R_s for s = 0..7
  __shared__ float4 tqa[SYM_WAVES][64], tqb[SYM_WAVES][64];
  __shared__ float4 tR[SYM_WAVES][64][NA / 4];
  __shared__ unsigned char apos[SYM_WAVES][RC];   // row position of each sub-list member
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int i = blockIdx.x * SYM_WAVES + w;
  if (i >= N) return;   // only wave-level synchronisation below
  int jq[RC / 64];
  row_slots<RC>(jq, nbr, i, lane, ldr);
  const int n = min(ncnt[i], RC), m = min(acnt[i], lda);
  const int le = min(lane, a.nele);
  const int rv = min(rseg[(long)i * (a.nele + 1) + le], n);
  const int av = min(aseg[(long)i * (a.nele + 1) + le], m);
  for (int x = lane; x < m; x += 64) apos[w][x] = (unsigned char)ang[(long)i * lda + x];
  const float kr = a.kr, ka = a.ka;
  const double uxi = du[3 * i], uyi = du[3 * i + 1], uzi = du[3 * i + 2];
  load_row<RC>(i, w, lane, pos, box, mol, jq, n, a, L, [&](int q, int j, const float4& d) {
    const float tx = (float)(du[3 * j] - uxi), ty = (float)(du[3 * j + 1] - uyi);
    const float tz = (float)(du[3 * j + 2] - uzi);
    T.t[w][q] = make_float4(tx, ty, tz, (d.x * tx + d.y * ty + d.z * tz) * __builtin_amdgcn_rcpf(d.w));
    T.dfc[w][q] = -0.5f * kr * __sinf(kr * d.w);
  });
  __syncwarp();
  float* Vi = nullptr;
  unsigned short* Xi = nullptr;
  if constexpr (ROWS) {
    Xi = reinterpret_cast<unsigned short*>(places[4l * i + 1]);
    if (lane == 0) {
      const float y = ybar[i];
      *reinterpret_cast<float*>(places[4l * i + 2]) = y;
      *reinterpret_cast<unsigned short*>(places[4l * i + 3]) = bf16_of(y);
    }
  } else {
    Vi = V + (long)i * ldg;
  }
  auto put = [&](int f, float v) {
    if constexpr (ROWS) Xi[f] = bf16_of(v);
    else Vi[f] = v;
  };
  // ---------------- radial: lane = (half h, shell s)
  {
    const int h = lane >> 5, s = lane & 31;
    for (int e = 0; e < a.nele; ++e) {
      const int lo = seg_at(rv, e), hi = seg_at(rv, e + 1);
      for (int s0 = 0; s0 < a.nr; s0 += 32) {
        int ss = s0 + s;
        float rs = ss < a.nr ? a.rs_r[ss] : 0.f;
        float acc = 0.f;
#pragma unroll 4
        for (int q = lo + h; q < hi; q += 2) {
          float r = L.d[w][q].w;
          float x = r - rs;
          acc += __expf(-a.eta * x * x) * (T.dfc[w][q] - 2.0f * a.eta * x * L.fc[w][q]) *
                 T.t[w][q].w;
        }
        acc += __shfl_xor(acc, 32, 64);
        if (h == 0 && ss < a.nr) put(e * a.nr + ss, acc);
      }
    }
  }
  // ---------------- angular
  // Phase B forms (1 + cos(theta - theta_t))^zeta and its derivative once per
  // triple and theta point, and adds
  //   X R_s + Y R'_s,  X = A' v' c' F + A F',  Y = A r' F
  // to the shells (A = (1 + v)^zeta, v = cos(theta - theta_t), c', r', F' the
  // tangents of cos theta, ravg and fc_j fc_k).
  const float ct = a.cos_t[lane >> 3], st = a.sin_t[lane >> 3];
  angular_pass(
      lane, a.nele, a.nelep, av, m * (m - 1) / 2, a.two_1mz,
      [&](int f, float v) { put(a.nele * a.nr + f, v); },
      [&](int ja, int kb) {
        const int qj = apos[w][ja], qk = apos[w][kb];
        float4 dj = L.d[w][qj], dk = L.d[w][qk];
        float4 uj = T.t[w][qj], uk = T.t[w][qk];
        float rj = dj.w, rk = dk.w;
        const float irj = __builtin_amdgcn_rcpf(rj), irk = __builtin_amdgcn_rcpf(rk);
        float inv = irj * irk;
        float c = (dj.x * dk.x + dj.y * dk.y + dj.z * dk.z) * inv;
        c = fminf(fmaxf(c, -1.0f), 1.0f);
        float sn = sin_between(dj, dk, inv);
        float dc = (uj.x * dk.x + uj.y * dk.y + uj.z * dk.z + dj.x * uk.x + dj.y * uk.y +
                    dj.z * uk.z) * inv - c * (uj.w * irj + uk.w * irk);
        const float fj = cutoff_fc(ka, rj), fk = cutoff_fc(ka, rk);
        const float dfj = cutoff_dfc(ka, rj), dfk = cutoff_dfc(ka, rk);
        float ravg = 0.5f * (rj + rk);
        tqa[w][lane] = make_float4(c, sn, sn > 1e-6f ? c * __builtin_amdgcn_rcpf(sn) : 0.f,
                                   fj * fk);
        tqb[w][lane] = make_float4(dfj * uj.w * fk + fj * dfk * uk.w, dc, 0.5f * (uj.w + uk.w),
                                   ravg);
        float R[NA];
#pragma unroll
        for (int s = 0; s < NA; ++s) {
          float x = ravg - a.rs_a[s];
          R[s] = __expf(-a.eta * x * x);
        }
        tR[w][lane][0] = make_float4(R[0], R[1], R[2], R[3]);
        tR[w][lane][1] = make_float4(R[4], R[5], R[6], R[7]);
      },
      [&](int u, float (&acc)[NA]) {
        const float4 qa = tqa[w][u], qb = tqb[w][u];
        float Az, dAz;
        powz_pair<ZI>(1.0f + (qa.x * ct + qa.y * st), a, Az, dAz);
        const float dv = ct - qa.z * st;
        const float X = dAz * dv * qb.y * qa.w + Az * qb.x;
        const float Y2 = -2.0f * a.eta * Az * qb.z * qa.w;   // times (ravg - R_s) R_s
        const float4 r0 = tR[w][u][0], r1 = tR[w][u][1];
        const float R[NA] = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w};
#pragma unroll
        for (int s = 0; s < NA; ++s) acc[s] += R[s] * (X + Y2 * (qb.w - a.rs_a[s]));
      });
}

__global__ void total_energy_kernel(int B, const double* __restrict__ bp,
                                    const double* __restrict__ ext, double* __restrict__ out) {
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m < B) out[m] = (bp[m] + ext[2 * m]) + ext[2 * m + 1];
}

int fill_args(SymArgs& a, int nele, int nr, float eta, float zeta, float rr, float ra,
              const float* rs_r, const float* rs_a, const float* thetas) {
  TM_REQUIRE(nele > 0 && nele <= TM_MAX_ELE, "sym: bad nele %d", nele);
  TM_REQUIRE(nr > 0 && nr <= NR_MAX, "sym: radial shells %d outside 1..%d", nr, NR_MAX);
  a.nele = nele;
  a.nelep = nele * (nele + 1) / 2;
  a.nr = nr;
  a.D = nele * nr + a.nelep * NA * NT;
  TM_REQUIRE(a.D <= 1024, "sym: descriptor length %d above 1024", a.D);
  a.eta = eta; a.zeta = zeta; a.rr = rr; a.ra = ra;
  a.kr = PI_LIT / rr;
  a.ka = PI_LIT / ra;
  a.two_1mz = powf(2.0f, 1.0f - zeta);
  a.zeta_int = (zeta == floorf(zeta) && zeta >= 1.f && zeta <= 64.f) ? (int)zeta : 0;
  for (int s = 0; s < nr; ++s) a.rs_r[s] = rs_r[s];
  for (int s = 0; s < NA; ++s) a.rs_a[s] = rs_a[s];
  for (int t = 0; t < NT; ++t) {
    a.cos_t[t] = cosf(thetas[t]);
    a.sin_t[t] = sinf(thetas[t]);
  }
  return TM_OK;
}

}  // namespace

template <bool ROWS>
static int sym_forward(int N, const double* pos, const double* box, const int* mol, const int* elem,
                   const int* nbr, const int* ncnt, const int* rseg, const int* ang,
                   const int* acnt, const int* aseg, int ldr, int lda, int nele, int nr,
                   float eta, float zeta, float rr, float ra, const float* rs_r,
                   const float* rs_a, const float* thetas, float* G, int ldg, int* rev,
                   int* flags, const long* places, void* stream) {
  SymArgs a;
  int st = fill_args(a, nele, nr, eta, zeta, rr, ra, rs_r, rs_a, thetas);
  if (st) return st;
  TM_REQUIRE(ldg >= a.D, "tm_sym_forward: ldg %d < D %d", ldg, a.D);
  TM_REQUIRE(rev == nullptr || flags != nullptr, "tm_sym_forward: rev needs flags");
  TM_REQUIRE(ldr > 0 && ldr <= MAX_ROW && lda > 0 && lda <= ldr,
             "tm_sym_forward: strides %d/%d (need 0 < lda <= ldr <= %d)", ldr, lda, MAX_ROW);
  if (N == 0) return TM_OK;
  hipStream_t s = (hipStream_t)stream;
  // rows up to 128 entries stage in the smaller LDS layout (more waves per CU)
  decltype(&sym_fwd_kernel<0, 128, ROWS>) k =
      ldr <= 128 ? (a.zeta_int == 8 ? sym_fwd_kernel<8, 128, ROWS> : sym_fwd_kernel<0, 128, ROWS>)
                 : (a.zeta_int == 8 ? sym_fwd_kernel<8, 256, ROWS> : sym_fwd_kernel<0, 256, ROWS>);
  k<<<tm_div_up(N, SYM_WAVES), SYM_WAVES * 64, 0, s>>>(N, pos, box, mol, elem, nbr, ncnt, rseg,
                                                       ang, acnt, aseg, ldr, lda, a, G, ldg, rev,
                                                       flags, places);
  TM_LAUNCH_CHECK();
  return TM_OK;
}

template <bool ROWS>
static int sym_jvp(int N, const double* pos, const double* box, const int* mol, const int* elem,
               const int* nbr, const int* ncnt, const int* rseg, const int* ang, const int* acnt,
               const int* aseg, int ldr, int lda, int nele, int nr, float eta, float zeta,
               float rr, float ra, const float* rs_r, const float* rs_a, const float* thetas,
               const double* du, float* V, int ldg,
               const float* ybar, const long* places, void* stream) {
  SymArgs a;
  int st = fill_args(a, nele, nr, eta, zeta, rr, ra, rs_r, rs_a, thetas);
  if (st) return st;
  TM_REQUIRE(ROWS || ldg >= a.D, "tm_sym_jvp: ldg %d < D %d", ldg, a.D);
  TM_REQUIRE(ldr > 0 && ldr <= MAX_ROW && lda > 0 && lda <= ldr,
             "tm_sym_jvp: strides %d/%d (need 0 < lda <= ldr <= %d)", ldr, lda, MAX_ROW);
  if (N == 0) return TM_OK;
  hipStream_t s = (hipStream_t)stream;
  decltype(&sym_jvp_kernel<0, 128, ROWS>) k =
      ldr <= 128 ? (a.zeta_int == 8 ? sym_jvp_kernel<8, 128, ROWS> : sym_jvp_kernel<0, 128, ROWS>)
                 : (a.zeta_int == 8 ? sym_jvp_kernel<8, 256, ROWS> : sym_jvp_kernel<0, 256, ROWS>);
  k<<<tm_div_up(N, SYM_WAVES), SYM_WAVES * 64, 0, s>>>(N, pos, box, mol, elem, nbr, ncnt, rseg,
                                                       ang, acnt, aseg, ldr, lda, a, du, V, ldg,
                                                       ybar, places);
  TM_LAUNCH_CHECK();
  return TM_OK;
}

extern "C" {

// Host-side parameter arrays (rs_r[nr], rs_a[8], thetas[8]) are read on the
// host and passed to the kernels by value.
int tm_sym_forward(int N, const double* pos, const double* box, const int* mol, const int* elem,
                   const int* nbr, const int* ncnt, const int* rseg, const int* ang,
                   const int* acnt, const int* aseg, int ldr, int lda, int nele, int nr,
                   float eta, float zeta, float rr, float ra, const float* rs_r,
                   const float* rs_a, const float* thetas, float* G, int ldg, int* rev,
                   int* flags, void* stream) {
  return sym_forward<false>(N, pos, box, mol, elem, nbr, ncnt, rseg, ang, acnt, aseg, ldr, lda, nele, nr, eta,
                     zeta, rr, ra, rs_r, rs_a, thetas, G, ldg, rev, flags, nullptr, stream);
}

int tm_sym_forward_rows(int N, const double* pos, const double* box, const int* mol, const int* elem,
                   const int* nbr, const int* ncnt, const int* rseg, const int* ang,
                   const int* acnt, const int* aseg, int ldr, int lda, int nele, int nr,
                   float eta, float zeta, float rr, float ra, const float* rs_r,
                   const float* rs_a, const float* thetas, float* G, int ldg, int* rev,
                   int* flags, const long* places, void* stream) {
  TM_REQUIRE(places != nullptr, "tm_sym_forward_rows: places missing");
  return sym_forward<true>(N, pos, box, mol, elem, nbr, ncnt, rseg, ang, acnt, aseg, ldr, lda, nele, nr, eta,
                     zeta, rr, ra, rs_r, rs_a, thetas, G, ldg, rev, flags, places, stream);
}

int tm_sym_adjoint(int N, const double* pos, const double* box, const int* mol, const int* elem,
                   const int* nbr, const int* ncnt, const int* rseg, const int* ang,
                   const int* acnt, const int* aseg, int ldr, int lda, int nele, int nr,
                   float eta, float zeta, float rr, float ra, const float* rs_r,
                   const float* rs_a, const float* thetas, const float* gE, const float* gQ,
                   const float* u, const double* phi, const double* phimean, int ldg,
                   float* wslot, void* stream) {
  SymArgs a;
  int st = fill_args(a, nele, nr, eta, zeta, rr, ra, rs_r, rs_a, thetas);
  if (st) return st;
  TM_REQUIRE(ldg >= a.D, "tm_sym_adjoint: ldg %d < D %d", ldg, a.D);
  TM_REQUIRE(gQ == nullptr || u != nullptr || (phi != nullptr && phimean != nullptr),
             "tm_sym_adjoint: gQ needs u or phi and phimean");
  TM_REQUIRE(ldr > 0 && ldr <= MAX_ROW && lda > 0 && lda <= ldr,
             "tm_sym_adjoint: strides %d/%d (need 0 < lda <= ldr <= %d)", ldr, lda, MAX_ROW);
  if (N == 0) return TM_OK;
  hipStream_t s = (hipStream_t)stream;
  auto k = ldr <= 128 ? (a.zeta_int == 8 ? sym_adj_kernel<8, 128> : sym_adj_kernel<0, 128>)
                      : (a.zeta_int == 8 ? sym_adj_kernel<8, 256> : sym_adj_kernel<0, 256>);
  auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  const int off = nele * nr;
  const int vec4 = off % 4 == 0 && a.D % 4 == 0 && ldg % 4 == 0 && aligned(gE) && aligned(gQ);
  const int D4 = (a.D + ((off + 3) & ~3) - off + 3) / 4;
  k<<<tm_div_up(N, SYM_WAVES), SYM_WAVES * 64, sizeof(float4) * SYM_WAVES * D4, s>>>(
      N, pos, box, mol, elem, nbr, ncnt, ang, acnt, ldr, lda, a, gE, gQ, u, phi, phimean, ldg,
      vec4, (float4*)wslot);
  TM_LAUNCH_CHECK();
  return TM_OK;
}

int tm_sym_jvp(int N, const double* pos, const double* box, const int* mol, const int* elem,
               const int* nbr, const int* ncnt, const int* rseg, const int* ang, const int* acnt,
               const int* aseg, int ldr, int lda, int nele, int nr, float eta, float zeta,
               float rr, float ra, const float* rs_r, const float* rs_a, const float* thetas,
               const double* du, float* V, int ldg, void* stream) {
  return sym_jvp<false>(N, pos, box, mol, elem, nbr, ncnt, rseg, ang, acnt, aseg, ldr, lda, nele, nr, eta,
                     zeta, rr, ra, rs_r, rs_a, thetas, du, V, ldg, nullptr, nullptr, stream);
}

int tm_sym_jvp_rows(int N, const double* pos, const double* box, const int* mol, const int* elem,
               const int* nbr, const int* ncnt, const int* rseg, const int* ang, const int* acnt,
               const int* aseg, int ldr, int lda, int nele, int nr, float eta, float zeta,
               float rr, float ra, const float* rs_r, const float* rs_a, const float* thetas,
               const double* du, const float* ybar, const long* places,
                    void* stream) {
  TM_REQUIRE(ybar != nullptr && places != nullptr, "tm_sym_jvp_rows: ybar or places missing");
  return sym_jvp<true>(N, pos, box, mol, elem, nbr, ncnt, rseg, ang, acnt, aseg, ldr, lda, nele, nr, eta,
                     zeta, rr, ra, rs_r, rs_a, thetas, du, nullptr, 0, ybar, places, stream);
}

int tm_force_gather(int N, int ldr, const int* ncnt, const int* rev, const float* wslot,
                    const double* extra, double scale, double* grad, double* force,
                    void* stream) {
  if (N == 0) return TM_OK;
  hipStream_t s = (hipStream_t)stream;
  force_gather_kernel<false><<<tm_div_up(16l * N, 256), 256, 0, s>>>(
      N, ldr, ncnt, rev, (const float4*)wslot, extra, scale, grad, force, VVState{});
  TM_LAUNCH_CHECK();
  return TM_OK;
}

int tm_force_gather_sums(int N, int ldr, const int* ncnt, const int* rev, const float* wslot,
                         const double* extra, double scale, double* grad, double* force, int B,
                         const int* mol_start, int nsrc, const void* const* in, const int* f64,
                         const int* cols, const int* ld, double* const* out, double* scratch,
                         void* stream) {
  SumCols S;
  const int st = sum_cols("tm_force_gather_sums", B, N, nsrc, in, f64, cols, ld, out, &S);
  if (st) return st;
  const bool one = B == 1 && N > 2048;
  TM_REQUIRE(!one || scratch != nullptr, "tm_force_gather_sums: one large system needs scratch");
  const int nsum = one ? tm_div_up(N, 1024) : B;
  const int blocks = nsum + tm_div_up(16l * N, 256);
  if (blocks == 0) return TM_OK;
  auto k = one ? force_gather_sums_kernel<true> : force_gather_sums_kernel<false>;
  k<<<blocks, 256, 0, (hipStream_t)stream>>>(nsum, mol_start, S, scratch, N, ldr, ncnt, rev,
                                             (const float4*)wslot, extra, scale, grad, force);
  TM_LAUNCH_CHECK();
  return TM_OK;
}

// out[m] = (bp[m] + ext[2 m]) + ext[2 m + 1]
int tm_total_energy(int B, const double* bp, const double* ext, double* out, void* stream) {
  if (B == 0) return TM_OK;
  total_energy_kernel<<<tm_div_up(B, 256), 256, 0, (hipStream_t)stream>>>(B, bp, ext, out);
  TM_LAUNCH_CHECK();
  return TM_OK;
}

int tm_force_gather_vv(int N, int ldr, const int* ncnt, const int* rev, const float* wslot,
                       const double* extra, double scale, double* grad, double* force, double dt,
                       const double* m, double* v, double* a, double* ke, double* x,
                       void* stream) {
  TM_REQUIRE(m != nullptr && v != nullptr && a != nullptr && x != nullptr,
             "tm_force_gather_vv: m, v, a and x are required");
  if (N == 0) return TM_OK;
  hipStream_t s = (hipStream_t)stream;
  force_gather_kernel<true><<<tm_div_up(16l * N, 256), 256, 0, s>>>(
      N, ldr, ncnt, rev, (const float4*)wslot, extra, scale, grad, force,
      VVState{dt, m, v, a, ke, x});
  TM_LAUNCH_CHECK();
  return TM_OK;
}

}  // extern "C"
