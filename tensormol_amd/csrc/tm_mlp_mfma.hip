// Fused per-element MLPs on MFMA (gfx950): forward and input gradient of
// both the energy and the charge network in one launch.
//
// Math restates energy_inference / dipole_inference
// (TensorMol/TFNetworks/TFMolInstanceDirect.py:5164-5212, 5219-5272), three
// hidden layers h_k = act(h_{k-1} W_k + b_k), act(z) = log(1 + e^{a z})/a
// (Util.py:200-201), output y = h_3 w_o + b_o; and the adjoint that
// tf.gradients builds (:5761) for dy/dG:
//   dZ3 = w_o * act'(Z3), dH_{k-1} = dZ_k W_k^T, dZ_{k-1} = dH_{k-1} * act'(Z_{k-1}),
//   dG = dZ1 W_1^T, act'(z) = sigmoid(a z).
//
// Work decomposition: one 512-thread workgroup per tile of MT atoms of one
// (net, element) segment (atoms are element-sorted so a tile never straddles
// an element).  Every GEMM is computed transposed, out^T = W^T in^T, with
// v_mfma_f32_16x16x32_{bf16,f16}: A = weights (pre-packed in fragment order,
// one 1 KiB coalesced load per fragment), B = activations from LDS
// ([atom][feature], 16-byte reads), C = 16 features x 16 atoms.  Wave w owns
// output features [64w, 64w+64) of every hidden layer, so the activation
// derivative of its features stays in its registers from the forward to the
// backward pass; only activations / upstream gradients cross waves, through
// two LDS ping-pong buffers.  The descriptor block streams through LDS in
// 128-feature chunks, converted from FP32 on the fly, each loaded while the
// one before it is multiplied.
//
// What bounds it: a 64-row tile runs its matrix instructions in 60 % (split
// mode, D 256) and 44 % (FP16, D 768) of its cycles, the rest being the layer
// epilogues that the second wave of a SIMD cannot cover, the descriptor reads
// and the dG writes; at that load the card lowers its clock.  A 32-row tile is
// bound by the weight fragments, which one CU reads at 40-55 bytes a cycle.
// Weight fragments as a register ring, streamed descriptors and priorities
// took the 12,288-atom box from 149 to 130 us (bf16x3f), the 24,000-atom
// sphere from 244 to 220 us (FP16), a 2,139-atom batch from 78 to 63 us and
// 192 atoms from 51 to 41 us (bf16x3f).
//
// Modes: 0 bf16, 1 fp16 (operands rounded once, FP32 accumulation),
// 2 bf16 hi/lo split: x = hi + lo for weights and activations and
// acc += Whi*xhi + Wlo*xhi + Whi*xlo (near-FP32 products),
// 3 bf16 with split forward weights: the three forward GEMMs take
// acc += Whi*x + Wlo*x (weights carried to 16 significant bits, activations
// and descriptors rounded once to BF16), the input-gradient GEMMs plain BF16;
// 4 the same with FP16 operands (weights to 22 bits, activations to 11);
// 5 bf16 with the forward GEMMs split in weights and activations (three
// MFMAs, as mode 2) and plain BF16 input-gradient GEMMs.
// Rounding the weights shifts every atom's energy the same way, so that error
// adds up over a system; rounding activations gives an unbiased error that is
// decorrelated across atoms, so it averages out over large systems but not
// over a small molecule: modes 3 and 4 remove the first, mode 5 both.
#include <type_traits>

#include "tm_common.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned uint4v __attribute__((ext_vector_type(4)));

// f(0), f(1), ..., f(N - 1) with the index a compile-time constant
template <int N, int I = 0, class F>
__device__ __forceinline__ void unroll(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>());
    unroll<N, I + 1>(f);
  }
}

constexpr int NW = 8;       // waves per workgroup
constexpr int FT = 4;       // 16-feature tiles per wave (64 features)
constexpr int KC = 64;      // the descriptor length must be a multiple of KC
constexpr int HMAX = 512;   // widest hidden layer

struct MlpArgs {
  int N, D, H, ldg;
  int ntiles;
  const int* tiles;        // [ntiles][2] = (segment, first row in segment)
  const int* seg;          // [nseg][4] = (net, blob index, first row in perm, rows)
  const float* G;
  const int* perm;
  const unsigned short* const* blobs;   // device array of per-(net,element) weight blobs
  float alpha;
  float* y;                // [2][N]
  float* dG;               // [2][N][ldg]
  int* flags;
};

// ---- packed blob layout (elements of 2 bytes), identical on the host ----
__host__ __device__ inline long frag_elems(int rows16, int cols32) {
  return (long)rows16 * cols32 * 512;
}
struct BlobLayout {
  long f1, f2, f3, b3, b2, b1, fend;   // fragment planes (offsets in 2-byte elements)
  long bias_bytes;                     // byte offset of the float section
};
// planes of the forward (f*) and backward (b*) fragment arrays: 1 (one rounding)
// or 2 (hi plane, then lo plane)
__host__ __device__ constexpr int fwd_planes(int mode) { return mode >= 2 ? 2 : 1; }
__host__ __device__ constexpr int bwd_planes(int mode) { return mode == 2 ? 2 : 1; }
// activation (B operand) lo planes in the forward / backward GEMMs
__host__ __device__ constexpr bool act_split_fwd(int mode) { return mode == 2 || mode == 5; }
__host__ __device__ constexpr bool act_split_bwd(int mode) { return mode == 2; }
__host__ __device__ inline BlobLayout blob_layout(int D, int H, int fp, int bp) {
  BlobLayout L;
  long o = 0;
  L.f1 = o; o += fp * frag_elems(H / 16, D / 32);
  L.f2 = o; o += fp * frag_elems(H / 16, H / 32);
  L.f3 = o; o += fp * frag_elems(H / 16, H / 32);
  L.b3 = o; o += bp * frag_elems(H / 16, H / 32);
  L.b2 = o; o += bp * frag_elems(H / 16, H / 32);
  L.b1 = o; o += bp * frag_elems(D / 16, H / 32);
  L.fend = o;
  L.bias_bytes = ((o * 2 + 255) / 256) * 256;
  return L;
}
// float section: b1[H], b2[H], b3[H], wo[H], bo

template <int MODE>
struct Ty;
template <>
struct Ty<0> {
  typedef bf16x8 vec;
  static __device__ __forceinline__ unsigned short cvt(float x) {
    return __builtin_bit_cast(unsigned short, (__bf16)x);
  }
  static __device__ __forceinline__ float back(unsigned short b) {
    return (float)__builtin_bit_cast(__bf16, b);
  }
  static __device__ __forceinline__ floatx4 mma(const uint4v& a, const uint4v& b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
template <>
struct Ty<1> {
  static __device__ __forceinline__ unsigned short cvt(float x) {
    return __builtin_bit_cast(unsigned short, (_Float16)x);
  }
  static __device__ __forceinline__ float back(unsigned short b) {
    return (float)__builtin_bit_cast(_Float16, b);
  }
  static __device__ __forceinline__ floatx4 mma(const uint4v& a, const uint4v& b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};
template <>
struct Ty<2> : Ty<0> {};
template <>
struct Ty<3> : Ty<0> {};
template <>
struct Ty<4> : Ty<1> {};
template <>
struct Ty<5> : Ty<0> {};

// act(z) = log(1 + e^{a z}) / a and act'(z) = sigmoid(a z), sharing e = e^{-|a z|}:
// act = (max(a z, 0) + log(1 + e)) / a, sigmoid = 1/(1+e) for a z >= 0, e/(1+e) below.
// The hardware exp2 / log2 are used directly: the exp2 argument is <= 0 (a
// result below the normal range is flushed to 0, harmless here) and the log2
// argument lies in [1, 2], so the library's range fix-ups are not needed.
struct ActConst {
  float alpha, inv_alpha, k_exp, k_log;   // k_exp = -alpha log2(e), k_log = ln(2) / alpha
};
__device__ __forceinline__ ActConst act_const(float alpha) {
  ActConst c;
  c.alpha = alpha;
  c.inv_alpha = 1.0f / alpha;
  c.k_exp = -alpha * 1.4426950408889634f;
  c.k_log = 0.6931471805599453f / alpha;
  return c;
}
__device__ __forceinline__ void act_pair(float z, const ActConst& c, float& act, float& dact) {
  const float e = __builtin_amdgcn_exp2f(fabsf(z) * c.k_exp);
  const float r = __builtin_amdgcn_rcpf(1.0f + e);
  act = fmaxf(z, 0.f) + __builtin_amdgcn_logf(1.0f + e) * c.k_log;
  dact = z >= 0.f ? r : e * r;
}

// x as rounded to FP32: a product fused with its conversion to FP16 in one tile
// size and not in the other would make an atom's result depend on the tile it
// sits in
__device__ __forceinline__ float fp32(float x) {
  asm("" : "+v"(x));
  return x;
}

// Activation derivatives of a wave's features, kept from the forward to the
// backward pass: packed FP16 pairs in the BF16 / FP16 modes (the backward
// operands are rounded to 8 / 11 bits anyway), FP32 in the split mode.
typedef __fp16 half2v __attribute__((ext_vector_type(2)));
template <int MODE, int NFT, int AT>
struct DerivRegs {
  half2v h[NFT][AT][2];   // two derivatives per register
  __device__ __forceinline__ void set4(int ft, int at, const float d[4]) {
    h[ft][at][0] = __builtin_amdgcn_cvt_pkrtz(d[0], d[1]);
    h[ft][at][1] = __builtin_amdgcn_cvt_pkrtz(d[2], d[3]);
  }
  __device__ __forceinline__ float get(int ft, int at, int i) const {
    return (float)h[ft][at][i >> 1][i & 1];
  }
};
template <int NFT, int AT>
struct DerivRegs<2, NFT, AT> {
  float h[NFT][AT][4];
  __device__ __forceinline__ void set4(int ft, int at, const float d[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) h[ft][at][i] = d[i];
  }
  __device__ __forceinline__ float get(int ft, int at, int i) const { return h[ft][at][i]; }
};

// Activation buffers.  Two ping-pong buffers X, Y (the descriptor tile staged
// across both), or, where two would not fit (split activations in 64-row
// tiles), one buffer used in place by every layer: the descriptor tile
// streams through its first columns, and each layer's GEMM reads the whole
// buffer before (a barrier) its epilogue overwrites it with the layer's output.
template <int MODE, int MT>
constexpr bool in_place() { return act_split_fwd(MODE) && MT > 32; }

template <int MODE, int MT, bool INPLACE = in_place<MODE, MT>()>
struct Smem {
  static constexpr int PL = act_split_fwd(MODE) ? 2 : 1;
  static constexpr int SH = HMAX + 8;                // activation row stride (elements)
  union {
    struct {
      unsigned short X[PL][MT][SH];
      unsigned short Y[PL][MT][SH];
    };
    // layer 1: the whole descriptor tile, row stride D + 8 <= 2 SH
    unsigned short Gt[2 * PL * MT * SH];
  };
  float bias[4][HMAX];   // b1, b2, b3, w_o
  float epart[NW][MT];
  int atoms[MT];
};
template <int MODE, int MT>
struct Smem<MODE, MT, true> {
  static constexpr int PL = act_split_fwd(MODE) ? 2 : 1;
  static constexpr int SH = HMAX + 8;
  unsigned short X[PL][MT][SH];
  float bias[4][HMAX];
  float epart[NW][MT];
  int atoms[MT];
};

// ---- the GEMMs ---------------------------------------------------------------
// A weight stream: the fragments of one wave's row tiles of one GEMM, taken in
// substeps.  A k-step (32 k) is one substep, or two with split weights: its hi
// fragments, then its lo fragments.  Every field is wave-uniform, a byte
// offset into the blob, so a fragment load is one buffer instruction with a
// scalar offset.
struct WStream {
  int row[FT];   // offset of each row tile's first fragment, hi plane
  int plane;     // bytes from the hi to the lo plane
  int nsub;      // substeps
};

// Row tiles rt0 .. (the last one there is, rtmax, stands in for those past it)
// of the fragment array at element off, kstride k-steps each.
__device__ __forceinline__ WStream wstream(long off, long plane_elems, int kstride, int rt0,
                                           int rtmax, int wp) {
  WStream s;
#pragma unroll
  for (int ft = 0; ft < FT; ++ft) s.row[ft] = (int)off * 2 + min(rt0 + ft, rtmax) * kstride * 1024;
  s.plane = (int)plane_elems * 2;
  s.nsub = kstride * wp;
  return s;
}

// Substep sub of stream s (WP planes per k-step), or, past its end, the
// substeps of the stream t that follows it (WPN planes).
template <int WP, int WPN>
__device__ __forceinline__ void load_sub(uint4v (&set)[FT], __amdgpu_buffer_rsrc_t blob,
                                         const WStream& s, const WStream& t, int sub, int lane) {
  const bool over = sub >= s.nsub;
  const int v = over ? sub - s.nsub : sub;
  const int off_s = (WP == 2 ? v >> 1 : v) * 1024 + (WP == 2 && (v & 1) ? s.plane : 0);
  const int off_t = (WPN == 2 ? v >> 1 : v) * 1024 + (WPN == 2 && (v & 1) ? t.plane : 0);
  const int off = over ? off_t : off_s;
#pragma unroll
  for (int ft = 0; ft < FT; ++ft)
    set[ft] = __builtin_amdgcn_raw_buffer_load_b128(blob, lane * 16,
                                                    (over ? t.row[ft] : s.row[ft]) + off, 0);
}

// Substeps [s0, s1) of a GEMM: acc[ft][at] += W x B, B read from LDS rows
// [atom][k] (two planes with XP 2).  Per k-step and accumulator the products
// are added in the order Whi xhi, Wlo xhi, Whi xlo.
//
// What bounds it is the latency of the weight fragments (every fragment is
// read once per workgroup, from L2 or beyond it), so NS sets of them form a
// ring: the sets of a k-step are refilled for the k-step NS / WP later as soon
// as its MFMAs are issued, and past the end of this GEMM with the first
// fragments of the next one, so that the fragments a layer starts with are on
// their way during the epilogue before it.  On entry the ring holds substeps
// s0 .. s0 + NS - 1, on exit those that follow.  The B fragments of the next
// k-step are read behind the MFMAs of the current one.  s0, s1 and the
// stream's length are multiples of NS.
template <int MODE, int MT, int NFT, int WP, int XP, int NS, int WPN>
__device__ __forceinline__ void gemm_ring(floatx4 (&acc)[NFT][MT / 16], uint4v (&ring)[NS][FT],
                                          __amdgpu_buffer_rsrc_t blob, const WStream& cur,
                                          const WStream& nxt, int s0, int s1,
                                          const unsigned short* bbase, int bplane, int lane,
                                          int stride) {
  constexpr int AT = MT / 16;
  static_assert(NS % WP == 0, "a ring holds whole k-steps");
  const unsigned short* bp = bbase + (lane & 15) * stride + (lane >> 4) * 8;
  uint4v bh[AT], bl[XP == 2 ? AT : 1];
  const int klast = (s1 - s0) / WP - 1;   // last k-step in the buffer
  auto ldb = [&](int at, int k) {
    bh[at] = *reinterpret_cast<const uint4v*>(bp + at * 16 * stride + k * 32);
    if constexpr (XP == 2)
      bl[at] = *reinterpret_cast<const uint4v*>(bp + bplane + at * 16 * stride + k * 32);
  };
#pragma unroll
  for (int at = 0; at < AT; ++at) ldb(at, 0);
  int sub = s0;
  do {   // s0 < s1
    unroll<NS / WP>([&](auto kc) {
      constexpr int u = decltype(kc)::value * WP;   // the k-step's first set
      const int kn = min((sub - s0 + u) / WP + 1, klast);
      if constexpr (WP == 2) {
#pragma unroll
        for (int at = 0; at < AT; ++at)
#pragma unroll
          for (int ft = 0; ft < NFT; ++ft)
            acc[ft][at] = Ty<MODE>::mma(ring[u][ft], bh[at], acc[ft][at]);
      }
#pragma unroll
      for (int at = 0; at < AT; ++at) {
#pragma unroll
        for (int ft = 0; ft < NFT; ++ft) {
          acc[ft][at] = Ty<MODE>::mma(ring[u + WP - 1][ft], bh[at], acc[ft][at]);
          if constexpr (XP == 2) acc[ft][at] = Ty<MODE>::mma(ring[u][ft], bl[at], acc[ft][at]);
        }
        ldb(at, kn);
      }
#pragma unroll
      for (int p = 0; p < WP; ++p)
        load_sub<WP, WPN>(ring[u + p], blob, cur, nxt, sub + u + p + NS, lane);
      __builtin_amdgcn_sched_barrier(0);
    });
    sub += NS;
  } while (sub < s1);
}

template <int MODE, int MT>
constexpr bool shares_cu() { return MT == 32 && !act_split_fwd(MODE); }
// Weight fragment sets in flight: four (64 of the 256 registers a lane has; the
// split mode's 32-row tiles have room for eight and gain nothing by them: 62.9
// against 65.1 us on 2,139 C/H/N/O atoms), two in the 32-row tiles that share a
// CU (128 registers).  Four need widths that make every stream a multiple of
// the ring, which 128-wide ones do; any other width takes the kernel with two.
template <int MODE, int MT>
constexpr int ring_sets() { return shares_cu<MODE, MT>() ? 2 : 4; }
inline bool ring_fits(int D, int H) { return D % 128 == 0 && H % 128 == 0; }

// One layer's values of a wave, rounded for the activation buffer: hi plane,
// and the lo plane where the forward operands are split.
template <int MODE, int MT, bool LO>
struct Packed {
  uint2 h[FT][MT / 16], l[LO ? FT : 1][LO ? MT / 16 : 1];
  __device__ __forceinline__ void set(int ft, int at, const float v[4]) {
    unsigned short x[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = Ty<MODE>::cvt(v[i]);
    h[ft][at] = make_uint2((unsigned)x[0] | ((unsigned)x[1] << 16),
                           (unsigned)x[2] | ((unsigned)x[3] << 16));
    // packed here, not where it is stored: the FP32 values would stay live
    asm volatile("" : "+v"(h[ft][at].x), "+v"(h[ft][at].y));
    if constexpr (LO) {
      unsigned short y[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) y[i] = Ty<MODE>::cvt(v[i] - Ty<MODE>::back(x[i]));
      l[ft][at] = make_uint2((unsigned)y[0] | ((unsigned)y[1] << 16),
                             (unsigned)y[2] | ((unsigned)y[3] << 16));
      asm volatile("" : "+v"(l[ft][at].x), "+v"(l[ft][at].y));
    }
  }
  // features 64 w + 16 ft + fq .. + 3 of atom 16 at + ca
  __device__ __forceinline__ void store(unsigned short (*buf)[MT][HMAX + 8], int w, int fq,
                                        int ca) const {
#pragma unroll
    for (int ft = 0; ft < FT; ++ft)
#pragma unroll
      for (int at = 0; at < MT / 16; ++at) {
        const int f = 64 * w + 16 * ft + fq;
        *reinterpret_cast<uint2*>(&buf[0][at * 16 + ca][f]) = h[ft][at];
        if constexpr (LO) *reinterpret_cast<uint2*>(&buf[1][at * 16 + ca][f]) = l[ft][at];
      }
  }
};

// A reader: streams one weight blob in the order the layers take it and drops
// it, so that it lies in the XCD's L2 when the tiles beside it ask.  A tile
// alone streams at what 128 KB in flight and the latency behind the L2 allow
// (40 bytes a cycle); a reader on a CU of its own has no layers to wait for and
// gets ahead.  One launch, bf16x3f, without / with readers: 192 water atoms
// 43.3 / 40.7 us, 1,200 44.9 / 41.9, two chains (D 768) 66.0 / 57.4, 2,139 chain
// atoms 64.8 / 62.0, 20 chains in FP16 48.5 / 44.9.  Two readers that share a
// blob are slower again (43 to 66 us).
__device__ __forceinline__ void read_ahead(const void* blob, long bytes) {
  constexpr int U = 8;
  const uint4v* p = static_cast<const uint4v*>(blob);
  const int n = (int)(bytes / 16);   // whole fragments
  for (int t = threadIdx.x; t < n; t += U * NW * 64) {
    uint4v v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = p[min(t + u * NW * 64, n - 1)];
#pragma unroll
    for (int u = 0; u < U; ++u) asm volatile("" ::"v"(v[u]));
  }
}

// 64-row tiles: one workgroup per CU (LDS); 32-row tiles in the BF16 / FP16
// modes fit two workgroups per CU when the waves stay within 128 VGPRs.
template <int MODE, int MT, int NS>
__global__ void __launch_bounds__(NW * 64)
__attribute__((amdgpu_waves_per_eu(shares_cu<MODE, MT>() ? 4 : 2)))
mlp_mfma_kernel(MlpArgs a) {
  constexpr int AT = MT / 16;
  constexpr bool LOF = act_split_fwd(MODE);   // forward operands carry lo planes
  constexpr bool LOB = act_split_bwd(MODE);   // backward operands carry lo planes
  constexpr bool INPLACE = in_place<MODE, MT>();
  constexpr int SH = HMAX + 8;
  constexpr int WPF = fwd_planes(MODE), WPB = bwd_planes(MODE);
  constexpr int XPF = LOF ? 2 : 1, XPB = LOB ? 2 : 1;
  typedef Smem<MODE, MT> S;
  __shared__ S sm;
  // output buffer of layers 2, bwd 3 (read by layer 3, bwd 2): Y, or X in place
  unsigned short (*const Yb)[MT][SH] = [&]() {
    if constexpr (INPLACE) return sm.X; else return sm.Y;
  }();
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int tile = blockIdx.x;
  const int s = a.tiles[2 * tile], row0 = a.tiles[2 * tile + 1];
  if (s < 0) {   // no tile (whole workgroup): padding of the XCD-ordered table, or a reader
    if (s < -1)
      read_ahead(a.blobs[a.seg[4 * (-2 - s) + 1]],
                 blob_layout(a.D, a.H, fwd_planes(MODE), bwd_planes(MODE)).bias_bytes);
    return;
  }
  const int net = a.seg[4 * s], blob = a.seg[4 * s + 1], first = a.seg[4 * s + 2];
  const int rows = a.seg[4 * s + 3];
  const int D = a.D, H = a.H;
  const BlobLayout BL = blob_layout(D, H, fwd_planes(MODE), bwd_planes(MODE));
  const unsigned short* wb = a.blobs[blob];
  const float* fsec = reinterpret_cast<const float*>(reinterpret_cast<const char*>(wb) + BL.bias_bytes);
  // The two waves of a SIMD run the same layer between two barriers.  With
  // different priorities the first finishes its MFMAs early and does its
  // epilogue under the MFMAs of the second, instead of both at the same time
  // (45.4 -> 43.3 us on 192 atoms, 223 -> 220 us on the 24,000-atom sphere).
  if (w < NW / 2) __builtin_amdgcn_s_setprio(2);
  const bool wact = (w * 64) < H;   // this wave owns hidden features
  const int fq = (lane >> 4) * 4;   // first of the 4 features this lane holds in a C tile
  const int ca = lane & 15;         // atom column of this lane in a C tile
  // activation derivatives of layers 1 and 2 for this wave's features
  DerivRegs<MODE, FT, AT> s1, s2;
  const ActConst ac = act_const(a.alpha);
  const long phh = frag_elems(H / 16, H / 32), p1 = frag_elems(H / 16, D / 32);
  const int hk = H / 32, hmax = H / 16 - 1, ntile = D / 16;
  __amdgpu_buffer_rsrc_t blob_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<unsigned short*>(wb), 0, (int)BL.bias_bytes, 0x00020000);
  const WStream W1 = wstream(BL.f1, p1, D / 32, FT * w, hmax, WPF);
  const WStream W2 = wstream(BL.f2, phh, hk, FT * w, hmax, WPF);
  const WStream W3 = wstream(BL.f3, phh, hk, FT * w, hmax, WPF);
  const WStream V3 = wstream(BL.b3, phh, hk, FT * w, hmax, WPB);
  const WStream V2 = wstream(BL.b2, phh, hk, FT * w, hmax, WPB);
  // backward 1: dG tiles [nf1 w, nf1 w + nf1), then + nf1 NW, ...; three tiles
  // per pass where that divides the tiles of a wave, else two
  const int nf1 = (ntile + NW - 1) / NW % 3 == 0 ? 3 : 2;
  auto w1stream = [&](int t0) {
    return wstream(BL.b1, frag_elems(ntile, hk), hk, t0, ntile - 1, WPB);
  };
  uint4v ring[NS][FT];
  if (wact) {
#pragma unroll
    for (int u = 0; u < NS; ++u) load_sub<WPF, WPF>(ring[u], blob_rsrc, W1, W2, u, lane);
  }
  // the four values of row `layer` of sm.bias this lane's features take
  auto bias4 = [&](int layer, int ft) {
    return *reinterpret_cast<const floatx4*>(&sm.bias[layer][64 * w + 16 * ft + fq]);
  };
  auto clear = [&](floatx4 (&acc)[FT][AT]) {
#pragma unroll
    for (int ft = 0; ft < FT; ++ft)
#pragma unroll
      for (int at = 0; at < AT; ++at) acc[ft][at] = floatx4{0.f, 0.f, 0.f, 0.f};
  };
  const int bpl = MT * SH;   // element offset of the lo plane

  // ------------------------------------------------------------ layer 1
  // The descriptor tile G[atom][0 .. D) streams through LDS in chunks of CW
  // columns: a chunk is loaded while the one before it is multiplied.  In
  // place, the chunks take the buffer's columns in turn (chunk c + HMAX / CW
  // overwrites chunk c, which every wave finished two barriers earlier);
  // otherwise the whole tile is laid out across both buffers, row stride D + 8.
  floatx4 acc1[FT][AT];
  clear(acc1);
  {
    constexpr int CW = 128;
    constexpr int GL = MT * CW / 4 / (NW * 64);   // float4 loads per thread and chunk
    const int SG = INPLACE ? SH : D + 8;
    const int gpl = MT * SG;
    unsigned short* Gt = reinterpret_cast<unsigned short*>(&sm);
    int atoms[GL];
#pragma unroll
    for (int i = 0; i < GL; ++i) {
      const int r = row0 + (tid >> 5) + 16 * i;
      atoms[i] = r < rows ? a.perm[first + r] : -1;
      if ((tid & 31) == 0) sm.atoms[(tid >> 5) + 16 * i] = atoms[i];
    }
    for (int t = tid; t < 4 * H; t += NW * 64) sm.bias[t / H][t % H] = fsec[t];
    const int c4 = (tid & 31) * 4;
    float4 g[GL];
    auto fetch = [&](int c0) {
#pragma unroll
      for (int i = 0; i < GL; ++i)
        g[i] = (atoms[i] >= 0 && c0 + c4 < D)
                   ? *reinterpret_cast<const float4*>(a.G + (long)atoms[i] * a.ldg + c0 + c4)
                   : make_float4(0.f, 0.f, 0.f, 0.f);
    };
    fetch(0);
    for (int c0 = 0; c0 < D; c0 += CW) {
      const int lc = INPLACE ? c0 & (HMAX - 1) : c0;
      if (c0 + c4 < D) {
#pragma unroll
        for (int i = 0; i < GL; ++i) {
          const float v[4] = {g[i].x, g[i].y, g[i].z, g[i].w};
          unsigned short* dst = Gt + (long)((tid >> 5) + 16 * i) * SG + lc + c4;
          unsigned short h[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) h[q] = Ty<MODE>::cvt(v[q]);
          *reinterpret_cast<uint2*>(dst) = make_uint2((unsigned)h[0] | ((unsigned)h[1] << 16),
                                                      (unsigned)h[2] | ((unsigned)h[3] << 16));
          if constexpr (LOF) {
            unsigned short l[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) l[q] = Ty<MODE>::cvt(v[q] - Ty<MODE>::back(h[q]));
            *reinterpret_cast<uint2*>(dst + gpl) =
                make_uint2((unsigned)l[0] | ((unsigned)l[1] << 16),
                           (unsigned)l[2] | ((unsigned)l[3] << 16));
          }
        }
      }
      if (c0 + CW < D) fetch(c0 + CW);
      __syncthreads();
      if (wact) {
        gemm_ring<MODE, MT, FT, WPF, XPF, NS, WPF>(
            acc1, ring, blob_rsrc, W1, W2, c0 / 32 * WPF, min(c0 + CW, D) / 32 * WPF, Gt + lc, gpl, lane, SG);
      }
    }
  }
  // act(z) of a hidden layer, and its derivative for the backward pass
  auto epilogue = [&](int layer, const floatx4 (&acc)[FT][AT], auto& P, auto& ds) {
#pragma unroll
    for (int ft = 0; ft < FT; ++ft) {
      const floatx4 b = bias4(layer, ft);
#pragma unroll
      for (int at = 0; at < AT; ++at) {
        float v[4], d[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) act_pair(acc[ft][at][i] + b[i], ac, v[i], d[i]);
        ds.set4(ft, at, d);
        P.set(ft, at, v);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  // dZ = dH * act'
  auto scale = [&](const floatx4 (&acc)[FT][AT], auto& P, const auto& ds) {
#pragma unroll
    for (int ft = 0; ft < FT; ++ft)
#pragma unroll
      for (int at = 0; at < AT; ++at) {
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = fp32(acc[ft][at][i] * ds.get(ft, at, i));
        P.set(ft, at, v);
        __builtin_amdgcn_sched_barrier(0);
      }
  };
  {
    Packed<MODE, MT, LOF> P;
    if (wact) epilogue(0, acc1, P, s1);
    __syncthreads();   // every wave has read the tile before it is overwritten
    if (wact) P.store(sm.X, w, fq, ca);
  }
  __syncthreads();
  // ------------------------------------------------------------ layer 2
  {
    Packed<MODE, MT, LOF> P;
    if (wact) {
      floatx4 acc[FT][AT];
      clear(acc);
      gemm_ring<MODE, MT, FT, WPF, XPF, NS, WPF>(acc, ring, blob_rsrc, W2, W3, 0, W2.nsub,
                                                 &sm.X[0][0][0], bpl, lane, SH);
      epilogue(1, acc, P, s2);
    }
    if constexpr (INPLACE) __syncthreads();
    if (wact) P.store(Yb, w, fq, ca);
  }
  __syncthreads();
  // ------------------------------------------------------------ layer 3 + head
  {
    Packed<MODE, MT, LOB> P;
    if (wact) {
      floatx4 acc[FT][AT];
      clear(acc);
      gemm_ring<MODE, MT, FT, WPF, XPF, NS, WPB>(acc, ring, blob_rsrc, W3, V3, 0, W3.nsub,
                                                 &Yb[0][0][0], bpl, lane, SH);
      float ep[AT];
#pragma unroll
      for (int at = 0; at < AT; ++at) ep[at] = 0.f;
#pragma unroll
      for (int ft = 0; ft < FT; ++ft) {
        const floatx4 b = bias4(2, ft), wv = bias4(3, ft);
#pragma unroll
        for (int at = 0; at < AT; ++at) {
          float v[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float act, d;
            act_pair(acc[ft][at][i] + b[i], ac, act, d);
            ep[at] += act * wv[i];
            v[i] = fp32(wv[i] * d);   // dZ3 with upstream 1
          }
          P.set(ft, at, v);
          asm volatile("" : "+v"(ep[at]));   // summed here, not sunk to its use
          __builtin_amdgcn_sched_barrier(0);
        }
      }
#pragma unroll
      for (int at = 0; at < AT; ++at) {
        float p = ep[at];
        p += __shfl_xor(p, 16, 64);
        p += __shfl_xor(p, 32, 64);
        if (lane < 16) sm.epart[w][at * 16 + lane] = p;
      }
    } else {
      for (int t = lane; t < MT; t += 64) sm.epart[w][t] = 0.f;
    }
    if constexpr (INPLACE) __syncthreads();
    if (wact) P.store(sm.X, w, fq, ca);
  }
  __syncthreads();
  if (tid < MT) {
    int atom = sm.atoms[tid];
    if (atom >= 0) {
      float yv = fsec[4 * H];
#pragma unroll
      for (int q = 0; q < NW; ++q) yv += sm.epart[q][tid];
      a.y[(long)net * a.N + atom] = yv;
    }
  }
  // ------------------------------------------------------------ backward 3: dZ3 -> dZ2
  {
    Packed<MODE, MT, LOB> P;
    if (wact) {
      floatx4 acc[FT][AT];
      clear(acc);
      gemm_ring<MODE, MT, FT, WPB, XPB, NS, WPB>(acc, ring, blob_rsrc, V3, V2, 0, V3.nsub,
                                                 &sm.X[0][0][0], bpl, lane, SH);
      scale(acc, P, s2);
    }
    if constexpr (INPLACE) __syncthreads();
    if (wact) P.store(Yb, w, fq, ca);
  }
  __syncthreads();
  // ------------------------------------------------------------ backward 2: dZ2 -> dZ1
  const WStream V1 = w1stream(nf1 * w);
  {
    Packed<MODE, MT, LOB> P;
    if (wact) {
      floatx4 acc[FT][AT];
      clear(acc);
      gemm_ring<MODE, MT, FT, WPB, XPB, NS, WPB>(acc, ring, blob_rsrc, V2, V1, 0, V2.nsub,
                                                 &Yb[0][0][0], bpl, lane, SH);
      scale(acc, P, s1);
    } else {
#pragma unroll
      for (int u = 0; u < NS; ++u) load_sub<WPB, WPB>(ring[u], blob_rsrc, V1, V1, u, lane);
    }
    if constexpr (INPLACE) __syncthreads();
    if (wact) P.store(sm.X, w, fq, ca);
  }
  __syncthreads();
  // ------------------------------------------------------------ backward 1: dZ1 -> dG
  float* dGn = a.dG + (long)net * a.N * a.ldg;
  auto backward1 = [&](auto nf) {
    constexpr int NF1 = decltype(nf)::value;
    for (int t0 = NF1 * w; t0 < ntile; t0 += NF1 * NW) {
      const WStream c = w1stream(t0), n = w1stream(min(t0 + NF1 * NW, ntile - 1));
      floatx4 acc2[NF1][AT];
#pragma unroll
      for (int u = 0; u < NF1; ++u)
#pragma unroll
        for (int at = 0; at < AT; ++at) acc2[u][at] = floatx4{0.f, 0.f, 0.f, 0.f};
      gemm_ring<MODE, MT, NF1, WPB, XPB, NS, WPB>(acc2, ring, blob_rsrc, c, n, 0, c.nsub,
                                                  &sm.X[0][0][0], bpl, lane, SH);
#pragma unroll
      for (int at = 0; at < AT; ++at) {
        const int atom = sm.atoms[at * 16 + ca];
        if (atom < 0) continue;
#pragma unroll
        for (int u = 0; u < NF1; ++u)
          if (t0 + u < ntile)
            *reinterpret_cast<float4*>(dGn + (long)atom * a.ldg + 16 * (t0 + u) + fq) =
                make_float4(acc2[u][at][0], acc2[u][at][1], acc2[u][at][2], acc2[u][at][3]);
      }
    }
  };
  if (nf1 == 3) backward1(std::integral_constant<int, 3>());
  else backward1(std::integral_constant<int, 2>());
}

template <int MODE, int MT>
void launch(const MlpArgs& a, size_t pad, hipStream_t s) {
  constexpr int NS = ring_sets<MODE, MT>();
  if (NS == 2 || ring_fits(a.D, a.H))
    mlp_mfma_kernel<MODE, MT, NS><<<a.ntiles, NW * 64, pad, s>>>(a);
  else
    mlp_mfma_kernel<MODE, MT, 2><<<a.ntiles, NW * 64, pad, s>>>(a);
}

}  // namespace

extern "C" {

// out[0] = blob bytes, out[1] = byte offset of the float section,
// out[2..7] = element offsets of f1, f2, f3, b3, b2, b1 fragment arrays,
// out[8] = planes of the forward arrays, out[9] = planes of the backward arrays
int tm_mlp_mfma_pack_info(int D, int H, int nh, int mode, long* out) {
  TM_REQUIRE(nh == 3, "tm_mlp_mfma: exactly 3 hidden layers supported (got %d)", nh);
  TM_REQUIRE(H % 64 == 0 && H <= HMAX && H >= 64, "tm_mlp_mfma: hidden width %d not a multiple of 64 in 64..512", H);
  TM_REQUIRE(D % KC == 0 && D > 0 && D + 8 <= 2 * (HMAX + 8),
             "tm_mlp_mfma: descriptor length %d not a multiple of %d in %d..%d", D, KC, KC,
             2 * HMAX + 8);
  TM_REQUIRE(mode >= 0 && mode <= 5, "tm_mlp_mfma: bad mode %d", mode);
  BlobLayout L = blob_layout(D, H, fwd_planes(mode), bwd_planes(mode));
  out[0] = L.bias_bytes + (4l * H + 4) * 4;
  out[1] = L.bias_bytes;
  out[2] = L.f1; out[3] = L.f2; out[4] = L.f3; out[5] = L.b3; out[6] = L.b2; out[7] = L.b1;
  out[8] = fwd_planes(mode);
  out[9] = bwd_planes(mode);
  return TM_OK;
}

// tiles: device int32 [ntiles][2] = (segment, first row), one workgroup per
// entry (segment -1: skipped, -2 - s: reads segment s's weights ahead); seg: device int32
// [nseg][4] = (net, blob index, first row in perm, rows); blobs: device array
// of per-(net, element) weight blob pointers (layout of tm_mlp_mfma_pack_info).
int tm_mlp_mfma(int N, int D, int H, int ntiles, const int* tiles, const int* seg, int ldg,
                const float* G, const int* perm, const void* blobs, float alpha, int mode,
                int tile_rows, float* y, float* dG, void* stream) {
  long info[10];
  int st = tm_mlp_mfma_pack_info(D, H, 3, mode, info);
  if (st) return st;
  TM_REQUIRE(ldg % 4 == 0 && ldg >= D, "tm_mlp_mfma: ldg %d", ldg);
  TM_REQUIRE(alpha > 0.f, "tm_mlp_mfma: activation alpha %g must be positive", (double)alpha);
  TM_REQUIRE(ntiles >= 0, "tm_mlp_mfma: bad tile count");
  TM_REQUIRE(tile_rows == 32 || (tile_rows == 64 && mode != 2),
             "tm_mlp_mfma: tile_rows %d (64 or 32; 32 in mode 2)", tile_rows);
  if (ntiles == 0) return TM_OK;
  MlpArgs a;
  a.N = N; a.D = D; a.H = H; a.ldg = ldg;
  a.ntiles = ntiles;
  a.tiles = tiles;
  a.seg = seg;
  a.G = G;
  a.perm = perm;
  a.blobs = (const unsigned short* const*)blobs;
  a.alpha = alpha;
  a.y = y;
  a.dG = dG;
  a.flags = nullptr;
  hipStream_t s = (hipStream_t)stream;
  // 32-row tiles fit several workgroups per CU.  With no more tiles than CUs
  // that would let the dispatcher stack two on one CU while others idle, so
  // the launch then asks for extra LDS: one workgroup per CU (over half of
  // the CU's 160 KiB).
  size_t pad = 0;
  if (tile_rows == 32 && mode != 2) {
    int dev = 0, ncu = 0;
    TM_HIP_CHECK(hipGetDevice(&dev));
    TM_HIP_CHECK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    const size_t lds = mode == 5 ? sizeof(Smem<5, 32>) : sizeof(Smem<0, 32>);
    if (ntiles <= ncu && lds < 81920) pad = 81920 - lds + 256;
  }
  const bool big = tile_rows == 64;
  switch (mode) {
    case 0: big ? launch<0, 64>(a, 0, s) : launch<0, 32>(a, pad, s); break;
    case 1: big ? launch<1, 64>(a, 0, s) : launch<1, 32>(a, pad, s); break;
    case 2: launch<2, 32>(a, 0, s); break;
    case 3: big ? launch<3, 64>(a, 0, s) : launch<3, 32>(a, pad, s); break;
    case 4: big ? launch<4, 64>(a, 0, s) : launch<4, 32>(a, pad, s); break;
    default: big ? launch<5, 64>(a, 0, s) : launch<5, 32>(a, pad, s); break;
  }
  TM_LAUNCH_CHECK();
  return TM_OK;
}

}  // extern "C"
