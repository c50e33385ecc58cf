// The chunkwise WY forward and its backward in fp32 on fp32 matrix cores
// (v_mfma_f32_16x16x4_f32: fp32 products, fp32 sums), in chunks of 64 tokens:
// fp32 q/k/v, and the bf16 head sizes that the bf16 MFMA kernels do not take,
// at head_k_dim up to 128 (chunk_generic.hip chooses, and has the rest).
//
// Same mathematics as the bf16 kernels (X = w⊙V − kg·S, V' = T·X; neither U
// nor W is formed):
//   intra      one workgroup per chunk-head: scores, T = (I + tril(Akk,−1))⁻¹
//              by blocked substitution, operand tiles to the workspace;
//   scan       serial over chunks, four waves per 16 value columns;
//   rev_scan   the dS recurrence, the same split;
//   chunk_bwd  one workgroup per chunk-head, a wave per 16 key channels.
//
// Bound by the fp32 matrix rate (140 TFLOP/s in a large product) where the
// sequences fill the device, and by the chain of a chunk's products where they
// do not. At B=4 S=1000 H=8 K=V=128 (23 GFLOP forward and backward, 165 us at
// that rate; 256 teams of scan waves, one per CU), against the any-shape
// kernels that ran these calls before, whose scores and inverse were scalar
// loops over HBM: intra 769 -> 23 us, scan 605 -> 62, states scan 404 -> 48
// beside the reverse scan 661 -> 97, chunk_bwd 1601 -> 101; forward and
// backward through autograd 4812 -> 316 us. B=1 S=512 H=4 K=V=64: forward
// 592 -> 30 us.
//
// Tiles. Every operand is kept as 16×16 blocks of 256 floats. Element (i, j)
// of a block sits at blk(i, j): float4s along j in the order of the MFMA
// lanes, so that lane (m, g) reads its four A (or Bᵀ) values j = 4g … 4g+3 of
// row m as one 16-byte word, 64 lanes linear over the block's 1 KB; with the
// row XORed by the float4's index, the transposed read (row 4g + r, column m)
// is free of bank conflicts as four 4-byte words. A contraction over 16 then
// takes four MFMAs whose step r pairs index 4g + r on both sides, and an
// accumulator tile, rows 4g + r, is the B operand of the next product as it
// stands.
#pragma once


#include "dn_common.hpp"
#include "mfma_util.hpp"

namespace dn {
namespace {

constexpr int kC = 64;            // tokens per chunk
constexpr int kBlk = 256;         // floats per 16×16 block
constexpr int kTri = 10 * kBlk;   // a lower-triangular 64×64 tile: its ten lower blocks
constexpr float kMaxExp = 48.0f;  // src/delta/decay.rs:49

__host__ __device__ constexpr int tri_blk(int i, int j) { return i * (i + 1) / 2 + j; }
__device__ inline int blk(int i, int j) { return (((j >> 2) * 16) + (i ^ (j >> 2))) * 4 + (j & 3); }

// Workspace of a chunk-head, in floats. The scan that writes no y needs the
// part before q only. `fold`: the gates do not reduce to one factor per token
// (per-channel erase or forget gates), so the tiles carry them.
struct Lay {
  int a;     // fold: e⊙e^G⊙k, else k      [4][KB] blocks
  int u;     // fold: e^{G_last−G}⊙k        [4][KB] blocks (else = a)
  int t;     // T                           10 blocks
  int q;     // scale·q, fold: ⊙e^G         [4][KB] blocks
  int at;    // attn                        10 blocks
  int vec;   // xe, ys, gk, G [64] each, then egl [16·KB]
  int per;
};
__host__ __device__ constexpr Lay lay(int KB, bool fold) {
  Lay o{};
  const int tile = 4 * KB * kBlk;
  o.a = 0;
  o.u = fold ? tile : 0;
  o.t = fold ? 2 * tile : tile;
  o.q = o.t + kTri;
  o.at = o.q + tile;
  o.vec = o.at + kTri;
  o.per = o.vec + 4 * kC + 16 * KB;
  return o;
}

}  // namespace
struct FParams {
  Dims d;
  const void *q, *k, *v;
  const float *erase, *write, *g;
  float* ws;          // [G] chunk-heads of lay().per floats
  const float* s_in;  // scan
  void* y;
  float* s_out;
  // backward
  float *states, *ds_after;  // [G][KB][VB] blocks, accumulator order
  float *xs, *vn, *dvn, *z;  // [G][4][VB] blocks, accumulator order: X, V', dV', dVw = Tᵀ·dV'
  const void* dy;
  const float* ds_final;     // may be null
  float* dstate;
  void *dq, *dk, *dv;
  float *derase, *dwrite, *dg;
  int vec4;                  // q and k (and a per-channel erase gate) readable as 4-element words
};
namespace {

__device__ inline f32x4 zero4() { return f32x4{0.f, 0.f, 0.f, 0.f}; }
__device__ inline f32x4 ld4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ inline void st4(float* p, const f32x4& v) { *reinterpret_cast<f32x4*>(p) = v; }
// The workspace, which the caller aligns to its elements and no further.
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
__device__ inline f32x4 ldw(const float* p) { return *reinterpret_cast<const f32x4_any*>(p); }
__device__ inline void stw(float* p, const f32x4& v) { *reinterpret_cast<f32x4_any*>(p) = v; }

// acc += A·B over a 16-deep contraction from the two operands' lane values.
__device__ inline f32x4 mm(const f32x4& a, const f32x4& b, f32x4 acc) {
#pragma unroll
  for (int r = 0; r < 4; ++r) acc = mfma_f32(a[r], b[r], acc);
  return acc;
}

template <class T>
__device__ inline f32x4 load4(const T* p, size_t at, int n, bool vec) {
  f32x4 x = zero4();
  if (vec) {
    if constexpr (sizeof(T) == 4) {
      x = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(p) + at);
    } else {
      const uint2 w = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint16_t*>(p) + at);
      x = f32x4{lo_f(w.x), hi_f(w.x), lo_f(w.y), hi_f(w.y)};
    }
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (r < n) x[r] = ld(p, at + r);
  }
  return x;
}

// W floats of a chunk's tiles on their way to LDS, in the registers of the 256
// staging threads (t of them).
template <int W>
struct Piece {
  static constexpr int kWords = W / 4, N = (kWords + 255) / 256;
  f32x4 x[N];
  __device__ void load(const float* src, int t) {
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = ldw(src + 4 * min(t + 256 * i, kWords - 1));
  }
  __device__ void store(float* dst, int t) const {
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (256 * (i + 1) <= kWords || t + 256 * i < kWords) st4(dst + 4 * (t + 256 * i), x[i]);
  }
};

// Key blocks a launch is compiled for: head_k_dim rounded up to 32, 64, 96 or 128.
inline int key_blocks(int K) { return 2 * ((K + 31) / 32); }
inline bool folds(const Dims& d) { return d.ew > 1 || d.dw > 1; }
inline size_t chunk_heads(const Dims& d) { return size_t(d.B) * d.N * d.H; }
inline size_t bytes_of(size_t floats) { return align_up(floats * sizeof(float), 256); }

// Teams per scan workgroup: one (a CU of its own per 16 value columns) while
// the device holds them all, else two, which share a chunk's staged tiles.
inline int scan_teams(const Dims& d) {
  const int vb = (d.V + 15) / 16;
  return size_t(d.B) * d.H * vb <= size_t(device_cu_count()) || vb == 1 ? 1 : 2;
}
inline unsigned scan_blocks(const Dims& d, int teams) {
  const int vb = (d.V + 15) / 16;
  return unsigned(((d.B * d.H + 7) / 8) * 8 * ((vb + teams - 1) / teams));
}

inline FParams f32_params(const Dims& d, int qkv_dtype, const void* q, const void* k,
                          const void* v, const float* erase, const float* write, const float* g,
                          const float* state_in, void* ws) {
  FParams p{};
  p.d = d;
  p.q = q;
  p.k = k;
  p.v = v;
  p.erase = erase;
  p.write = write;
  p.g = g;
  p.s_in = state_in;
  p.ws = static_cast<float*>(ws);
  const uintptr_t qk = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k);
  p.vec4 = d.K % 4 == 0 && qk % (qkv_dtype == DN_BF16 ? 8 : 16) == 0 &&
           (d.ew == 1 || reinterpret_cast<uintptr_t>(erase) % 16 == 0);
  return p;
}

}  // namespace

// The intra kernel, and the scan (states: the backward's, else the forward's).
hipError_t f32_intra(const FParams& p, int qkv_dtype, hipStream_t stream);
hipError_t f32_scan(const FParams& p, int qkv_dtype, int y_dtype, bool states,
                    hipStream_t stream);

}  // namespace dn
