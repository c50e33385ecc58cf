// The chunk-local gradients of the chunkwise WY form on CDNA4 matrix cores
// with per-head gates, at head_k_dim 256 and in the smallest tiles
// (own_shape); chunk_bwd_local.hip holds the other shapes.
//
// combined_backward.rs:103-188 (WY and front-end terms), :240-319 (the
// per-chunk terms of the reverse walk) and :376-416 (the score backward),
// for one chunk-head per workgroup (8 waves), given what the two MFMA scans
// leave behind: the state S₀ entering the chunk and the cotangent dS of the
// state leaving it (fp32), and the intra kernel's T, Tᵀ (bf16 hi + lo) and
// attnᵀ tiles. With X = w⊙V − kg·S₀ (so that V' = U − W·S₀ = T·X):
//
//   phase A  (a wave per 16 value columns)
//            X;  V' = T·X;  dV' = attnᵀ·dY + kc·dS;  dVw = Tᵀ·dV'
//            d_v = w⊙dVw, d_write from dVw⊙v
//   phase B  (a wave per 16 key channels; contractions over the value axis)
//            d_kc = V'·dSᵀ;  d_qr = dY·S₀ᵀ;  d_kg = −dVw·S₀ᵀ (= Tᵀ·dW with
//            dW = −dV'·S₀ᵀ);  Σ_v dS⊙S₀;  dattn = dY·V'ᵀ
//   phase C  dT = dV'·Xᵀ (= dU·Vwᵀ + dW·kgᵀ, without the cancellation of the
//            two terms);  dAkk = −tril(Tᵀ·dT·Tᵀ, −1) as (dTᵀ·T)ᵀ·Tᵀ
//   phase D  (a wave per 16 key channels) the score backward of the head
//            decay, the gate terms and the reverse cumulative sum of d_g.
//
// Every product runs on v_mfma_f32_16x16x32_bf16 with fp32 intermediates as
// bf16 hi + lo parts (three MFMAs; two when one side is an exact bf16 input),
// which keeps the gradients at fp32-like accuracy. Intermediates pass between
// the phases through one LDS region that each phase re-carves.

#include <type_traits>

#include "dn_common.hpp"
#include "mfma_util.hpp"

namespace dn {
namespace {

constexpr int kL = 64;
constexpr int kW = 8;
constexpr int kNT = 64 * kW;

struct CbParams {
  int S, H, N;
  int gated;
  float scale;
  const uint16_t *q, *k, *v;
  const float *erase, *write, *g;
  const void* dy;
  const uint16_t *T, *Tlo, *Tt, *Ttl, *AtT;  // [G][64][64]
  const float* gc;                           // [G][64] in-chunk cumulative gate
  const float* states;                       // [G][K][V]
  const float* ds_after;                     // [G][K][V]
  void *dq, *dk, *dv;
  float *derase, *dwrite, *dg;
  // The value axis in passes of at most 128 columns: this pass covers
  // columns voff … voff + V − 1 of rows vs wide (v, dO, dv, S₀ and dS). pass 0: the only pass; 1: the first of several, whose
  // value-summed outputs go to the fp32 partials; 2: a middle one, added to
  // them by atomics (nothing waits on them); 3: the last, which adds them and
  // stores.
  int vs, voff, pass;
  // head_k_dim 256 (KA = 2K): each value pass runs as two
  // launches, one per half of the key channels; phase A contracts over all
  // KA keys in both and only the first (koff = 0) stores its outputs. rpass:
  // the pass code (as `pass`) of the sums over key channels (d_g,
  // d_erase) across all the launches of a call; `pass` where KA = K.
  int koff, rpass;
  float *pq, *pk, *pe, *pg, *pw;  // partials of d_q, d_k, d_erase, d_g, d_write
  // Several passes: each thread's partial sums of dattn
  // and dT (16 fp32 per thread per chunk-head), which the passes before the
  // last hand on so that the last runs the score backward once.
  float* pda;
};

// A value-summed output (d_q, d_k, d_erase, d_g, d_write): a sum
// over the value axis, so over the passes (CbParams::pass). The last pass
// reads the partial here, a round trip before the store, unless the caller
// loaded it ahead (st_last).
template <class T>
__device__ inline void st_sum(int pass, T* out, float* part, size_t i, float v) {
  if (pass == 1)
    part[i] = v;
  else if (pass == 2)
    atomicAdd(part + i, v);
  else
    st(out, i, pass == 3 ? v + part[i] : v);
}
// st_sum with the last pass's partial already in `pre` (0 when not the last).
template <class T>
__device__ inline void st_pre(int pass, T* out, float* part, size_t i, float v, float pre) {
  if (pass == 1)
    part[i] = v;
  else if (pass == 2)
    atomicAdd(part + i, v);
  else
    st(out, i, v + pre);
}

__device__ inline uint16_t bf_bits(float x) { return __builtin_bit_cast(uint16_t, (__bf16)x); }

// Four floats → packed bf16 hi parts and lo parts (8-byte LDS stores).
__device__ inline void split4(const float* f, uint2& h, uint2& l) {
  h = make_uint2(pk_bf16(f[0], f[1]), pk_bf16(f[2], f[3]));
  l = make_uint2(pk_bf16(f[0] - lo_f(h.x), f[1] - hi_f(h.x)),
                 pk_bf16(f[2] - lo_f(h.y), f[3] - hi_f(h.y)));
}

// A 64×64 bf16 tile (global, row-major) → LDS with the permuted column order:
// thread tid loads 16-byte chunk tid (512 threads, one each), then stores it.
__device__ inline uint4 load_perm(const uint16_t* src, int tid) {
  return *reinterpret_cast<const uint4*>(src + (tid >> 3) * kL + 8 * (tid & 7));
}
__device__ inline void store_perm(uint16_t* R, int dst, const uint4& v, int tid) {
  const int row = tid >> 3, c8 = tid & 7;
  *reinterpret_cast<uint2*>(&R[dst + tile_at<kL>(row, perm_pos(8 * c8))]) = make_uint2(v.x, v.y);
  *reinterpret_cast<uint2*>(&R[dst + tile_at<kL>(row, perm_pos(8 * c8 + 4))]) =
      make_uint2(v.z, v.w);
}
__device__ inline void stage_perm(uint16_t* R, int dst, const uint16_t* src, int tid) {
  store_perm(R, dst, load_perm(src, tid), tid);
}

// The 16 lower-or-diagonal and upper 16×16 tiles of a 64×64 matrix, two per
// wave: tile t = wave + 8u is (t/4, t%4).

// LASTP (the last of several value passes): the partials
// of the value-summed outputs are loaded at the start of phase D, so their
// round trip overlaps the score backward instead of preceding each store.
// EARLY (the passes before the last): dattn and dT are sums
// over the value axis, and everything after them is linear in them, so these
// passes add their partial sums to p.pda and stop after phase C's first
// product; the score backward (the rest of phase C and phase D's scores) runs
// once, in the last pass, on the summed dattn and dT. They still store their
// share of the value-summed gradients (phase B's terms).
// KA: the head_k_dim of the tensors; phase A's contractions run over all KA
// keys and phases B–D over K of them from channel p.koff on (KA = 2K: the
// key halves of head_k_dim 256).
template <int K, int V, class TG, bool LASTP = false, bool EARLY = false, int KA = K>
__global__ __launch_bounds__(kNT) void mfma_chunk_bwd_kernel(CbParams p) {
  static_assert(KA == K || KA == 2 * K, "all keys, or one of their halves");
  constexpr int KS = KA;  // row stride of q, k, the states and the key-channel outputs
  // The states and state cotangents in row groups of four, [G][K/4][V][4]
  // at head_k_dim 256 (mfma_bwd_scans), else [G][K][V].
  constexpr bool G4 = KA == 256;
  static_assert(!(EARLY && LASTP), "partial score sums: not the last pass");
  constexpr bool F32DY = std::is_same<TG, float>::value;
  constexpr int TT = kL * kL, TK = kL * K, TKA = kL * KA, TV = kL * V;
  constexpr int OFF_A1 = 4 * TV > 8 * TT ? 4 * TV : 8 * TT;
  constexpr int RBIG = OFF_A1 + 4 * TT;
  static_assert(5 * TT + TKA <= RBIG, "phase-A operands fit");
  static_assert((F32DY ? 6 : 5) * TV <= RBIG, "phase-B operands fit");
  static_assert(4 * TT + 2 * TK <= OFF_A1, "score operands fit");
  // Carvings of R (bf16 elements):
  //  A  T hi/lo, Tᵀ hi/lo (permuted), attnᵀ (permuted), k
  constexpr int oTh = 0, oTl = TT, oTth = 2 * TT, oTtl = 3 * TT, oAt = 4 * TT, oKop = 5 * TT;
  //  B  V' hi/lo, dVw hi/lo, dY hi(/lo)
  constexpr int oVh = 0, oVl = TV, oWh = 2 * TV, oWl = 3 * TV, oYh = 4 * TV, oYl = 5 * TV;
  //  C  X hi/lo, dV' hi/lo; dAqk as [i][j] and [j][i] (hi/lo) at OFF_A1 until the end
  constexpr int oXh = 0, oXl = TV, oDh = 2 * TV, oDl = 3 * TV;
  constexpr int oA1h = OFF_A1, oA1l = OFF_A1 + TT, oA1th = OFF_A1 + 2 * TT,
                oA1tl = OFF_A1 + 3 * TT;
  //     then T and Tᵀ again, dTᵀ (permuted over dT's rows), M₁ = Tᵀ·dT
  constexpr int oDTh = 4 * TT, oDTl = 5 * TT, oM1h = 6 * TT, oM1l = 7 * TT;
  //  D  dAkk as [i][j] and [j][i] (hi/lo); Kᵀ, Qᵀ
  constexpr int oA0h = 0, oA0l = TT, oA0th = 2 * TT, oA0tl = 3 * TT, oKC = 4 * TT,
                oQC = 4 * TT + TK;
  __shared__ __attribute__((aligned(16))) uint16_t R[RBIG];
  __shared__ __attribute__((aligned(16))) float Gc[kL];
  __shared__ float er_s[kL], wr_s[kL], eg_s[kL], ec_s[kL];
  __shared__ float racc[3][kL];  // row sums: d_write, d_erase, d_g

  const int cid = blockIdx.x;
  const int h = cid % p.H, n = (cid / p.H) % p.N, b = cid / (p.H * p.N);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r16 = lane & 15, g4 = lane >> 4, k8 = 8 * g4;
  const int tok0 = n * kL;
  const int valid = min(kL, p.S - tok0);
  const size_t row0 = size_t(b) * p.S * p.H + h + size_t(tok0) * p.H;
  auto row_of = [&](int t) { return row0 + size_t(t) * p.H; };
  // Global reads are unconditional: a row past the sequence end reads the
  // chunk's last row (valid ≥ 1) and the value is then dropped. A load under
  // a lane guard becomes a branch of its own with a full wait on every load
  // in flight, which serialised the staging.
  auto rowc = [&](int t) { return row_of(min(t, valid - 1)); };
  const size_t o64 = size_t(cid) * kL * kL;
  const int VS = p.vs, vo = p.voff;  // row stride and first column of the value axis
  // Row-major: element (row, column) at S0[row·VS + column]; in row groups
  // of four at S0[(row/4·VS + column)·4 + row%4] (the pass's first column
  // is then 4·vo floats in).
  const float* S0 = p.states + size_t(cid) * KS * VS + (G4 ? 4 * vo : vo);
  const float* dSa = p.ds_after + size_t(cid) * KS * VS + (G4 ? 4 * vo : vo);
  // This launch's first key channel (phases B–D), and whether it stores the
  // outputs of phase A and accumulates the value-summed dattn and dT.
  const int koff = KA == K ? 0 : p.koff;
  const bool store_a = koff == 0;
  const TG* dy = static_cast<const TG*>(p.dy);
  const bool gated = p.gated;
  auto rowi = [&](int ib, int r) { return 16 * ib + 4 * g4 + r; };
  // Row of the value sum16 leaves in this lane (index 4·ib + r).
  const int red_row = 16 * (r16 >> 2) + 4 * g4 + (r16 & 3);

  // ---- staging -----------------------------------------------------------
  // The gate and tile loads are issued together and written to LDS (one
  // round trip); phase A's operand loads follow, in flight across the
  // cumulative sum and the barriers. Loads complete in order, so issuing the
  // phase-A loads first would make every LDS write wait for them too.
  float e0 = 0.f, w0 = 0.f, gct = 0.f, gl = 0.f;
  if (tid < kL) {
    e0 = p.erase[rowc(tid)];
    w0 = p.write[rowc(tid)];
    if (gated) {
      gct = p.gc[size_t(cid) * kL + tid];
      gl = p.gc[size_t(cid) * kL + kL - 1];
    }
  }
  constexpr int NKR = kL * KA / 8 / kNT;  // 16-byte chunks per thread of a [64][KA] tile
  static_assert(NKR * kNT * 8 == kL * KA, "K-wide staging assumes whole rounds");
  uint4 tp[5], tk[NKR];
  tp[0] = load_perm(p.T + o64, tid);
  tp[1] = load_perm(p.Tlo + o64, tid);
  tp[2] = load_perm(p.Tt + o64, tid);
  tp[3] = load_perm(p.Ttl + o64, tid);
  tp[4] = load_perm(p.AtT + o64, tid);
#pragma unroll
  for (int m = 0; m < NKR; ++m) {
    const int idx = tid + kNT * m, row = idx / (KA / 8), c8 = idx % (KA / 8);
    const uint4 x = *reinterpret_cast<const uint4*>(p.k + rowc(row) * KS + 8 * c8);
    tk[m] = row < valid ? x : make_uint4(0u, 0u, 0u, 0u);
  }
  if (tid < kL) {
    const int t = tid;
    const bool ok = t < valid;
    er_s[t] = ok ? e0 : 0.f;
    wr_s[t] = ok ? w0 : 0.f;
    Gc[t] = gct;
    eg_s[t] = gated ? __expf(gct) : 1.f;
    ec_s[t] = gated ? __expf(gl - gct) : 1.f;
    racc[0][t] = racc[1][t] = racc[2][t] = 0.f;
  }
  store_perm(R, oTh, tp[0], tid);
  store_perm(R, oTl, tp[1], tid);
  store_perm(R, oTth, tp[2], tid);
  store_perm(R, oTtl, tp[3], tid);
  store_perm(R, oAt, tp[4], tid);
#pragma unroll
  for (int m = 0; m < NKR; ++m) {
    const int idx = tid + kNT * m, row = idx / (KA / 8), c8 = idx % (KA / 8);
    const int at = tile_at<KA>(row, 8 * c8);
    *reinterpret_cast<uint4*>(&R[oKop + at]) = tk[m];
  }

  // ---- phase A's global operands -------------------------------------------
  const bool vwave = wave < V / 16;
  const int col = 16 * wave + r16;  // this lane's value column in phase A
  // S₀ and dS for PDEP k-steps at a time: all of them at head_k_dim ≤ 128;
  // at 256 the first four, each register set reloaded with the k-step four
  // ahead once its fragments are split.
  constexpr int KAS = KA / 32, PDEP = KAS > 4 ? 4 : KAS;
  float pS[PDEP][8], pD[PDEP][8], vv[4][4], wv[4][4], dyv[2][8];
  auto load_sd = [&](float (&dst)[8], const float* src, int s) {
    if constexpr (G4) {
      // rows 32s + k8 … +3 and +4 … +7 of column col: two 16-byte loads
      const float4* b = reinterpret_cast<const float4*>(src) + size_t(8 * s + 2 * g4) * VS + col;
      const float4 lo = b[0], hi = b[VS];
      dst[0] = lo.x; dst[1] = lo.y; dst[2] = lo.z; dst[3] = lo.w;
      dst[4] = hi.x; dst[5] = hi.y; dst[6] = hi.z; dst[7] = hi.w;
    } else {
#pragma unroll
      for (int t = 0; t < 8; ++t) dst[t] = src[size_t(32 * s + k8 + t) * VS + col];
    }
  };
  if (vwave) {
    // S₀ and dS rows 32·s + 8·(lane/16) + t of this lane's column (B operands
    // of kg·S₀ and kc·dS).
    if constexpr (G4) {
#pragma unroll
      for (int s = 0; s < PDEP; ++s) {
        load_sd(pS[s], S0, s);
        load_sd(pD[s], dSa, s);
      }
    } else {
#pragma unroll
      for (int s = 0; s < PDEP; ++s)
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          pS[s][t] = S0[size_t(32 * s + k8 + t) * VS + col];
          pD[s][t] = dSa[size_t(32 * s + k8 + t) * VS + col];
        }
    }
#pragma unroll
    for (int ib = 0; ib < 4; ++ib)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = rowi(ib, r);
        const float x = bf16_to_f32(p.v[rowc(i) * VS + vo + col]);
        vv[ib][r] = i < valid ? x : 0.f;
      }
    // dY in the permuted token order of the attnᵀ fragments: token 4q+e /
    // 16+4q+e of each 32-token step at position 8q+e / 8q+4+e.
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int t = 32 * kk + (e < 4 ? 4 * g4 + e : 16 + 4 * g4 + e - 4);
        const float x = ld(dy, rowc(t) * VS + vo + col);
        dyv[kk][e] = t < valid ? x : 0.f;
      }
  }
  __syncthreads();

  // ---- phase A: value columns ---------------------------------------------
  f32x4 X[4], dV[4], Vn[4], dW[4];
  if (vwave) {
#pragma unroll
    for (int ib = 0; ib < 4; ++ib)
#pragma unroll
      for (int r = 0; r < 4; ++r) wv[ib][r] = wr_s[rowi(ib, r)];
    // X = w⊙V − kg·S₀ (S₀ as hi + lo parts; k exact, e·e^G per row).
#pragma unroll
    for (int ib = 0; ib < 4; ++ib) X[ib] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KAS; ++s) {
      uint4 sh, sl;
      split8(pS[s % PDEP], sh, sl);
      if (s + PDEP < KAS) {
        // (a scheduling barrier: hoisted to the staging, these reloads
        // spilled the loaded values there, each load waited for in turn)
        __builtin_amdgcn_sched_barrier(0);
        load_sd(pS[s % PDEP], S0, s + PDEP);
      }
#pragma unroll
      for (int ib = 0; ib < 4; ++ib) {
        const int at = tile_at<KA>(16 * ib + r16, 32 * s + k8);
        const uint4 a = ld8u(&R[oKop + at]);
        X[ib] = mfma16(a, sh, X[ib]);
        X[ib] = mfma16(a, sl, X[ib]);
      }
    }
#pragma unroll
    for (int ib = 0; ib < 4; ++ib)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = rowi(ib, r);
        const float sc = er_s[i] * eg_s[i];
        X[ib][r] = vv[ib][r] * wv[ib][r] - sc * X[ib][r];
      }
    // V' = T·X (hi + lo parts of both).
#pragma unroll
    for (int ib = 0; ib < 4; ++ib) Vn[ib] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const uint4 xh = frag_hi(X[2 * kk], X[2 * kk + 1]);
      const uint4 xl = frag_lo(X[2 * kk], X[2 * kk + 1], xh);
#pragma unroll
      for (int ib = 0; ib < 4; ++ib) {
        if (kk > (ib >> 1)) continue;  // T is lower triangular
        const int at = tile_at<kL>(16 * ib + r16, 32 * kk + k8);
        const uint4 th = ld8u(&R[oTh + at]), tl = ld8u(&R[oTl + at]);
        Vn[ib] = mfma16(th, xh, Vn[ib]);
        Vn[ib] = mfma16(tl, xh, Vn[ib]);
        Vn[ib] = mfma16(th, xl, Vn[ib]);
      }
    }
    // dV' = attnᵀ·dY + kc·dS (dY fragments: token 4q+e / 16+4q+e of each
    // 32-token step at position 8q+e / 8q+4+e, the permuted order).
    uint4 yh[2], yl[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) split8(dyv[kk], yh[kk], yl[kk]);
#pragma unroll
    for (int ib = 0; ib < 4; ++ib) {
      dV[ib] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        if (kk < (ib >> 1)) continue;  // attnᵀ is upper triangular
        const uint4 a = ld8u(&R[oAt + tile_at<kL>(16 * ib + r16, 32 * kk + k8)]);
        dV[ib] = mfma16(a, yh[kk], dV[ib]);
        if constexpr (F32DY) dV[ib] = mfma16(a, yl[kk], dV[ib]);
      }
    }
    {
      f32x4 kd[4];
#pragma unroll
      for (int ib = 0; ib < 4; ++ib) kd[ib] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KAS; ++s) {
        uint4 dh, dl;
        split8(pD[s % PDEP], dh, dl);
        if (s + PDEP < KAS) {
          __builtin_amdgcn_sched_barrier(0);
          load_sd(pD[s % PDEP], dSa, s + PDEP);
        }
#pragma unroll
        for (int ib = 0; ib < 4; ++ib) {
          const uint4 a = ld8u(&R[oKop + tile_at<KA>(16 * ib + r16, 32 * s + k8)]);
          kd[ib] = mfma16(a, dh, kd[ib]);
          kd[ib] = mfma16(a, dl, kd[ib]);
        }
      }
#pragma unroll
      for (int ib = 0; ib < 4; ++ib)
#pragma unroll
        for (int r = 0; r < 4; ++r) dV[ib][r] += ec_s[rowi(ib, r)] * kd[ib][r];
    }
    // dVw = Tᵀ·dV'.
#pragma unroll
    for (int ib = 0; ib < 4; ++ib) dW[ib] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const uint4 vh = frag_hi(dV[2 * kk], dV[2 * kk + 1]);
      const uint4 vl = frag_lo(dV[2 * kk], dV[2 * kk + 1], vh);
#pragma unroll
      for (int ib = 0; ib < 4; ++ib) {
        if (kk < (ib >> 1)) continue;  // Tᵀ is upper triangular
        const int at = tile_at<kL>(16 * ib + r16, 32 * kk + k8);
        const uint4 th = ld8u(&R[oTth + at]), tl = ld8u(&R[oTtl + at]);
        dW[ib] = mfma16(th, vh, dW[ib]);
        dW[ib] = mfma16(tl, vh, dW[ib]);
        dW[ib] = mfma16(th, vl, dW[ib]);
      }
    }
    // d_v = w⊙dVw; d_write = dVw⊙v, summed over the value axis for width 1.
    TG* gv = static_cast<TG*>(p.dv);
    float rs[16];
#pragma unroll
    for (int ib = 0; ib < 4; ++ib)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = rowi(ib, r);
        if (store_a && i < valid) st(gv, row_of(i) * VS + vo + col, dW[ib][r] * wv[ib][r]);
        rs[4 * ib + r] = dW[ib][r] * vv[ib][r];
      }
    atomicAdd(&racc[0][red_row], sum16(rs, lane));
  }
  // dY rows for LDS, then phase B's global operands: S₀ and dS rows of this
  // lane's key channel.
  constexpr int NY = kL * V / 8 / kNT;  // 16-byte chunks of dY rows per thread
  static_assert(NY * kNT * 8 == kL * V, "dY staging assumes whole rounds");
  float ydat[NY][8];
#pragma unroll
  for (int m = 0; m < NY; ++m) {
    const int idx = tid + kNT * m, i = idx / (V / 8), c8 = idx % (V / 8);
    if constexpr (F32DY) {
      const float4* src = reinterpret_cast<const float4*>(dy + rowc(i) * VS + vo + 8 * c8);
      float4 a = src[0], b2 = src[1];
      if (i >= valid) a = b2 = make_float4(0.f, 0.f, 0.f, 0.f);
      ydat[m][0] = a.x; ydat[m][1] = a.y; ydat[m][2] = a.z; ydat[m][3] = a.w;
      ydat[m][4] = b2.x; ydat[m][5] = b2.y; ydat[m][6] = b2.z; ydat[m][7] = b2.w;
    } else {
      uint4 v = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(dy) +
                                                rowc(i) * VS + vo + 8 * c8);
      if (i >= valid) v = make_uint4(0u, 0u, 0u, 0u);
      unpack8(v, ydat[m]);
    }
  }
  const bool kwave = wave < K / 16;
  const int c = 16 * wave + r16;  // this lane's key channel in phases B and D
  float bS[V / 32][8], bD[V / 32][8];
  if (kwave) {
    if constexpr (G4) {
      // row koff + c: element (koff + c)%4 of each column's row group
      const int row = koff + c;
      const size_t o = size_t(row >> 2) * VS * 4 + (row & 3);
#pragma unroll
      for (int s = 0; s < V / 32; ++s)
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          bS[s][t] = S0[o + size_t(32 * s + k8 + t) * 4];
          bD[s][t] = dSa[o + size_t(32 * s + k8 + t) * 4];
        }
    } else {
#pragma unroll
      for (int s = 0; s < V / 32; ++s) {
        const float4* s0r = reinterpret_cast<const float4*>(S0 + size_t(koff + c) * VS + 32 * s + k8);
        const float4* dsr = reinterpret_cast<const float4*>(dSa + size_t(koff + c) * VS + 32 * s + k8);
        *reinterpret_cast<float4*>(bS[s]) = s0r[0];
        *reinterpret_cast<float4*>(bS[s] + 4) = s0r[1];
        *reinterpret_cast<float4*>(bD[s]) = dsr[0];
        *reinterpret_cast<float4*>(bD[s] + 4) = dsr[1];
      }
    }
  }
  __syncthreads();

  // ---- V', dVw and dY rows into LDS ---------------------------------------
  if (vwave) {
#pragma unroll
    for (int ib = 0; ib < 4; ++ib)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int at = tile_at<V>(rowi(ib, r), col);
        const uint16_t vh = bf_bits(Vn[ib][r]), wh = bf_bits(dW[ib][r]);
        R[oVh + at] = vh;
        R[oVl + at] = bf_bits(Vn[ib][r] - bf16_to_f32(vh));
        R[oWh + at] = wh;
        R[oWl + at] = bf_bits(dW[ib][r] - bf16_to_f32(wh));
      }
  }
#pragma unroll
  for (int m = 0; m < NY; ++m) {
    const int idx = tid + kNT * m, i = idx / (V / 8), c8 = idx % (V / 8);
    const int at = tile_at<V>(i, 8 * c8);
    uint4 hh, ll;
    split8(ydat[m], hh, ll);
    *reinterpret_cast<uint4*>(&R[oYh + at]) = hh;
    if constexpr (F32DY) *reinterpret_cast<uint4*>(&R[oYl + at]) = ll;
  }
  __syncthreads();

  // ---- phase B: key channels; contractions over the value axis ------------
  f32x4 dkA[4], dqA[4], dkeA[4];
  float degl = 0.f;
  if (kwave) {
    f32x4 aKc[4], aQr[4], aKg[4];
#pragma unroll
    for (int ib = 0; ib < 4; ++ib)
      aKc[ib] = aQr[ib] = aKg[ib] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < V / 32; ++s) {
#pragma unroll
      for (int t = 0; t < 8; ++t) degl += bS[s][t] * bD[s][t];
      uint4 sh, sl, dh, dl;
      split8(bS[s], sh, sl);
      split8(bD[s], dh, dl);
#pragma unroll
      for (int ib = 0; ib < 4; ++ib) {
        const int at = tile_at<V>(16 * ib + r16, 32 * s + k8);
        const uint4 vh = ld8u(&R[oVh + at]), vl = ld8u(&R[oVl + at]);
        aKc[ib] = mfma16(vh, dh, aKc[ib]);
        aKc[ib] = mfma16(vl, dh, aKc[ib]);
        aKc[ib] = mfma16(vh, dl, aKc[ib]);
        const uint4 yh = ld8u(&R[oYh + at]);
        aQr[ib] = mfma16(yh, sh, aQr[ib]);
        aQr[ib] = mfma16(yh, sl, aQr[ib]);
        if constexpr (F32DY) aQr[ib] = mfma16(ld8u(&R[oYl + at]), sh, aQr[ib]);
        const uint4 wh = ld8u(&R[oWh + at]), wl = ld8u(&R[oWl + at]);
        aKg[ib] = mfma16(wh, sh, aKg[ib]);
        aKg[ib] = mfma16(wl, sh, aKg[ib]);
        aKg[ib] = mfma16(wh, sl, aKg[ib]);
      }
    }
    degl += __shfl_xor(degl, 16);
    degl += __shfl_xor(degl, 32);
    // The scan's cotangents through the gates (combined_backward.rs:284-313):
    // d_k = d_kc⊙e^{G_last−G}, d_q = d_qr⊙e^G, d_ke = d_kg⊙e^G (their d_G
    // pieces follow in phase D, where K and Q are staged).
#pragma unroll
    for (int ib = 0; ib < 4; ++ib)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = rowi(ib, r);
        const float eg = eg_s[i], ec = ec_s[i];
        dkA[ib][r] = aKc[ib][r] * ec;
        dqA[ib][r] = aQr[ib][r] * eg;
        dkeA[ib][r] = -aKg[ib][r] * eg;
      }
  }
  // dattn = dY·V'ᵀ on the lower tiles.
  f32x4 dat[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int t = wave + 8 * u, ti = t >> 2, tj = t & 3;
    dat[u] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (tj <= ti) {
#pragma unroll
      for (int s = 0; s < V / 32; ++s) {
        const int aa = tile_at<V>(16 * ti + r16, 32 * s + k8);
        const int ab = tile_at<V>(16 * tj + r16, 32 * s + k8);
        const uint4 yh = ld8u(&R[oYh + aa]);
        const uint4 bh = ld8u(&R[oVh + ab]), bl = ld8u(&R[oVl + ab]);
        dat[u] = mfma16(yh, bh, dat[u]);
        dat[u] = mfma16(yh, bl, dat[u]);
        if constexpr (F32DY) dat[u] = mfma16(ld8u(&R[oYl + aa]), bh, dat[u]);
      }
    }
  }
  // The earlier passes' dattn and dT partial sums (this thread's 16 slots).
  float* const da = !p.pda ? nullptr : p.pda + (size_t(cid) * kNT + tid) * 16;
  f32x4 pda_r[4];
  if (LASTP || (EARLY && p.pass == 2 && store_a))
#pragma unroll
    for (int j = 0; j < 4; ++j) pda_r[j] = reinterpret_cast<const f32x4*>(da)[j];
  __syncthreads();

  // ---- X, dV' rows and the dAqk layouts into LDS --------------------------
  if (vwave) {
#pragma unroll
    for (int ib = 0; ib < 4; ++ib)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int at = tile_at<V>(rowi(ib, r), col);
        const uint16_t xh = bf_bits(X[ib][r]), dh = bf_bits(dV[ib][r]);
        R[oXh + at] = xh;
        R[oXl + at] = bf_bits(X[ib][r] - bf16_to_f32(xh));
        R[oDh + at] = dh;
        R[oDl + at] = bf_bits(dV[ib][r] - bf16_to_f32(dh));
      }
  }
  if (LASTP || (EARLY && p.pass == 2 && store_a))
#pragma unroll
    for (int u = 0; u < 2; ++u) dat[u] += pda_r[u];
  if constexpr (EARLY) {
    if (store_a)
#pragma unroll
      for (int u = 0; u < 2; ++u) reinterpret_cast<f32x4*>(da)[u] = dat[u];
  }
  // dAqk = tril(dattn) ⊙ e^{Gᵢ−Gⱼ} (the head mask) as [i][j] and as [j][i]
  // (times the readout scale).
  if constexpr (!EARLY) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int t = wave + 8 * u, ti = t >> 2, tj = t & 3;
      const int j = 16 * tj + r16;
      float f[4], ft[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 16 * ti + 4 * g4 + r;
        float val = 0.f;
        if (j <= i) {
          val = dat[u][r];
          if (gated) val *= __expf(Gc[i] - Gc[j]);
        }
        f[r] = val;
        ft[r] = val * p.scale;
        const int at = tile_at<kL>(i, j);
        const uint16_t vh = bf_bits(val);
        R[oA1h + at] = vh;
        R[oA1l + at] = bf_bits(val - bf16_to_f32(vh));
      }
      uint2 hh, ll;
      split4(ft, hh, ll);
      const int at = tile_at<kL>(j, 16 * ti + 4 * g4);
      *reinterpret_cast<uint2*>(&R[oA1th + at]) = hh;
      *reinterpret_cast<uint2*>(&R[oA1tl + at]) = ll;
    }
  }
  __syncthreads();

  // ---- phase C: dT = dV'·Xᵀ (strict lower) --------------------------------
  f32x4 dTt[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int t = wave + 8 * u, ti = t >> 2, tj = t & 3;
    dTt[u] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (tj <= ti) {
#pragma unroll
      for (int s = 0; s < V / 32; ++s) {
        const int aa = tile_at<V>(16 * ti + r16, 32 * s + k8);
        const int ab = tile_at<V>(16 * tj + r16, 32 * s + k8);
        const uint4 ah = ld8u(&R[oDh + aa]), al = ld8u(&R[oDl + aa]);
        const uint4 bh = ld8u(&R[oXh + ab]), bl = ld8u(&R[oXl + ab]);
        dTt[u] = mfma16(ah, bh, dTt[u]);
        dTt[u] = mfma16(al, bh, dTt[u]);
        dTt[u] = mfma16(ah, bl, dTt[u]);
      }
    }
  }
  __syncthreads();
  if (LASTP || (EARLY && p.pass == 2 && store_a))
#pragma unroll
    for (int u = 0; u < 2; ++u) dTt[u] += pda_r[2 + u];
  if constexpr (EARLY) {
    if (store_a)
#pragma unroll
      for (int u = 0; u < 2; ++u) reinterpret_cast<f32x4*>(da)[2 + u] = dTt[u];
  } else {
    // dTᵀ with dT's row index permuted (it is the contraction index of dTᵀ·T);
    // T and Tᵀ staged again.
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int t = wave + 8 * u, ti = t >> 2, tj = t & 3;
      float f[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int a = 16 * ti + 4 * g4 + r, bcol = 16 * tj + r16;
        f[r] = bcol < a ? dTt[u][r] : 0.f;
      }
      uint2 hh, ll;
      split4(f, hh, ll);
      const int at = tile_at<kL>(16 * tj + r16, 32 * (ti >> 1) + 8 * g4 + 4 * (ti & 1));
      *reinterpret_cast<uint2*>(&R[oDTh + at]) = hh;
      *reinterpret_cast<uint2*>(&R[oDTl + at]) = ll;
    }
    stage_perm(R, oTh, p.T + o64, tid);
    stage_perm(R, oTl, p.Tlo + o64, tid);
    stage_perm(R, oTth, p.Tt + o64, tid);
    stage_perm(R, oTtl, p.Ttl + o64, tid);
    __syncthreads();
    // M₁ᵀ = dTᵀ·T (all 16 tiles), stored as M₁ with its column index permuted.
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int t = wave + 8 * u, bt = t >> 2, it = t & 3;
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        // dTᵀ and Tᵀ are upper triangular: k-step 0 (j < 32) vanishes for
        // row blocks 2 and 3 of either.
        if (kk < (max(bt, it) >> 1)) continue;
        const int aa = tile_at<kL>(16 * bt + r16, 32 * kk + k8);
        const int ab = tile_at<kL>(16 * it + r16, 32 * kk + k8);
        const uint4 ah = ld8u(&R[oDTh + aa]), al = ld8u(&R[oDTl + aa]);
        const uint4 bh = ld8u(&R[oTth + ab]), bl = ld8u(&R[oTtl + ab]);
        acc = mfma16(ah, bh, acc);
        acc = mfma16(al, bh, acc);
        acc = mfma16(ah, bl, acc);
      }
      float f[4] = {acc[0], acc[1], acc[2], acc[3]};
      uint2 hh, ll;
      split4(f, hh, ll);
      const int at = tile_at<kL>(16 * it + r16, 32 * (bt >> 1) + 8 * g4 + 4 * (bt & 1));
      *reinterpret_cast<uint2*>(&R[oM1h + at]) = hh;
      *reinterpret_cast<uint2*>(&R[oM1l + at]) = ll;
    }
    __syncthreads();
    // dAkk = −tril(M₁·Tᵀ, −1); T[j][b] vanishes for b > j.
    f32x4 dak[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int t = wave + 8 * u, ti = t >> 2, tj = t & 3;
      dak[u] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (tj <= ti) {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          if (kk > (tj >> 1)) continue;
          const int aa = tile_at<kL>(16 * ti + r16, 32 * kk + k8);
          const int ab = tile_at<kL>(16 * tj + r16, 32 * kk + k8);
          const uint4 ah = ld8u(&R[oM1h + aa]), al = ld8u(&R[oM1l + aa]);
          const uint4 bh = ld8u(&R[oTh + ab]), bl = ld8u(&R[oTl + ab]);
          dak[u] = mfma16(ah, bh, dak[u]);
          dak[u] = mfma16(al, bh, dak[u]);
          dak[u] = mfma16(ah, bl, dak[u]);
        }
      }
    }
    __syncthreads();
    // dAkk ⊙ the head mask as [i][j] and as [j][i] (times the erase gate of
    // row i); Kᵀ and Qᵀ.
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int t = wave + 8 * u, ti = t >> 2, tj = t & 3;
      const int j = 16 * tj + r16;
      float ft[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 16 * ti + 4 * g4 + r;
        float val = 0.f;
        if (j < i) {
          val = -dak[u][r];
          if (gated) val *= __expf(Gc[i] - Gc[j]);
        }
        ft[r] = val * er_s[i];
        const int at = tile_at<kL>(i, j);
        const uint16_t vh = bf_bits(val);
        R[oA0h + at] = vh;
        R[oA0l + at] = bf_bits(val - bf16_to_f32(vh));
      }
      uint2 hh, ll;
      split4(ft, hh, ll);
      const int at = tile_at<kL>(j, 16 * ti + 4 * g4);
      *reinterpret_cast<uint2*>(&R[oA0th + at]) = hh;
      *reinterpret_cast<uint2*>(&R[oA0tl + at]) = ll;
    }
  }
  for (int idx = tid; idx < kL * K / 8; idx += kNT) {
    const int i = idx / (K / 8), c8 = idx % (K / 8);
    uint4 kv = *reinterpret_cast<const uint4*>(p.k + rowc(i) * KS + koff + 8 * c8);
    uint4 qv = *reinterpret_cast<const uint4*>(p.q + rowc(i) * KS + koff + 8 * c8);
    if (i >= valid) kv = qv = make_uint4(0u, 0u, 0u, 0u);
    const uint32_t kw[4] = {kv.x, kv.y, kv.z, kv.w}, qw[4] = {qv.x, qv.y, qv.z, qv.w};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int at = tile_at<kL>(8 * c8 + e, i);
      R[oKC + at] = uint16_t(kw[e >> 1] >> (16 * (e & 1)));
      R[oQC + at] = uint16_t(qw[e >> 1] >> (16 * (e & 1)));
    }
  }
  __syncthreads();

  // ---- phase D: score backward, gates, stores -----------------------------
  // The last pass's partials: d_q and d_k at this lane's 16 rows and channel;
  // d_write at row `lane` (stored by wave 0).
  float pre_q[16], pre_k[16], pre_w = 0.f;
  if constexpr (LASTP) {
    if (kwave) {
#pragma unroll
      for (int ib = 0; ib < 4; ++ib)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const size_t at = rowc(rowi(ib, r)) * KS + koff + c;
          pre_q[4 * ib + r] = p.pq[at];
          pre_k[4 * ib + r] = p.pk[at];
        }
    }
    if (wave == 0) {
      // (d_erase and d_g, sums over key channels too, go through st_sum(rpass))
      pre_w = p.pw[rowc(lane)];
    }
  }
  if (kwave) {
    TG* gq = static_cast<TG*>(p.dq);
    TG* gk = static_cast<TG*>(p.dk);
    // d_G of the scan (combined_backward.rs:284-313): −d_carry + (d_qr⊙qs +
    // d_kg⊙ke)⊙e^G = −dkA⊙k + dqA⊙q·scale + dkeA⊙k⊙e with phase B's
    // accumulators, and d(G_last) = Σ_i d_carry + (Σ_v dS⊙S₀)·e^{G_last}.
    if (gated) {
      float carry = 0.f, rowv[16];
#pragma unroll
      for (int ib = 0; ib < 4; ++ib) {
        const uint2 k4 = *reinterpret_cast<const uint2*>(&R[oKC + tile_at<kL>(c, 16 * ib + 4 * g4)]);
        const uint2 q4 = *reinterpret_cast<const uint2*>(&R[oQC + tile_at<kL>(c, 16 * ib + 4 * g4)]);
        const float kv[4] = {lo_f(k4.x), hi_f(k4.x), lo_f(k4.y), hi_f(k4.y)};
        const float qv[4] = {lo_f(q4.x), hi_f(q4.x), lo_f(q4.y), hi_f(q4.y)};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float e = er_s[rowi(ib, r)];
          const float dcarry = dkA[ib][r] * kv[r];
          const float val = -dcarry + dqA[ib][r] * qv[r] * p.scale + dkeA[ib][r] * kv[r] * e;
          carry += dcarry;
          rowv[4 * ib + r] = val;
        }
      }
      atomicAdd(&racc[2][red_row], sum16(rowv, lane));
      // d(G_last) of the whole head: Σ d_carry + Σ_channels (dS⊙S₀)·e^{G_last}.
      float tot = carry + (g4 == 0 ? degl * eg_s[kL - 1] : 0.f);
#pragma unroll
      for (int m = 32; m >= 1; m >>= 1) tot += __shfl_xor(tot, m);
      if (lane == 0) atomicAdd(&racc[2][kL - 1], tot);
    }
    if constexpr (!EARLY) {  // (the score backward runs in the last pass)
      // head_scores_backward (combined_backward.rs:376-416) with drkk = dAkk⊙M,
      // drqk = dAqk⊙M: d_ke += drkk·K, d_qs += drqk·K, d_k += drkkᵀ·ke +
      // drqkᵀ·qs. The d_G term Σⱼ d_diff[i][j] − d_diff[j][i] of
      // d_diff = (dAkk⊙KeKᵀ + dAqk⊙QsKᵀ)⊙M equals, per row, Σ_c of
      // ke⊙(drkk·K) + qs⊙(drqk·K) − k⊙(drkkᵀ·ke + drqkᵀ·qs).
      f32x4 SK1[4], SQ1[4], SK2[4], SQ2[4];
#pragma unroll
      for (int ib = 0; ib < 4; ++ib)
        SK1[ib] = SQ1[ib] = SK2[ib] = SQ2[ib] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const uint4 kb = ld8u(&R[oKC + tile_at<kL>(c, 32 * s + k8)]);
        const uint4 qb = ld8u(&R[oQC + tile_at<kL>(c, 32 * s + k8)]);
#pragma unroll
        for (int ib = 0; ib < 4; ++ib) {
          const int at = tile_at<kL>(16 * ib + r16, 32 * s + k8);
          if (s <= (ib >> 1)) {
            SK1[ib] = mfma16(ld8u(&R[oA0h + at]), kb, SK1[ib]);
            SK1[ib] = mfma16(ld8u(&R[oA0l + at]), kb, SK1[ib]);
            SQ1[ib] = mfma16(ld8u(&R[oA1h + at]), kb, SQ1[ib]);
            SQ1[ib] = mfma16(ld8u(&R[oA1l + at]), kb, SQ1[ib]);
          }
          if (s >= (ib >> 1)) {
            SK2[ib] = mfma16(ld8u(&R[oA0th + at]), kb, SK2[ib]);
            SK2[ib] = mfma16(ld8u(&R[oA0tl + at]), kb, SK2[ib]);
            SQ2[ib] = mfma16(ld8u(&R[oA1th + at]), qb, SQ2[ib]);
            SQ2[ib] = mfma16(ld8u(&R[oA1tl + at]), qb, SQ2[ib]);
          }
        }
      }
      float rowv[16];
#pragma unroll
      for (int ib = 0; ib < 4; ++ib) {
        float kv[4], qv[4];
        {
          const uint2 k4 = *reinterpret_cast<const uint2*>(&R[oKC + tile_at<kL>(c, 16 * ib + 4 * g4)]);
          const uint2 q4 = *reinterpret_cast<const uint2*>(&R[oQC + tile_at<kL>(c, 16 * ib + 4 * g4)]);
          kv[0] = lo_f(k4.x); kv[1] = hi_f(k4.x); kv[2] = lo_f(k4.y); kv[3] = hi_f(k4.y);
          qv[0] = lo_f(q4.x); qv[1] = hi_f(q4.x); qv[2] = lo_f(q4.y); qv[3] = hi_f(q4.y);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = rowi(ib, r);
          dkeA[ib][r] += SK1[ib][r];
          dqA[ib][r] += SQ1[ib][r];
          dkA[ib][r] += SK2[ib][r] + SQ2[ib][r];
          rowv[4 * ib + r] = er_s[i] * kv[r] * SK1[ib][r] + p.scale * qv[r] * SQ1[ib][r] -
                             kv[r] * (SK2[ib][r] + SQ2[ib][r]);
        }
      }
      if (gated) atomicAdd(&racc[2][red_row], sum16(rowv, lane));
    }
    // Front end (combined_backward.rs:153-188) and the stores.
    float rde[16];
#pragma unroll
    for (int ib = 0; ib < 4; ++ib) {
      const uint2 k4 = *reinterpret_cast<const uint2*>(&R[oKC + tile_at<kL>(c, 16 * ib + 4 * g4)]);
      const float kv[4] = {lo_f(k4.x), hi_f(k4.x), lo_f(k4.y), hi_f(k4.y)};
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = rowi(ib, r);
        const bool ok = i < valid;
        if (ok) {
          const size_t at = row_of(i) * KS + koff + c;
          const float vq = dqA[ib][r] * p.scale, vk = dkA[ib][r] + dkeA[ib][r] * er_s[i];
          if constexpr (LASTP) {
            st_pre(p.pass, gq, p.pq, at, vq, pre_q[4 * ib + r]);
            st_pre(p.pass, gk, p.pk, at, vk, pre_k[4 * ib + r]);
          } else {
            st_sum(p.pass, gq, p.pq, at, vq);
            st_sum(p.pass, gk, p.pk, at, vk);
          }
        }
        rde[4 * ib + r] = dkeA[ib][r] * kv[r];
      }
    }
    atomicAdd(&racc[1][red_row], sum16(rde, lane));
  }
  __syncthreads();
  if (gated && wave == 0) {
    float v = racc[2][lane];
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float t = __shfl_down(v, off);
      if (lane + off < 64) v += t;
    }
    if (lane < valid) st_sum(p.rpass, p.dg, p.pg, row_of(lane), v);
  }
  if (tid < valid) {
    if constexpr (LASTP) {
      if (store_a) st_pre(p.pass, p.dwrite, p.pw, row_of(tid), racc[0][tid], pre_w);
    } else {
      if (store_a) st_sum(p.pass, p.dwrite, p.pw, row_of(tid), racc[0][tid]);
    }
    st_sum(p.rpass, p.derase, p.pe, row_of(tid), racc[1][tid]);
  }
}

}  // namespace

// Per-head gates: head_k_dim 256, or 64 with head_v_dim 64 or 128, where these
// kernels are the faster ones (measured with 64 heads of 32 chunks and with 4
// of 7, against local_bwd: 191 against 199 us and 23.4 against 26.4 at
// head_v_dim 64, 240 against 240 and 28.1 against 31.2 at 128; at 192, which
// took two passes, 421 against 279 and 47 against 37; at head_k_dim 128 the
// other is ahead from head_v_dim 64 on, 234 against 219 and 27.8 against
// 28.5, and with per-channel gates everywhere but in the smallest calls).
static bool own_shape(const Dims& d) {
  return d.dw <= 1 && d.ew == 1 && d.ww == 1 && (d.K == 256 || (d.K == 64 && d.V <= 128));
}

bool local_bwd_takes(const Dims& d) { return !own_shape(d); }

// The fp32 partial sums of the value-summed gradients across head_k_dim 256's
// launches: per (token, head) d_q, d_k (K each), d_erase, d_g and d_write,
// and past one pass of values the partial sums of dattn and dT.
size_t mfma_chunk_bwd_partials(const Dims& d) {
  if (d.K != 256) return 0;
  const size_t rows = size_t(d.B) * d.S * d.H, G = size_t(d.B) * d.N * d.H;
  return align_up(rows * (2 * d.K + d.dw + 2) * sizeof(float), 256) +
         (d.V <= 128 ? 0 : G * kNT * 16 * sizeof(float));
}

hipError_t mfma_chunk_bwd(const Dims& d, int grad_dtype, const void* dy, const void* q,
                          const void* k, const void* v, const float* erase, const float* write,
                          const float* g, const float* states, const float* ds_after, void* dq,
                          void* dk, void* dv, float* derase, float* dwrite, float* dg,
                          const MfmaTiles& tiles, float* partials, hipStream_t stream) {
  // The chunk-local kernels read the row-group layout exactly at head_k_dim 256.
  CbParams p;
  p.S = d.S;
  p.H = d.H;
  p.N = d.N;
  p.gated = d.dw > 0;
  p.scale = d.scale;
  p.q = static_cast<const uint16_t*>(q);
  p.k = static_cast<const uint16_t*>(k);
  p.v = static_cast<const uint16_t*>(v);
  p.erase = erase;
  p.write = write;
  p.g = g;
  p.dy = dy;
  p.T = tiles.T;
  p.Tlo = tiles.Tlo;
  p.Tt = tiles.Tt;
  p.Ttl = tiles.Ttl;
  p.AtT = tiles.AtT;
  p.gc = tiles.gc;
  p.states = states;
  p.ds_after = ds_after;
  p.dq = dq;
  p.dk = dk;
  p.dv = dv;
  p.derase = derase;
  p.dwrite = dwrite;
  p.dg = dg;
  const size_t G = size_t(d.B) * d.N * d.H;
  const bool f32 = grad_dtype == DN_F32;
  const int passes = d.V <= 128 ? 1 : int(d.V / 128);
  const size_t rows = size_t(d.B) * d.S * d.H;
  p.vs = int(d.V);
  p.pq = partials;
  p.pk = p.pq ? p.pq + rows * d.K : nullptr;
  p.pe = p.pk ? p.pk + rows * d.K : nullptr;
  p.pg = p.pe ? p.pe + rows : nullptr;
  p.pw = p.pg ? p.pg + rows * d.dw : nullptr;
  p.pda = nullptr;
  p.koff = p.voff = p.pass = p.rpass = 0;
  if (partials && d.V > 128) {
    const size_t head = align_up(rows * (2 * d.K + d.dw + 2) * sizeof(float), 256);
    p.pda = reinterpret_cast<float*>(reinterpret_cast<char*>(partials) + head);
  }
  ProfScope ps("dn_mfma_chunk_bwd", stream);
#define DN_CB(KD, VD, LP, EP, KA)                                                            \
  do {                                                                                       \
    if (f32)                                                                                 \
      hipLaunchKernelGGL((mfma_chunk_bwd_kernel<KD, VD, float, LP, EP, KA>), dim3(unsigned(G)), \
                         dim3(kNT), 0, stream, p);                                           \
    else                                                                                     \
      hipLaunchKernelGGL((mfma_chunk_bwd_kernel<KD, VD, bf16, LP, EP, KA>), dim3(unsigned(G)), \
                         dim3(kNT), 0, stream, p);                                           \
  } while (0)
  if (d.K == 64) {
    if (d.V == 128) DN_CB(64, 128, false, false, 64);
    else DN_CB(64, 64, false, false, 64);
    return hipGetLastError();
  }
  // Per value pass, the two key halves; the sums over key channels pass
  // through the partials across all 2·passes launches (rpass).
  const int launches = 2 * passes;
  for (int j = 0; j < launches; ++j) {
    const int i = j / 2;
    p.voff = 128 * i;
    p.koff = 128 * (j % 2);
    p.pass = passes == 1 ? 0 : i == 0 ? 1 : i + 1 == passes ? 3 : 2;
    p.rpass = j == 0 ? 1 : j + 1 == launches ? 3 : 2;
    if (p.pass == 3) DN_CB(128, 128, true, false, 256);
    else if (p.pass != 0) DN_CB(128, 128, false, true, 256);
    else DN_CB(128, 128, false, false, 256);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
#undef DN_CB
  return hipSuccess;
}

}  // namespace dn
