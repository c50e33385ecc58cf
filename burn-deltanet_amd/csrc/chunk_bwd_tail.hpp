// The end of a chunk's backward, shared by the fp32 and the bf16 kernels: from
// the sums over the value axis (d_kc, d_qr, d_kg and the cotangents of attn
// and T) to the gradients of q, k, the erase gate and the forget gate, in fp32
// (combined_backward.rs:103-188, 376-513). In the fp32 kernels' blocks
// (chunk_f32.hpp).
#pragma once

#include "chunk_f32.hpp"

namespace dn {
namespace {

struct ChunkTail {
  const Dims& d;
  size_t row0;  // token row of the chunk's first token and its head
  int rl;       // its valid rows
  const float *erase, *g;
  float *derase, *dg;
};

// q, k and their gradients straight from and to memory, an element at a time.
template <class TQ, class TG>
struct DirectRows {
  const ChunkTail& x;
  const void *q, *k;
  void *dq, *dk;
  __device__ size_t at(int tok, int c) const {
    return (x.row0 + size_t(tok) * x.d.H) * x.d.K + c;
  }
  __device__ void load(int tok, int c, float& kv, float& qv) const {
    const size_t i = at(min(tok, x.rl - 1), c);
    kv = ld(static_cast<const TQ*>(k), i);
    qv = ld(static_cast<const TQ*>(q), i);
  }
  __device__ void store(int tok, int c, float kv, float qv) const {
    if (tok >= x.rl) return;
    st(static_cast<TG*>(dq), at(tok, c), qv);
    st(static_cast<TG*>(dk), at(tok, c), kv);
  }
};

// NW waves; wave w < KB holds key channels 16w … 16w+15 of V'·dSᵀ (dkc),
// dY·S₀ᵀ (dqr) and Z·S₀ᵀ (dkg), four token blocks each, and degl, whose sum
// over the lane groups is Σ_v dS⊙S₀ of its channel; block pairs w, w + NW, …
// of dY·V'ᵀ (dat) and dV'·Xᵀ (dtt). lds: 5·kTri floats, T in the first kTri
// (no barrier since). sG: the cumulative forget gate (per head). First
// dAkk = −tril(Tᵀ·dT·Tᵀ, −1) through LDS, then the score backward per channel
// block, its k, q and gates in registers in the accumulators' own layout.
// Rows: where q and k come from and their gradients go.
template <int KB, int NW, bool PCG, bool EK, class Rows, int NP>
__device__ void chunk_bwd_tail(const ChunkTail& x, const Rows& rows, float* lds, float (&red)[2][NW][kC],
                               const float* sG, f32x4 (&dkc)[4], f32x4 (&dqr)[4],
                               f32x4 (&dkg)[4], f32x4 (&dat)[NP], f32x4 (&dtt)[NP], float degl) {
  const Dims& d = x.d;
  const size_t row0 = x.row0;
  const int rl = x.rl;
  // Hidden from the optimiser: lane indices and addresses formed here are not
  // kept live through what comes before.
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m16 = lane & 15, g4 = lane >> 4;
  const int fo = (g4 * 16 + (m16 ^ g4)) * 4;
  int to[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) to[r] = blk(4 * g4 + r, m16);
  auto tr = [&](const float* y) { return f32x4{y[to[0]], y[to[1]], y[to[2]], y[to[3]]}; };
  const bool gated = d.dw > 0;

  // --- phase C: dAkk and the decayed score cotangents -------------------------
  float *const lT = lds, *lD = lds + kTri, *lP = lds + 2 * kTri, *rkk = lds + 3 * kTri,
        *rqk = lds + 4 * kTri;
#pragma unroll
  for (int u = 0; u < NP; ++u) {
    const int pr = wave + NW * u;
    if (pr >= 10) continue;
    const int ti = pr < 1 ? 0 : pr < 3 ? 1 : pr < 6 ? 2 : 3, tj = pr - tri_blk(ti, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * ti + 4 * g4 + r, j = 16 * tj + m16;
      const float m = PCG ? 1.f : expf(sG[i] - sG[j]);
      // (What lies on and above the diagonal reaches no result but as 0 × it.)
      lD[pr * kBlk + to[r]] = j < i ? dtt[u][r] : 0.f;
      rqk[pr * kBlk + to[r]] = j <= i ? dat[u][r] * m : 0.f;
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < NP; ++u) {
    const int pr = wave + NW * u;
    if (pr >= 10) continue;
    const int ti = pr < 1 ? 0 : pr < 3 ? 1 : pr < 6 ? 2 : 3, tj = pr - tri_blk(ti, 0);
    f32x4 acc = zero4();  // (dT·Tᵀ)(ti, tj)
    for (int bi = 0; bi <= tj; ++bi)
      acc = mm(ld4(&lD[tri_blk(ti, bi) * kBlk + fo]), ld4(&lT[tri_blk(tj, bi) * kBlk + fo]), acc);
    st4(&lP[pr * kBlk + 4 * lane], acc);
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < NP; ++u) {
    const int pr = wave + NW * u;
    if (pr >= 10) continue;
    const int ti = pr < 1 ? 0 : pr < 3 ? 1 : pr < 6 ? 2 : 3, tj = pr - tri_blk(ti, 0);
    f32x4 acc = zero4();  // (Tᵀ·dT·Tᵀ)(ti, tj)
    for (int ai = ti; ai < 4; ++ai)
      acc = mm(tr(&lT[tri_blk(ai, ti) * kBlk]), ld4(&lP[tri_blk(ai, tj) * kBlk + 4 * lane]), acc);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * ti + 4 * g4 + r, j = 16 * tj + m16;
      const float m = PCG ? 1.f : expf(sG[i] - sG[j]);
      rkk[pr * kBlk + to[r]] = j < i ? -acc[r] * m : 0.f;
    }
  }
  __syncthreads();

  // --- phase D: per key channel ------------------------------------------------
  if (wave < KB) {
    const int c = 16 * wave + m16, cc = min(c, d.K - 1);
    const bool cok = c < d.K;
    f32x4 k[4], q[4], e[4], G[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int tok = 16 * t + 4 * g4 + r;
        const size_t row = row0 + size_t(min(tok, rl - 1)) * d.H;
        const bool ok = cok && tok < rl;
        float kx, qx;
        rows.load(tok, cc, kx, qx);
        const float ex = x.erase[EK ? row * d.K + cc : row];
        const float gx = PCG ? x.g[row * d.K + cc] : 0.f;
        k[t][r] = ok ? kx : 0.f;
        q[t][r] = ok ? qx * d.scale : 0.f;
        e[t][r] = ok ? ex : 0.f;
        G[t][r] = PCG ? (ok ? gx : 0.f) : sG[tok];
      }
    float Gl;
    if constexpr (PCG) {
      // Cumulative sums down the channel: within a lane's four rows, over the
      // four lane groups of a block, then over the blocks.
      float base = 0.f;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
#pragma unroll
        for (int r = 1; r < 4; ++r) G[t][r] += G[t][r - 1];
        float sum = G[t][3];
        float up = __shfl_up(sum, 16, 64);
        if (g4 >= 1) sum += up;
        up = __shfl_up(sum, 32, 64);
        if (g4 >= 2) sum += up;
        const float ex = base + (sum - G[t][3]);
        base += __shfl(sum, 48 + m16, 64);
#pragma unroll
        for (int r = 0; r < 4; ++r) G[t][r] += ex;
      }
      Gl = base;
    } else {
      Gl = sG[63];
    }
    f32x4 dG[4];
    float carry = 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float eg = expf(G[t][r]), ec = expf(Gl - G[t][r]);
        const float dkg_ = -dkg[t][r];
        const float cr = dkc[t][r] * k[t][r] * ec;
        carry += cr;
        dG[t][r] = (dqr[t][r] * q[t][r] + dkg_ * k[t][r] * e[t][r]) * eg - cr;
        dkc[t][r] *= ec;        // → d_k
        dqr[t][r] *= eg;        // → d_q
        dkg[t][r] = dkg_ * eg;  // → d(e⊙k)
      }
    carry += degl * expf(Gl);
    carry += __shfl_xor(carry, 16, 64);
    carry += __shfl_xor(carry, 32, 64);
    if (g4 == 3) dG[3][3] += carry;

    if constexpr (!PCG) {
      // head_scores_backward (combined_backward.rs:376-416); the gate's share,
      // Σ_j of the masked score cotangents against the raw scores, is per row
      // Σ_c of the products below against ke, q and k.
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        f32x4 a1 = zero4(), a2 = zero4(), a3 = zero4();
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (j <= t) {
            a1 = mm(ld4(&rkk[tri_blk(t, j) * kBlk + fo]), k[j], a1);
            a2 = mm(ld4(&rqk[tri_blk(t, j) * kBlk + fo]), k[j], a2);
          }
          if (j >= t) {
            f32x4 ke;
#pragma unroll
            for (int r = 0; r < 4; ++r) ke[r] = k[j][r] * e[j][r];
            a3 = mm(tr(&rkk[tri_blk(j, t) * kBlk]), ke, a3);
            a3 = mm(tr(&rqk[tri_blk(j, t) * kBlk]), q[j], a3);
          }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          dkg[t][r] += a1[r];
          dqr[t][r] += a2[r];
          dkc[t][r] += a3[r];
          dG[t][r] += k[t][r] * e[t][r] * a1[r] + q[t][r] * a2[r] - k[t][r] * a3[r];
        }
      }
    } else {
      // channel_scores_backward (combined_backward.rs:421-513): row block pb
      // through its reference token 8; a clamped exponent passes no gradient.
#pragma unroll
      for (int pb = 0; pb < 4; ++pb) {
        const float Gr = __shfl(G[pb][0], 32 + m16, 64);
        f32x4 rf, rk, rq, accE = zero4(), accQ = zero4();
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          rf[r] = expf(fminf(G[pb][r] - Gr, kMaxExp));
          rk[r] = k[pb][r] * e[pb][r] * rf[r];
          rq[r] = q[pb][r] * rf[r];
        }
        float dref = 0.f;
#pragma unroll
        for (int jb = 0; jb <= pb; ++jb) {
          __builtin_amdgcn_sched_barrier(0);  // one block pair's factors at a time
          f32x4 ce, cb;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            ce[r] = expf(fminf(Gr - G[jb][r], kMaxExp));
            cb[r] = k[jb][r] * ce[r];
          }
          const float *xk = &rkk[tri_blk(pb, jb) * kBlk], *xq = &rqk[tri_blk(pb, jb) * kBlk];
          accE = mm(ld4(xk + fo), cb, accE);
          accQ = mm(ld4(xq + fo), cb, accQ);
          f32x4 dc = mm(tr(xk), rk, zero4());
          dc = mm(tr(xq), rq, dc);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            dkc[jb][r] += dc[r] * ce[r];
            const float gx = Gr - G[jb][r] >= kMaxExp ? 0.f : dc[r] * cb[r];
            dG[jb][r] -= gx;
            dref += gx;
          }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          dkg[pb][r] += accE[r] * rf[r];
          dqr[pb][r] += accQ[r] * rf[r];
          const float gx =
              G[pb][r] - Gr >= kMaxExp ? 0.f : accE[r] * rk[r] + accQ[r] * rq[r];
          dG[pb][r] += gx;
          dref -= gx;
        }
        dref += __shfl_xor(dref, 16, 64);
        dref += __shfl_xor(dref, 32, 64);
        if (g4 == 2) dG[pb][0] += dref;
        // Left to itself the compiler moves these sums into the stores at the
        // end, every term of them live until then.
#pragma unroll
        for (int t = 0; t <= pb; ++t) asm volatile("" : "+v"(dkc[t]), "+v"(dG[t]));
        asm volatile("" : "+v"(dkg[pb]), "+v"(dqr[pb]));
      }
    }
    // Front end (combined_backward.rs:153-188).
    if constexpr (PCG) {
      // d_g: the reverse of the cumulative sum.
      float base = 0.f;
#pragma unroll
      for (int t = 3; t >= 0; --t) {
#pragma unroll
        for (int r = 2; r >= 0; --r) dG[t][r] += dG[t][r + 1];
        float sum = dG[t][0];
        float dn = __shfl_down(sum, 16, 64);
        if (g4 <= 2) sum += dn;
        dn = __shfl_down(sum, 32, 64);
        if (g4 <= 1) sum += dn;
        const float ex = base + (sum - dG[t][0]);
        base += __shfl(sum, m16, 64);
#pragma unroll
        for (int r = 0; r < 4; ++r) dG[t][r] += ex;
      }
    }
    float de[16], dg[16];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int tok = 16 * t + 4 * g4 + r;
        de[4 * t + r] = dkg[t][r] * k[t][r];
        dg[4 * t + r] = dG[t][r];
        if (cok) rows.store(tok, c, dkc[t][r] + dkg[t][r] * e[t][r], dqr[t][r] * d.scale);
      }
    if constexpr (EK || PCG) {
      float* pe = EK ? x.derase : nullptr;
      float* pg = PCG ? x.dg : nullptr;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int tok = 16 * t + 4 * g4 + r;
          const size_t at = (row0 + size_t(tok) * d.H) * d.K + c;
          if (cok && tok < rl) {
            if constexpr (EK) pe[at] = de[4 * t + r];
            if constexpr (PCG)
              if (pg) pg[at] = dg[4 * t + r];
          }
        }
    }
    // Width-1 gates: sums over the key channels, per token (channels past
    // head_k_dim hold zeros).
    const int tok = 16 * (m16 >> 2) + 4 * g4 + (m16 & 3);
    if constexpr (!EK) red[0][wave][tok] = sum16(de, lane);
    if constexpr (!PCG) red[1][wave][tok] = sum16(dg, lane);
  }
  if constexpr (!EK || !PCG) {
    __syncthreads();
    if (wave == 0) {
      float se = 0.f, sg = 0.f;
#pragma unroll
      for (int w = 0; w < KB; ++w) {
        se += red[0][w][lane];
        sg += red[1][w][lane];
      }
      // d_g of a token sums the cumulative gate's cotangents from it on.
#pragma unroll
      for (int s = 1; s < 64; s *= 2) {
        const float dn = __shfl_down(sg, s, 64);
        if (lane + s < 64) sg += dn;
      }
      if (lane < rl) {
        const size_t row = row0 + size_t(lane) * d.H;
        if constexpr (!EK) x.derase[row] = se;
        if constexpr (!PCG)
          if (gated && x.dg) x.dg[row] = sg;
      }
    }
  }
}

}  // namespace
}  // namespace dn
