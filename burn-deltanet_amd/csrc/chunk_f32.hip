// The fp32 chunk forward: the intra kernel and the scan (chunk_f32.hpp).
#include "chunk_f32.hpp"
#include "wy_inverse.hpp"

namespace dn {
namespace {

// ---------------------------------------------------------------------------
// intra
// ---------------------------------------------------------------------------
// One workgroup of four waves per chunk-head. PCG: the forget gate is per
// key channel; EK: the erase gate is.
template <int KB, bool PCG, bool EK, class TQ>
__global__ __launch_bounds__(256) void f32_intra_kernel(FParams p) {
  constexpr bool kFold = PCG || EK;
  constexpr Lay o = lay(KB, kFold);
  constexpr int kTile = 4 * KB * kBlk;
  constexpr int kSolve = 2 * kC * (kC + 1) + 32 * 33;  // A, T and the merges' scratch
  constexpr int kQR = kTile > kSolve ? kTile : kSolve;
  __shared__ __attribute__((aligned(16))) float tK[kTile];
  // q until the scores are formed, then A, T and scratch
  __shared__ __attribute__((aligned(16))) float region[kQR];
  __shared__ __attribute__((aligned(16))) float tE[EK ? kTile : 1];   // e⊙k
  __shared__ __attribute__((aligned(16))) float tG[PCG ? kTile : 1];  // cumulative gate
  __shared__ float sE[kC], sG[kC];
  float* tQ = region;

  const Dims& d = p.d;
  const int cid = blockIdx.x;  // (b·N + n)·H + h
  const int h = cid % d.H, n = (cid / d.H) % d.N, b = cid / (d.H * d.N);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m16 = lane & 15, g4 = lane >> 4;
  const int fo = (g4 * 16 + (m16 ^ g4)) * 4;  // this lane's word of a block
  const int rl = min(kC, d.S - n * kC);       // valid rows
  const size_t row0 = (size_t(b) * d.S + size_t(n) * kC) * d.H + h;  // token row of the chunk
  float* ws = p.ws + size_t(cid) * o.per;
  const TQ* qp = static_cast<const TQ*>(p.q);
  const TQ* kp = static_cast<const TQ*>(p.k);

  // q, k: KB units of four channels per thread, loads first.
  f32x4 kr[KB], qr[KB], er[EK ? KB : 1];
#pragma unroll
  for (int i = 0; i < KB; ++i) {
    const int u = tid + 256 * i, row = u / (4 * KB), c = 4 * (u % (4 * KB));
    const int left = row < rl ? d.K - c : 0;
    const size_t at = (row0 + size_t(min(row, rl - 1)) * d.H) * d.K + min(c, d.K - 1);
    // Whole words are read unconditionally from a clamped place, and dropped.
    const bool vec = p.vec4 != 0;
    const size_t va = vec ? (row0 + size_t(min(row, rl - 1)) * d.H) * d.K + min(c, d.K - 4) : at;
    kr[i] = load4(kp, va, left, vec);
    qr[i] = load4(qp, va, left, vec);
    if constexpr (EK) er[i] = load4(p.erase, va, left, vec);
    if (vec && left <= 0) {
      kr[i] = zero4();
      qr[i] = zero4();
      if constexpr (EK) er[i] = zero4();
    }
  }
  if constexpr (!EK) {
    if (tid < kC) {
      const float e = p.erase[row0 + size_t(min(tid, rl - 1)) * d.H];
      sE[tid] = tid < rl ? e : 0.f;
    }
  }
  if constexpr (PCG) {
    for (int c = tid; c < 16 * KB; c += 256) {
      const float* gp = p.g + row0 * d.K + min(c, d.K - 1);
      const bool ok = c < d.K;
      float acc = 0.f;
#pragma unroll
      for (int t0 = 0; t0 < kC; t0 += 16) {
        float gv[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) gv[i] = gp[size_t(min(t0 + i, rl - 1)) * d.H * d.K];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int t = t0 + i;
          acc += ok && t < rl ? gv[i] : 0.f;
          tG[((t >> 4) * KB + (c >> 4)) * kBlk + blk(t & 15, c & 15)] = acc;
        }
      }
    }
  } else if (wave == 0) {
    float x = 0.f;
    if (d.dw > 0) {
      const float gv = p.g[row0 + size_t(min(lane, rl - 1)) * d.H];
      x = lane < rl ? gv : 0.f;
    }
#pragma unroll
    for (int s = 1; s < 64; s *= 2) {
      const float up = __shfl_up(x, s, 64);
      if (lane >= s) x += up;
    }
    sG[lane] = x;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < KB; ++i) {
    const int u = tid + 256 * i, row = u / (4 * KB), c4 = u % (4 * KB);
    const int at = ((row >> 4) * KB + (c4 >> 2)) * kBlk + blk(row & 15, 4 * (c4 & 3));
    f32x4 q = qr[i], ke = kr[i];
#pragma unroll
    for (int r = 0; r < 4; ++r) q[r] *= d.scale;
    if constexpr (EK)
#pragma unroll
      for (int r = 0; r < 4; ++r) ke[r] *= er[i][r];
    st4(&tK[at], kr[i]);
    st4(&tQ[at], q);
    if constexpr (EK) st4(&tE[at], ke);
    if constexpr (kFold) {
      f32x4 G, Gl;
      if constexpr (PCG) {
        G = ld4(&tG[at]);
        Gl = ld4(&tG[(3 * KB + (c4 >> 2)) * kBlk + blk(15, 4 * (c4 & 3))]);
      } else {
        G = f32x4{sG[row], sG[row], sG[row], sG[row]};
        Gl = f32x4{sG[63], sG[63], sG[63], sG[63]};
      }
      f32x4 a, uu, qq;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float eg = expf(G[r]);
        a[r] = (EK ? ke[r] : kr[i][r] * sE[row]) * eg;
        uu[r] = kr[i][r] * expf(Gl[r] - G[r]);
        qq[r] = q[r] * eg;
      }
      stw(&ws[o.a + at], a);
      stw(&ws[o.u + at], uu);
      stw(&ws[o.q + at], qq);
    } else {
      stw(&ws[o.a + at], kr[i]);
      stw(&ws[o.q + at], q);
    }
  }
  if (tid < kC) {
    const float G = PCG ? 0.f : sG[tid], Gl = PCG ? 0.f : sG[63];
    ws[o.vec + tid] = kFold ? 1.f : sE[tid] * expf(G);
    ws[o.vec + 64 + tid] = kFold ? 1.f : expf(G);
    ws[o.vec + 128 + tid] = kFold ? 1.f : expf(Gl - G);
    ws[o.vec + 192 + tid] = G;
  }
  if (tid < 16 * KB)
    ws[o.vec + 256 + tid] =
        expf(PCG ? tG[(3 * KB + (tid >> 4)) * kBlk + blk(15, tid & 15)] : sG[63]);
  __syncthreads();

  // Scores of the ten lower block pairs, dealt to the waves: Akk = (e⊙k)·kᵀ
  // and Aqk = scale·q·kᵀ, with the decay on the result (one factor per token
  // pair) or, per channel, through the row block's reference token 8
  // (decay.rs:39-60): e^{min(G[i]−G[ref],48)} on the row, and
  // e^{min(G[ref]−G[j],48)} on the column operand, formed per fragment.
  f32x4 akk[3], aqk[3];
#pragma unroll
  for (int u = 0; u < 3; ++u) {
    const int pr = wave + 4 * u;
    akk[u] = zero4();
    aqk[u] = zero4();
    if (pr >= 10) continue;
    const int ti = pr < 1 ? 0 : pr < 3 ? 1 : pr < 6 ? 2 : 3, tj = pr - tri_blk(ti, 0);
#pragma unroll
    for (int cb = 0; cb < KB; ++cb) {
      f32x4 a = ld4(&(EK ? tE : tK)[(ti * KB + cb) * kBlk + fo]);
      f32x4 q = ld4(&tQ[(ti * KB + cb) * kBlk + fo]);
      f32x4 bk = ld4(&tK[(tj * KB + cb) * kBlk + fo]);
      if constexpr (PCG) {
        const f32x4 Gi = ld4(&tG[(ti * KB + cb) * kBlk + fo]);
        const f32x4 Gj = ld4(&tG[(tj * KB + cb) * kBlk + fo]);
        const f32x4 Gr = ld4(&tG[(ti * KB + cb) * kBlk + (g4 * 16 + (8 ^ g4)) * 4]);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float rf = expf(fminf(Gi[r] - Gr[r], kMaxExp));
          a[r] *= rf;
          q[r] *= rf;
          bk[r] *= expf(fminf(Gr[r] - Gj[r], kMaxExp));
        }
      }
      akk[u] = mm(a, bk, akk[u]);
      aqk[u] = mm(q, bk, aqk[u]);
    }
  }
  __syncthreads();  // q is read: its place becomes A and T
  float(*A)[kC + 1] = reinterpret_cast<float(*)[kC + 1]>(region);
  float(*Tm)[kC + 1] = reinterpret_cast<float(*)[kC + 1]>(region + kC * (kC + 1));
  float(*Xs)[33] = reinterpret_cast<float(*)[33]>(region + 2 * kC * (kC + 1));
#pragma unroll
  for (int u = 0; u < 3; ++u) {
    const int pr = wave + 4 * u;
    if (pr >= 10) continue;
    const int ti = pr < 1 ? 0 : pr < 3 ? 1 : pr < 6 ? 2 : 3, tj = pr - tri_blk(ti, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * ti + 4 * g4 + r, j = 16 * tj + m16;
      const float m = PCG ? 1.f : expf(sG[i] - sG[j]);
      const float kk = akk[u][r] * (EK ? 1.f : sE[i]);
      A[i][j] = j < i ? kk * m : 0.f;
      ws[o.at + pr * kBlk + blk(4 * g4 + r, m16)] = j <= i ? aqk[u][r] * m : 0.f;
    }
  }
  __syncthreads();
  diag_inverse<true>(A, Tm, wave, lane);
  __syncthreads();
  merge_T(A, Tm, Xs, wave, lane, [] { __syncthreads(); });
#pragma unroll
  for (int i = 0; i < 10; ++i) {
    constexpr int ti_[10] = {0, 1, 1, 2, 2, 2, 3, 3, 3, 3}, tj_[10] = {0, 0, 1, 0, 1, 2, 0, 1, 2, 3};
    const int r = tid >> 4, c = tid & 15;
    const float x = Tm[16 * ti_[i] + r][16 * tj_[i] + c];
    ws[o.t + i * kBlk + blk(r, c)] = x;
  }
}

// ---------------------------------------------------------------------------
// scan
// ---------------------------------------------------------------------------
// A workgroup owns 16·C value columns of one (b, h) and walks the chunks; the
// four waves of a 16-column team each take one 16-token block of a chunk's
// products and every fourth 16-row block of the state. The state crosses the
// team through LDS (an accumulator tile is the next product's B operand as
// stored), so a chunk's chain is 128 MFMAs per wave at K = 128 rather than
// the 464 of one wave with all rows. Odd teams take the token blocks in
// reverse, which evens out the triangular products of the waves that share a
// SIMD. ST: the state entering each chunk, X and V' go to the workspace, no y.
//
// Four more waves only stage: they hold the next chunk's tiles in registers
// and write each where the phase that reads it has just ended. With the
// teams' waves loading and staging between two barriers of their own at each
// chunk's end, B=4 T=1000 H=8 K=V=128 took 75 us forward and 124 in reverse,
// B=1 T=512 H=4 K=V=64 28; so, 62, 97 and 20. What is left at K = 128 is half
// matrix units (4100 cycles of a wave's fp32 MFMAs a chunk), the rest LDS
// latency around the three exchanges.
template <int KB, int C, bool FOLD, bool ST, class TV, class TY>
__global__ __launch_bounds__(256 * C + 256) void f32_scan_kernel(FParams p) {
  constexpr Lay o = lay(KB, FOLD);
  constexpr int kTile = 4 * KB * kBlk;
  constexpr int kVec = 4 * kC + 16 * KB;  // xe, ys, gk, G, egl
  constexpr int NR = (KB + 3) / 4;        // state row blocks per wave
  // One buffer is enough for what one phase alone reads: a chunk's phases 1, 2
  // and 3 end at a barrier each, and the other two leave time to replace it.
  constexpr int kQ = ST ? 16 : kTile, kAt = ST ? 16 : kTri, kU = FOLD ? kTile : 16;
  __shared__ __attribute__((aligned(16))) float tA[FOLD ? 1 : 2][kTile], tU[kU], tQ[kQ], tT[kTri],
      tAt[kAt], vecs[2][kVec];
  __shared__ __attribute__((aligned(16))) float Sx[C][KB * kBlk];
  __shared__ __attribute__((aligned(16))) float Xx[C][4 * kBlk], Vx[C][4 * kBlk];

  const Dims& d = p.d;
  const int BH = d.B * d.H, VB = (d.V + 15) / 16, ntile = (VB + C - 1) / C;
  // The workgroups of one (b, h) share an XCD (ids equal mod 8): its L2 then
  // serves their common tiles.
  const int group = blockIdx.x / (8 * ntile), within = blockIdx.x % (8 * ntile);
  const int tile = within / 8, bh = group * 8 + within % 8;
  if (bh >= BH) return;
  const int b = bh / d.H, h = bh % d.H;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int team = wave >> 2, tw = wave & 3;
  const int tb = (team & 1) ? 3 - tw : tw;
  const int m16 = lane & 15, g4 = lane >> 4;
  const int fo = (g4 * 16 + (m16 ^ g4)) * 4;
  int to[4];  // the transposed read's words
#pragma unroll
  for (int r = 0; r < 4; ++r) to[r] = blk(4 * g4 + r, m16);
  auto chunk = [&](int n) { return (size_t(b) * d.N + n) * d.H + h; };
  if (__builtin_amdgcn_readfirstlane(wave) >= 4 * C) {
    // --- the staging waves ---
    const int t = tid - 256 * C, last = d.N - 1;
    auto src = [&](int n) { return p.ws + chunk(min(n, last)) * o.per; };
    Piece<kTile> a;
    Piece<kU> u;
    Piece<kQ> q;
    Piece<kTri> T;
    Piece<kAt> at;
    Piece<kVec> v;
    a.load(src(0) + o.a, t);
    T.load(src(0) + o.t, t);
    v.load(src(0) + o.vec, t);
    if constexpr (!ST) q.load(src(0) + o.q, t);
    a.store(tA[0], t);
    T.store(tT, t);
    v.store(vecs[0], t);
    if constexpr (!ST) q.store(tQ, t);
    if constexpr (FOLD) u.load(src(0) + o.u, t);
    if constexpr (!ST) at.load(src(0) + o.at, t);
    a.load(src(1) + o.a, t);
    v.load(src(1) + o.vec, t);
    if constexpr (!ST) q.load(src(1) + o.q, t);
    T.load(src(1) + o.t, t);
    __syncthreads();
    for (int n = 0; n < d.N; ++n) {
      // Beside phase 1: what phase 3 reads, and the next chunk's other halves.
      if constexpr (FOLD) {
        u.store(tU, t);
        u.load(src(n + 1) + o.u, t);
      } else {
        a.store(tA[(n + 1) & 1], t);
        a.load(src(n + 2) + o.a, t);
      }
      if constexpr (!ST) {
        at.store(tAt, t);
        at.load(src(n + 1) + o.at, t);
      }
      v.store(vecs[(n + 1) & 1], t);
      v.load(src(n + 2) + o.vec, t);
      lds_barrier();
      // Beside phase 2: the next chunk's operands of phase 1.
      if constexpr (FOLD) {
        a.store(tA[0], t);
        a.load(src(n + 2) + o.a, t);
      }
      if constexpr (!ST) {
        q.store(tQ, t);
        q.load(src(n + 2) + o.q, t);
      }
      lds_barrier();
      // Beside phase 3: the next chunk's T.
      T.store(tT, t);
      T.load(src(n + 2) + o.t, t);
      lds_barrier();
    }
    return;
  }
  const int ct = tile * C + team, col = 16 * ct + m16;
  const bool live = col < d.V;
  const int cl = min(col, d.V - 1);
  const TV* vp = static_cast<const TV*>(p.v);

  f32x4 S[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int rb = tw + 4 * i;
    S[i] = zero4();
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * rb + 4 * g4 + r;
      const float x = p.s_in[(size_t(bh) * d.K + min(row, d.K - 1)) * d.V + cl];
      S[i][r] = live && row < d.K ? x : 0.f;
    }
    if (rb < KB) st4(&Sx[team][rb * kBlk + 4 * lane], S[i]);
  }
  float vr[4], wr[4];
  auto load_v = [&](int n) {
    const int rl = min(kC, d.S - n * kC);
    const size_t row0 = (size_t(b) * d.S + size_t(n) * kC) * d.H + h;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = 16 * tb + 4 * g4 + r;
      const size_t row = row0 + size_t(min(t, rl - 1)) * d.H;
      const float x = ld(vp, row * d.V + cl);
      const float w = p.write[d.ww == 1 ? row : row * d.V + cl];
      vr[r] = x;
      wr[r] = live && t < rl ? w : 0.f;
    }
  };
  load_v(0);
  __syncthreads();
  for (int n = 0; n < d.N; ++n) {
    const int nn = min(n + 1, d.N - 1);
    const size_t cid = chunk(n);
    const float *la = tA[FOLD ? 0 : n & 1], *lu = FOLD ? tU : la, *vec = vecs[n & 1];
    if constexpr (ST) {
      if (ct < VB)
#pragma unroll
        for (int i = 0; i < NR; ++i)
          if (tw + 4 * i < KB)
            stw(p.states + ((cid * KB + tw + 4 * i) * VB + ct) * kBlk + 4 * lane, S[i]);
    }
    // K·S and Q·S of this wave's token block.
    f32x4 ks = zero4(), qs = zero4();
#pragma unroll
    for (int cb = 0; cb < KB; ++cb) {
      const f32x4 s = ld4(&Sx[team][cb * kBlk + 4 * lane]);
      const f32x4 a = ld4(&la[(tb * KB + cb) * kBlk + fo]);
      if constexpr (ST) {
        ks = mm(a, s, ks);
      } else {
        const f32x4 q = ld4(&tQ[(tb * KB + cb) * kBlk + fo]);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          ks = mfma_f32(a[r], s[r], ks);
          qs = mfma_f32(q[r], s[r], qs);
        }
      }
    }
    f32x4 X;
    {
      const f32x4 xe = ld4(&vec[16 * tb + 4 * g4]);
#pragma unroll
      for (int r = 0; r < 4; ++r) X[r] = wr[r] * vr[r] - (FOLD ? ks[r] : xe[r] * ks[r]);
    }
    load_v(nn);
    st4(&Xx[team][tb * kBlk + 4 * lane], X);
    if (ST && ct < VB) stw(p.xs + ((cid * 4 + tb) * VB + ct) * kBlk + 4 * lane, X);
    lds_barrier();
    // V' = T·X
    f32x4 Vn = zero4();
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j <= tb)
        Vn = mm(ld4(&tT[tri_blk(tb, j) * kBlk + fo]),
                ld4(&Xx[team][j * kBlk + 4 * lane]), Vn);
    st4(&Vx[team][tb * kBlk + 4 * lane], Vn);
    if (ST && ct < VB) stw(p.vn + ((cid * 4 + tb) * VB + ct) * kBlk + 4 * lane, Vn);
    lds_barrier();
    // y = ys⊙(Q·S) + attn·V' and S ← egl⊙S + Uᵀ·V'.
    if constexpr (!ST) {
      const f32x4 ys = ld4(&vec[64 + 16 * tb + 4 * g4]);
      if constexpr (!FOLD)
#pragma unroll
        for (int r = 0; r < 4; ++r) qs[r] *= ys[r];
    }
#pragma unroll
    for (int i = 0; i < NR; ++i)
      if (tw + 4 * i < KB) {
        const f32x4 e = ld4(&vec[256 + 16 * (tw + 4 * i) + 4 * g4]);
#pragma unroll
        for (int r = 0; r < 4; ++r) S[i][r] *= e[r];
      }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f32x4 vj = ld4(&Vx[team][j * kBlk + 4 * lane]);
      if constexpr (!ST)
        if (j <= tb) qs = mm(ld4(&tAt[tri_blk(tb, j) * kBlk + fo]), vj, qs);
      f32x4 vk = vj;
      if constexpr (!FOLD) {
        const f32x4 gk = ld4(&vec[128 + 16 * j + 4 * g4]);
#pragma unroll
        for (int r = 0; r < 4; ++r) vk[r] *= gk[r];
      }
#pragma unroll
      for (int i = 0; i < NR; ++i)
        if (tw + 4 * i < KB) {
          const float* ub = &lu[(j * KB + tw + 4 * i) * kBlk];
#pragma unroll
          for (int r = 0; r < 4; ++r) S[i] = mfma_f32(ub[to[r]], vk[r], S[i]);
        }
    }
#pragma unroll
    for (int i = 0; i < NR; ++i)
      if (tw + 4 * i < KB) st4(&Sx[team][(tw + 4 * i) * kBlk + 4 * lane], S[i]);
    if constexpr (!ST) {
      const int rl = d.S - n * kC;
      const size_t row0 = (size_t(b) * d.S + size_t(n) * kC) * d.H + h;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = 16 * tb + 4 * g4 + r;
        if (live && t < rl)
          st(static_cast<TY*>(p.y), (row0 + size_t(t) * d.H) * d.V + col, qs[r]);
      }
    }
    lds_barrier();
  }
#pragma unroll
  for (int i = 0; i < NR; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * (tw + 4 * i) + 4 * g4 + r;
      if (live && row < d.K) p.s_out[(size_t(bh) * d.K + row) * d.V + col] = S[i][r];
    }
}

}  // namespace

hipError_t f32_intra(const FParams& p, int qkv_dtype, hipStream_t stream) {
  const Dims& d = p.d;
  const bool pcg = d.dw > 1, ek = d.ew > 1, b16 = qkv_dtype == DN_BF16;
  const dim3 grid(unsigned(chunk_heads(d))), block(256);
  ProfScope ps("dn_f32_intra", stream);
#define DN_I(KB, PC, EK)                                                                         \
  do {                                                                                           \
    if (b16)                                                                                     \
      hipLaunchKernelGGL((f32_intra_kernel<KB, PC, EK, bf16>), grid, block, 0, stream, p);       \
    else                                                                                         \
      hipLaunchKernelGGL((f32_intra_kernel<KB, PC, EK, float>), grid, block, 0, stream, p);      \
  } while (0)
#define DN_IG(KB)                                                             \
  do {                                                                        \
    if (pcg) { if (ek) DN_I(KB, true, true); else DN_I(KB, true, false); }    \
    else { if (ek) DN_I(KB, false, true); else DN_I(KB, false, false); }      \
  } while (0)
  switch (key_blocks(d.K)) {
    case 2: DN_IG(2); break;
    case 4: DN_IG(4); break;
    case 6: DN_IG(6); break;
    default: DN_IG(8); break;
  }
#undef DN_IG
#undef DN_I
  return hipGetLastError();
}

hipError_t f32_scan(const FParams& p, int qkv_dtype, int y_dtype, bool states,
                    hipStream_t stream) {
  const Dims& d = p.d;
  const int teams = scan_teams(d);
  const dim3 grid(scan_blocks(d, teams)), block(256 * teams + 256);
  const bool b16 = qkv_dtype == DN_BF16, y16 = y_dtype == DN_BF16, fold = folds(d);
  ProfScope ps(states ? "dn_f32_scan_states" : "dn_f32_scan", stream);
#define DN_S(KB, C, F, ST, TV, TY) \
  hipLaunchKernelGGL((f32_scan_kernel<KB, C, F, ST, TV, TY>), grid, block, 0, stream, p)
#define DN_ST(KB, C, F)                                               \
  do {                                                                \
    if (states) {                                                     \
      if (b16) DN_S(KB, C, F, true, bf16, float);                     \
      else DN_S(KB, C, F, true, float, float);                        \
    } else if (b16) {                                                 \
      if (y16) DN_S(KB, C, F, false, bf16, bf16);                     \
      else DN_S(KB, C, F, false, bf16, float);                        \
    } else {                                                          \
      if (y16) DN_S(KB, C, F, false, float, bf16);                    \
      else DN_S(KB, C, F, false, float, float);                       \
    }                                                                 \
  } while (0)
#define DN_SK(KB)                                                              \
  do {                                                                         \
    if (teams == 1) { if (fold) DN_ST(KB, 1, true); else DN_ST(KB, 1, false); } \
    else { if (fold) DN_ST(KB, 2, true); else DN_ST(KB, 2, false); }           \
  } while (0)
  switch (key_blocks(d.K)) {
    case 2: DN_SK(2); break;
    case 4: DN_SK(4); break;
    case 6: DN_SK(6); break;
    default: DN_SK(8); break;
  }
#undef DN_SK
#undef DN_ST
#undef DN_S
  return hipGetLastError();
}

bool f32_supported(const Dims& d) {
  return d.K <= 128 && d.L == kC && (d.ew == 1 || d.ew == d.K) && (d.ww == 1 || d.ww == d.V) &&
         (d.dw <= 1 || d.dw == d.K);
}

size_t f32_fwd_workspace(const Dims& d) {
  return bytes_of(chunk_heads(d) * size_t(lay(key_blocks(d.K), folds(d)).per));
}

hipError_t f32_fwd(const Dims& d, int qkv_dtype, int y_dtype, const void* q, const void* k,
                   const void* v, const float* erase, const float* write, const float* g,
                   const float* state_in, void* y, float* state_out, void* ws,
                   hipStream_t stream) {
  FParams p = f32_params(d, qkv_dtype, q, k, v, erase, write, g, state_in, ws);
  p.y = y;
  p.s_out = state_out;
  hipError_t e = f32_intra(p, qkv_dtype, stream);
  return e != hipSuccess ? e : f32_scan(p, qkv_dtype, y_dtype, false, stream);
}

}  // namespace dn
