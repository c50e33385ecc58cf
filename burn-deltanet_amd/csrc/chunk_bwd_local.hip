// The chunk-local gradients of the bf16 MFMA backward at head_k_dim 64 and 128
// (combined_backward.rs:103-188, :240-319, :376-513), one workgroup per
// chunk-head, given the state S₀ entering the chunk and the cotangent dS of
// the state leaving it (fp32) and the intra kernel's tiles. With X = w⊙V −
// kg·S₀, V' = T·X, dV' = attnᵀ·dY + kc·dS and Z = Tᵀ·dV' (= dVw):
//
//   per 32 value columns, all in LDS as bf16 hi and lo parts:
//     1  X and dV' (contractions over the keys), a wave per 16 × 16 tile
//     2  V' and Z; d_v = w⊙Z, d_write from Z⊙v
//     3  the sums over the value axis: wave w owns key channels 16w … 16w+15
//        of V'·dSᵀ, dY·S₀ᵀ and Z·S₀ᵀ for all 64 tokens; the lower blocks of
//        dY·V'ᵀ and dV'·Xᵀ are dealt over the waves
//   then chunk_bwd_tail, in fp32.
//
// Every product runs on v_mfma_f32_16x16x32_bf16 with fp32 operands as hi + lo
// parts (three MFMAs; two when one side is an exact bf16 input). S₀ and dS are
// read once, split once on their way to LDS, and serve the contractions over
// keys (through the LDS transpose read) and over values alike; the next
// columns' loads are in flight while these are worked on.
//
// One value column block after another in one launch, so the score backward
// runs once whatever head_v_dim is and nothing goes through memory between
// passes of 128 columns (partial sums of d_q, d_k, dattn and dT did, with
// fp32 atomics between). Bound by LDS and by issue: at 135 KB of LDS one
// workgroup owns its CU, two waves a SIMD, and of 98000 cycles at head_v_dim
// 256 the eight steps' products take 36000 and their waits on loads 26000,
// the fp32 tail 32000. q and k pass through LDS tiles in the tail, and their
// gradients leave by whole rows: two-byte accesses of a lane's own tokens
// took 30000 cycles there. All of the kernel at B=8 T=2048 H=16
// dk=128 dv=256, per-head gates: 1190 us in two passes, 715 here; at B=2
// T=16384 H=16 dk=dv=128, per-channel gates: 1600 and 1341.
#include "chunk_bwd_tail.hpp"

namespace dn {
namespace {

// Accesses to the caller's gates and gradients, which are aligned to their
// elements and no further, and to v, which is to 4 bytes (q, k and dO are to 16).
typedef float f4_any __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u2_any __attribute__((ext_vector_type(2), aligned(2)));
typedef uint32_t u4_any __attribute__((ext_vector_type(4), aligned(2)));

struct LocalParams {
  Dims d;
  const uint16_t *q, *k, *v;
  const float *erase, *write, *g;
  const void* dy;
  MfmaTiles t;
  const float *states, *ds_after;  // [G][K][V]
  void *dq, *dk, *dv;
  float *derase, *dwrite, *dg;
};

// Word (row m, indices 8g … 8g+7) of a 16 × 32 block. `rows` tiles are read
// mostly as fragments, whose phases pair two g's rows; `cols` tiles (S₀, dS)
// mostly through the transpose read, which takes two g's words of four rows.
__device__ inline int rows_slot(int m, int g) { return 16 * g + (m ^ (2 * g)); }
__device__ inline int cols_slot(int m, int g) { return 16 * g + (m ^ (4 * g)); }

// q and k of the chunk in LDS tiles ([64][K] of 16 × 32 blocks), which their
// gradients replace where they are bf16; fp32 ones go to memory.
template <int K, class TG>
struct TileRows {
  uint16_t *kt, *qt;
  DirectRows<bf16, TG> direct;
  __device__ static int at(int tok, int c) {
    return (((tok >> 4) * (K / 32) + (c >> 5)) * 64 + rows_slot(tok & 15, (c & 31) >> 3)) * 8 +
           (c & 7);
  }
  __device__ void load(int tok, int c, float& kv, float& qv) const {
    kv = bf16_to_f32(kt[at(tok, c)]);
    qv = bf16_to_f32(qt[at(tok, c)]);
  }
  __device__ void store(int tok, int c, float kv, float qv) const {
    if constexpr (sizeof(TG) == 2) {
      kt[at(tok, c)] = f32_to_bf16_dev(kv);
      qt[at(tok, c)] = f32_to_bf16_dev(qv);
    } else {
      direct.store(tok, c, kv, qv);
    }
  }
};

template <int K, bool PCG, bool EK, class TG>
__global__ __launch_bounds__(4 * K) void local_bwd_kernel(LocalParams p) {
  constexpr int KK = K / 32, RB = K / 16, NW = RB, NT = 64 * NW;
  constexpr int TPW = 8 / NW;             // 16 × 16 tiles of 32 columns per wave
  constexpr int NP = (10 + NW - 1) / NW;  // lower block pairs per wave
  constexpr bool kYlo = sizeof(TG) == 4;  // dY as hi + lo parts
  constexpr int kWide = 4 * KK * 64;      // words of a [64][K] tile
  constexpr int kTri6 = 6 * 64;
  constexpr int oX = 4 * RB * 64, oY = oX + 8 * 256, kSteps = oY + (kYlo ? 2 : 1) * 256;
  // Then the tail's tiles take the region's place, and q's (per-channel gates:
  // it takes kg lo's).
  constexpr int oQ = 5 * kTri / 4, kTail = oQ + (PCG ? 0 : kWide),
                kRegion = kSteps > kTail ? kSteps : kTail;
  __shared__ uint4 tK[kWide], tKl[PCG ? kWide : 1], tKc[PCG ? kWide : 1];
  __shared__ uint4 tT[2][kTri6], tU[2][kTri6], tA[kTri6];  // T, Tᵀ (hi, lo), attnᵀ
  // S₀ hi, lo, dS hi, lo; X, V', dV', Z hi, lo; dY
  __shared__ uint4 region[kRegion];
  __shared__ float red[2][NW][kC], sG[kC], sdw[2][kC], sdeg[K];

  const Dims& d = p.d;
  const int cid = blockIdx.x;
  const int h = cid % d.H, n = (cid / d.H) % d.N, b = cid / (d.H * d.N);
  const int V = d.V, rl = min(kC, d.S - n * kC);
  const size_t row0 = (size_t(b) * d.S + size_t(n) * kC) * d.H + h;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m16 = lane & 15, g4 = lane >> 4;
  const TG* dyp = static_cast<const TG*>(p.dy);
  auto as8 = [](const uint4& x) { return __builtin_bit_cast(bf16x8, x); };

  // --- the values' loads, one step of 32 columns ahead -------------------------
  const int c = tid >> 2, part = tid & 3;  // S₀ and dS: row c, columns 8·part …
  const float* s0p = p.states + (size_t(cid) * K + c) * V + 8 * part;
  const float* dsp = p.ds_after + (size_t(cid) * K + c) * V + 8 * part;
  const bool ythread = tid < 256;
  const TG* yp = dyp + (row0 + size_t(min(c & 63, rl - 1)) * d.H) * V + 8 * part;
  const int tb = wave & 3, tok = 16 * tb + m16;  // this wave's token block
  const bool tok_ok = tok < rl;
  const size_t trow = row0 + size_t(min(tok, rl - 1)) * d.H;
  f32x4 ps[2], pd[2];
  uint4 py;
  f32x4 pyf[kYlo ? 2 : 1];
  u2_any pv[TPW];
  f32x4 pw[PCG ? TPW : 1];
  auto load = [&](int v0) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      ps[i] = ld4(s0p + v0 + 4 * i);
      pd[i] = ld4(dsp + v0 + 4 * i);
    }
    if (ythread) {
      if constexpr (kYlo) {
#pragma unroll
        for (int i = 0; i < 2; ++i) pyf[i] = ld4(reinterpret_cast<const float*>(yp) + v0 + 4 * i);
      } else {
        py = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(yp) + v0);
      }
    }
#pragma unroll
    for (int u = 0; u < TPW; ++u) {
      const int v = v0 + 16 * ((wave + NW * u) >> 2) + 4 * g4;
      pv[u] = *reinterpret_cast<const u2_any*>(p.v + trow * V + v);
      if constexpr (PCG)
        if (d.ww != 1) pw[u] = *reinterpret_cast<const f4_any*>(p.write + trow * V + v);
    }
  };
  // With the last columns worked on: q, and k where its tile holds kg.
  constexpr int NKQ = kWide / NT;
  uint4 wq[NKQ], wkk[PCG ? NKQ : 1];
  auto load_kq = [&] {
#pragma unroll
    for (int i = 0; i < NKQ; ++i) {
      const int u = tid + NT * i, row = u / (K / 8), c8 = u % (K / 8);
      const size_t at = (row0 + size_t(min(row, rl - 1)) * d.H) * K + 8 * c8;
      wq[i] = *reinterpret_cast<const uint4*>(p.q + at);
      if constexpr (PCG) wkk[i] = *reinterpret_cast<const uint4*>(p.k + at);
    }
  };
  load(0);

  // --- the chunk's tiles ----------------------------------------------------------
  {
    auto word = [](const uint16_t* x, size_t at) { return *reinterpret_cast<const uint4*>(x + at); };
    uint4 wk[kWide / NT], wl[PCG ? kWide / NT : 1], wc[PCG ? kWide / NT : 1];
#pragma unroll
    for (int i = 0; i < kWide / NT; ++i) {
      const int u = tid + NT * i, row = u / (K / 8), c8 = u % (K / 8);
      if constexpr (PCG) {
        const size_t at = (size_t(cid) * kC + row) * K + 8 * c8;
        wk[i] = word(p.t.Kg, at);
        wl[i] = word(p.t.Kglo, at);
        wc[i] = word(p.t.Kc, at);
      } else {
        wk[i] = word(p.k, (row0 + size_t(min(row, rl - 1)) * d.H) * K + 8 * c8);
      }
    }
    constexpr int NS = (5 * kTri6 + NT - 1) / NT;
    uint4 wt[NS];
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      const int u = min(tid + NT * i, 5 * kTri6 - 1), which = u / kTri6, w = u % kTri6, st = w >> 6;
      const bool up = which >= 2;  // T, T lo below; Tᵀ, Tᵀ lo, attnᵀ above the diagonal
      const int rb = up ? triu_tb(st) : tril_tb(st);
      const int kk = up ? triu_kk(st) : tril_kk(st);
      const uint16_t* x = which == 0   ? p.t.T
                          : which == 1 ? p.t.Tlo
                          : which == 2 ? p.t.Tt
                          : which == 3 ? p.t.Ttl
                                       : p.t.AtT;
      wt[i] = word(x, size_t(cid) * kC * kC + (16 * rb + ((w >> 2) & 15)) * kC + 32 * kk + 8 * (w & 3));
    }
#pragma unroll
    for (int i = 0; i < kWide / NT; ++i) {
      const int u = tid + NT * i, row = u / (K / 8), c8 = u % (K / 8);
      const int at = ((row >> 4) * KK + (c8 >> 2)) * 64 + rows_slot(row & 15, c8 & 3);
      tK[at] = wk[i];
      if constexpr (PCG) {
        tKl[at] = wl[i];
        tKc[at] = wc[i];
      }
    }
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      const int u = tid + NT * i;
      if (u < 5 * kTri6) {
        const int which = u / kTri6, w = u % kTri6;
        const int at = (w & ~63) + rows_slot((w >> 2) & 15, w & 3);
        (which < 2 ? tT[which] : which < 4 ? tU[which - 2] : tA)[at] = wt[i];
      }
    }
  }
  float xe = 1.f, gk = 1.f, wt1 = 0.f;  // this lane's token: e·e^G, e^{G_last−G}, w
  if constexpr (!PCG) {
    const float G = p.t.gc[size_t(cid) * kC + tok], Gl = p.t.gc[size_t(cid) * kC + kC - 1];
    const float e = p.erase[trow];
    xe = tok_ok ? e * expf(G) : 0.f;
    gk = tok_ok ? expf(Gl - G) : 0.f;
    if (tid < kC) sG[tid] = p.t.gc[size_t(cid) * kC + tid];
  }
  if (!PCG || d.ww == 1) wt1 = tok_ok ? p.write[trow] : 0.f;

  // --- the value axis ---------------------------------------------------------------
  uint4 *S0 = region, *Sd = region + 2 * RB * 64;          // hi, then lo
  uint4 *Xt = region + oX, *Vt = Xt + 512, *Dt = Vt + 512, *Zt = Dt + 512, *Yt = region + oY;
  // Fragment of rows 16rb …: word (m16, g4) of a block.
  auto frag = [&](const uint4* t, int rb) { return as8(t[rb * 64 + rows_slot(m16, g4)]); };
  // Columns 16ct … as rows, contraction over rows 32kk …: lane 4j + c of each
  // 16-lane group supplies columns 4c … of row 8g + j (then 8g + 4 + j).
  auto trans = [&](const uint4* t, int kk, int ct, bool cols) {
    typedef short v4s __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) v4s lds_v4s;
    const int g = 2 * ct + ((m16 & 3) >> 1), r = 8 * (g4 & 1) + (m16 >> 2);
    const uint4* blk = t + (2 * kk + (g4 >> 1)) * 64;
    auto at = [&](int row) {
      return (lds_v4s*)(reinterpret_cast<const uint16_t*>(
                            &blk[cols ? cols_slot(row, g) : rows_slot(row, g)]) + 4 * (m16 & 1));
    };
    const v4s x = __builtin_amdgcn_ds_read_tr16_b64_v4i16(at(r));
    const v4s y = __builtin_amdgcn_ds_read_tr16_b64_v4i16(at(r + 4));
    const uint2 ux = __builtin_bit_cast(uint2, x), uy = __builtin_bit_cast(uint2, y);
    return __builtin_bit_cast(bf16x8, make_uint4(ux.x, ux.y, uy.x, uy.y));
  };
  // A tile's lane values (columns 4g4 … of token m16) as hi and lo half words.
  auto put = [&](uint4* t, int ct, const f32x4& x) {
    const int at = 2 * (tb * 64 + rows_slot(m16, 2 * ct + (g4 >> 1))) + (g4 & 1);
    const uint2 hi = make_uint2(pk_bf16(x[0], x[1]), pk_bf16(x[2], x[3]));
    reinterpret_cast<uint2*>(t)[at] = hi;
    reinterpret_cast<uint2*>(t + 256)[at] =
        make_uint2(pk_bf16(x[0] - lo_f(hi.x), x[1] - hi_f(hi.x)),
                   pk_bf16(x[2] - lo_f(hi.y), x[3] - hi_f(hi.y)));
  };
  f32x4 dkc[4], dqr[4], dkg[4], dat[NP], dtt[NP];
#pragma unroll
  for (int t = 0; t < 4; ++t) dkc[t] = dqr[t] = dkg[t] = zero4();
#pragma unroll
  for (int u = 0; u < NP; ++u) dat[u] = dtt[u] = zero4();
  float deg = 0.f, dwr[TPW];
#pragma unroll
  for (int u = 0; u < TPW; ++u) dwr[u] = 0.f;

  for (int v0 = 0; v0 < V; v0 += 32) {
    if (v0 > 0) lds_barrier();  // the last columns' tiles have been read
    {
      const int at = (c >> 4) * 64 + cols_slot(c & 15, part);
      float s8[8], d8[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        s8[i] = ps[i >> 2][i & 3];
        d8[i] = pd[i >> 2][i & 3];
        deg += s8[i] * d8[i];
      }
      uint4 hi, lo;
      split8(s8, hi, lo);
      S0[at] = hi;
      S0[RB * 64 + at] = lo;
      split8(d8, hi, lo);
      Sd[at] = hi;
      Sd[RB * 64 + at] = lo;
      if (ythread) {
        const bool ok = c < rl;
        const int ya = (c >> 4) * 64 + rows_slot(c & 15, part);
        if constexpr (kYlo) {
          float y8[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) y8[i] = ok ? pyf[i >> 2][i & 3] : 0.f;
          split8(y8, hi, lo);
          Yt[ya] = hi;
          Yt[256 + ya] = lo;
        } else {
          Yt[ya] = ok ? py : make_uint4(0u, 0u, 0u, 0u);
        }
      }
    }
    uint2 v4[TPW];
    f32x4 w4[TPW];
#pragma unroll
    for (int u = 0; u < TPW; ++u) {
      v4[u] = make_uint2(pv[u].x, pv[u].y);
      w4[u] = f32x4{wt1, wt1, wt1, wt1};
      if constexpr (PCG)
        if (d.ww != 1) w4[u] = tok_ok ? pw[u] : zero4();
    }
    lds_barrier();
    if (v0 + 32 < V)
      load(v0 + 32);
    else
      load_kq();
    // 1: Xᵀ and dV'ᵀ, rows the columns, columns the tokens.
#pragma unroll
    for (int u = 0; u < TPW; ++u) {
      const int ct = (wave + NW * u) >> 2;
      f32x4 xa = zero4(), xb = zero4(), da = zero4(), db = zero4(), ya = zero4();
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        // Fragments of two k-steps at a time (all of them read ahead spill).
        if (kk % 2 == 0) __builtin_amdgcn_sched_barrier(0);
        const int at = (tb * KK + kk) * 64 + rows_slot(m16, g4);
        const bf16x8 kf = as8(tK[at]);
        const bf16x8 sh = trans(S0, kk, ct, true), sl = trans(S0 + RB * 64, kk, ct, true);
        xa = mfma16(sh, kf, xa);
        xb = mfma16(sl, kf, xb);
        if constexpr (PCG) xb = mfma16(sh, as8(tKl[at]), xb);
        const bf16x8 kc = PCG ? as8(tKc[at]) : kf;
        da = mfma16(trans(Sd, kk, ct, true), kc, da);
        db = mfma16(trans(Sd + RB * 64, kk, ct, true), kc, db);
      }
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        if (kk < (tb >> 1)) continue;
        const bf16x8 af = frag(tA, triu_step(tb, kk));
        ya = mfma16(trans(Yt, kk, ct, false), af, ya);
        if constexpr (kYlo) ya = mfma16(trans(Yt + 256, kk, ct, false), af, ya);
      }
      const float vv[4] = {lo_f(v4[u].x), hi_f(v4[u].x), lo_f(v4[u].y), hi_f(v4[u].y)};
      f32x4 X, D;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float ks = xa[r] + xb[r], kd = da[r] + db[r];
        X[r] = w4[u][r] * vv[r] - (PCG ? ks : xe * ks);
        D[r] = ya[r] + (PCG ? kd : gk * kd);
      }
      put(Xt, ct, X);
      put(Dt, ct, D);
    }
    lds_barrier();
    // 2: V'ᵀ = Xᵀ·Tᵀ and Zᵀ = dV'ᵀ·T.
#pragma unroll
    for (int u = 0; u < TPW; ++u) {
      const int ct = (wave + NW * u) >> 2;
      f32x4 va = zero4(), vb = zero4(), za = zero4(), zb = zero4();
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        if (kk <= (tb >> 1)) {
          const bf16x8 th = frag(tT[0], tril_step(tb, kk)), tl = frag(tT[1], tril_step(tb, kk));
          const bf16x8 xh = trans(Xt, kk, ct, false);
          va = mfma16(xh, th, va);
          vb = mfma16(xh, tl, vb);
          vb = mfma16(trans(Xt + 256, kk, ct, false), th, vb);
        }
        if (kk >= (tb >> 1)) {
          const bf16x8 uh = frag(tU[0], triu_step(tb, kk)), ul = frag(tU[1], triu_step(tb, kk));
          const bf16x8 dh = trans(Dt, kk, ct, false);
          za = mfma16(dh, uh, za);
          zb = mfma16(dh, ul, zb);
          zb = mfma16(trans(Dt + 256, kk, ct, false), uh, zb);
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        va[r] += vb[r];
        za[r] += zb[r];
      }
      put(Vt, ct, va);
      put(Zt, ct, za);
      const float vv[4] = {lo_f(v4[u].x), hi_f(v4[u].x), lo_f(v4[u].y), hi_f(v4[u].y)};
      f32x4 dw;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        dw[r] = za[r] * vv[r];
        dwr[u] += dw[r];
        za[r] *= w4[u][r];
      }
      if (tok_ok) {
        const size_t at = trow * V + v0 + 16 * ct + 4 * g4;
        if constexpr (kYlo)
          *reinterpret_cast<f4_any*>(static_cast<float*>(p.dv) + at) = za;
        else
          *reinterpret_cast<u2_any*>(static_cast<uint16_t*>(p.dv) + at) =
              u2_any{pk_bf16(za[0], za[1]), pk_bf16(za[2], za[3])};
        if constexpr (PCG)
          if (d.ww != 1) *reinterpret_cast<f4_any*>(p.dwrite + at) = dw;
      }
    }
    lds_barrier();
    // 3: the sums over these columns.
    {
      const int at = wave * 64 + cols_slot(m16, g4);
      const bf16x8 sh = as8(S0[at]), sl = as8(S0[RB * 64 + at]);
      const bf16x8 dh = as8(Sd[at]), dl = as8(Sd[RB * 64 + at]);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (t % 2 == 0) __builtin_amdgcn_sched_barrier(0);
        const bf16x8 vh = frag(Vt, t), zh = frag(Zt, t), yh = frag(Yt, t);
        dkc[t] = mfma16(vh, dh, dkc[t]);
        dqr[t] = mfma16(yh, sh, dqr[t]);
        dkg[t] = mfma16(zh, sh, dkg[t]);
        dkc[t] = mfma16(vh, dl, dkc[t]);
        dqr[t] = mfma16(yh, sl, dqr[t]);
        dkg[t] = mfma16(zh, sl, dkg[t]);
        dkc[t] = mfma16(frag(Vt + 256, t), dh, dkc[t]);
        if constexpr (kYlo) dqr[t] = mfma16(frag(Yt + 256, t), sh, dqr[t]);
        dkg[t] = mfma16(frag(Zt + 256, t), sh, dkg[t]);
      }
    }
#pragma unroll
    for (int u = 0; u < NP; ++u) {
      const int pr = wave + NW * u;
      if (pr >= 10) continue;
      const int ti = pr < 1 ? 0 : pr < 3 ? 1 : pr < 6 ? 2 : 3, tj = pr - tri_blk(ti, 0);
      const bf16x8 yh = frag(Yt, ti), vh = frag(Vt, tj), dh = frag(Dt, ti), xh = frag(Xt, tj);
      dat[u] = mfma16(yh, vh, dat[u]);
      dat[u] = mfma16(yh, frag(Vt + 256, tj), dat[u]);
      if constexpr (kYlo) dat[u] = mfma16(frag(Yt + 256, ti), vh, dat[u]);
      dtt[u] = mfma16(dh, xh, dtt[u]);
      dtt[u] = mfma16(dh, frag(Xt + 256, tj), dtt[u]);
      dtt[u] = mfma16(frag(Dt + 256, ti), xh, dtt[u]);
    }
  }
  // Σ_v dS⊙S₀ per channel, and a width-1 write gate's gradient per token.
  deg += __shfl_xor(deg, 1, 64);
  deg += __shfl_xor(deg, 2, 64);
  if (part == 0) sdeg[c] = deg;
  if (d.ww == 1) {
    float x = dwr[0];
    if constexpr (TPW > 1) x += dwr[TPW - 1];
    x += __shfl_xor(x, 16, 64);
    x += __shfl_xor(x, 32, 64);
    if (g4 == 0) sdw[wave >> 2][tok] = x;
  }
  __syncthreads();
  if (d.ww == 1 && tid < rl)
    p.dwrite[row0 + size_t(tid) * d.H] = sdw[0][tid] + (NW > 4 ? sdw[1][tid] : 0.f);
  uint4* tQ = PCG ? tKl : region + oQ;
  auto wide_at = [&](int u) {
    const int row = u / (K / 8), c8 = u % (K / 8);
    return ((row >> 4) * KK + (c8 >> 2)) * 64 + rows_slot(row & 15, c8 & 3);
  };
#pragma unroll
  for (int i = 0; i < NKQ; ++i) {
    tQ[wide_at(tid + NT * i)] = wq[i];
    if constexpr (PCG) tK[wide_at(tid + NT * i)] = wkk[i];
  }
  // T in fp32 in the tail's blocks.
  float* lds = reinterpret_cast<float*>(region);
  for (int w = tid; w < kTri6; w += NT) {
    const int st = w >> 6, m = (w >> 2) & 15, g = w & 3, ti = tril_tb(st);
    const int tj = 2 * tril_kk(st) + (g >> 1);
    if (tj > ti) continue;
    const int at = (w & ~63) + rows_slot(m, g);
    float hi[8], lo[8];
    unpack8(tT[0][at], hi);
    unpack8(tT[1][at], lo);
    float* dst = lds + tri_blk(ti, tj) * kBlk;
    st4(dst + blk(m, 8 * (g & 1)), f32x4{hi[0] + lo[0], hi[1] + lo[1], hi[2] + lo[2], hi[3] + lo[3]});
    st4(dst + blk(m, 8 * (g & 1) + 4),
        f32x4{hi[4] + lo[4], hi[5] + lo[5], hi[6] + lo[6], hi[7] + lo[7]});
  }
  const float degl = g4 == 0 ? sdeg[16 * wave + m16] : 0.f;
  const ChunkTail x{d, row0, rl, p.erase, p.g, p.derase, p.dg};
  const TileRows<K, TG> rows{reinterpret_cast<uint16_t*>(tK), reinterpret_cast<uint16_t*>(tQ),
                             DirectRows<bf16, TG>{x, p.q, p.k, p.dq, p.dk}};
  chunk_bwd_tail<RB, NW, PCG, EK>(x, rows, lds, red, sG, dkc, dqr, dkg, dat, dtt, degl);
  if constexpr (!kYlo) {
    // d_q and d_k by whole rows.
    auto store = [](void* out, size_t at, const uint4& x) {
      *reinterpret_cast<u4_any*>(static_cast<uint16_t*>(out) + at) = u4_any{x.x, x.y, x.z, x.w};
    };
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NKQ; ++i) {
      const int u = tid + NT * i, row = u / (K / 8), c8 = u % (K / 8);
      if (row < rl) {
        const size_t at = (row0 + size_t(row) * d.H) * K + 8 * c8;
        store(p.dq, at, tQ[wide_at(u)]);
        store(p.dk, at, tK[wide_at(u)]);
      }
    }
  }
}

}  // namespace

hipError_t local_bwd(const Dims& d, int grad_dtype, const void* dy, const void* q, const void* k,
                     const void* v, const float* erase, const float* write, const float* g,
                     const float* states, const float* ds_after, void* dq, void* dk, void* dv,
                     float* derase, float* dwrite, float* dg, const MfmaTiles& tiles,
                     hipStream_t stream) {
  LocalParams p{d,
                static_cast<const uint16_t*>(q),
                static_cast<const uint16_t*>(k),
                static_cast<const uint16_t*>(v),
                erase,
                write,
                g,
                dy,
                tiles,
                states,
                ds_after,
                dq,
                dk,
                dv,
                derase,
                dwrite,
                dg};
  const bool pc = d.dw == d.K && d.K > 1, f32 = grad_dtype == DN_F32;
  const dim3 grid(unsigned(chunk_heads(d))), block(unsigned(4 * d.K));
  ProfScope ps("dn_mfma_chunk_bwd", stream);
#define DN_L(KD, PC, EK)                                                                  \
  do {                                                                                    \
    if (f32)                                                                              \
      hipLaunchKernelGGL((local_bwd_kernel<KD, PC, EK, float>), grid, block, 0, stream, p); \
    else                                                                                  \
      hipLaunchKernelGGL((local_bwd_kernel<KD, PC, EK, bf16>), grid, block, 0, stream, p);  \
  } while (0)
#define DN_LG(KD)                                                         \
  do {                                                                    \
    if (!pc) DN_L(KD, false, false);                                      \
    else if (d.ew > 1) DN_L(KD, true, true);                              \
    else DN_L(KD, true, false);                                           \
  } while (0)
  if (d.K == 128) DN_LG(128); else DN_LG(64);
#undef DN_LG
#undef DN_L
  return hipGetLastError();
}

}  // namespace dn
