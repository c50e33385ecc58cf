// The fp32 chunk backward (chunk_f32.hpp): the reverse scan and the
// chunk-local gradients. combined_backward.rs:72-513 with the identities of
// the bf16 kernels: dT = dV'·Xᵀ and d_kg = −(Tᵀ·dV')·S₀ᵀ.
#include "chunk_bwd_tail.hpp"

namespace dn {
namespace {

// ---------------------------------------------------------------------------
// reverse scan
// ---------------------------------------------------------------------------
// The forward scan's split (a team of four waves per 16 value columns, one
// token block each, dS's row blocks dealt to them, everything exchanged
// through LDS in accumulator order), walking the chunks backwards:
//   dV' = attnᵀ·dY + kc·dS,  Z = Tᵀ·dV',  dS ← egl⊙dS + qgᵀ·dY − kgᵀ·Z.
// Leaves dS (leaving each chunk), dV' and Z in the workspace.
template <int KB, int C, bool FOLD, class TG>
__global__ __launch_bounds__(256 * C + 256) void f32_rev_scan_kernel(FParams p) {
  constexpr Lay o = lay(KB, FOLD);
  constexpr int kTile = 4 * KB * kBlk;
  constexpr int kVec = 4 * kC + 16 * KB;
  constexpr int NR = (KB + 3) / 4;
  constexpr int kU = FOLD ? kTile : 16;
  __shared__ __attribute__((aligned(16))) float tA[FOLD ? 1 : 2][kTile], tU[kU], tQ[kTile], tT[kTri],
      tAt[kTri], vecs[2][kVec];
  __shared__ __attribute__((aligned(16))) float Sx[C][KB * kBlk];
  // dY and dV' change places from chunk to chunk: dV' is dead when the next
  // chunk's dY arrives.
  __shared__ __attribute__((aligned(16))) float YVx[2][C][4 * kBlk], Zx[C][4 * kBlk];

  const Dims& d = p.d;
  const int BH = d.B * d.H, VB = (d.V + 15) / 16, ntile = (VB + C - 1) / C;
  const int group = blockIdx.x / (8 * ntile), within = blockIdx.x % (8 * ntile);
  const int tile = within / 8, bh = group * 8 + within % 8;
  if (bh >= BH) return;
  const int b = bh / d.H, h = bh % d.H;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int team = wave >> 2, tw = wave & 3;
  const int tb = (team & 1) ? 3 - tw : tw;
  const int m16 = lane & 15, g4 = lane >> 4;
  const int fo = (g4 * 16 + (m16 ^ g4)) * 4;
  int to[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) to[r] = blk(4 * g4 + r, m16);
  auto chunk = [&](int n) { return (size_t(b) * d.N + n) * d.H + h; };
  if (__builtin_amdgcn_readfirstlane(wave) >= 4 * C) {
    // --- the staging waves (the forward scan's, for this walk's phases) ---
    const int t = tid - 256 * C;
    auto src = [&](int n) { return p.ws + chunk(max(n, 0)) * o.per; };
    const int N1 = d.N - 1;
    Piece<kTile> a, q;
    Piece<kU> u;
    Piece<kTri> T, at;
    Piece<kVec> v;
    at.load(src(N1) + o.at, t);
    T.load(src(N1) + o.t, t);
    v.load(src(N1) + o.vec, t);
    a.load(src(N1) + o.a, t);
    if constexpr (FOLD) u.load(src(N1) + o.u, t);
    at.store(tAt, t);
    T.store(tT, t);
    v.store(vecs[N1 & 1], t);
    if constexpr (FOLD) {
      u.store(tU, t);
    } else {
      a.store(tA[N1 & 1], t);
      a.load(src(N1 - 1) + o.a, t);
    }
    q.load(src(N1) + o.q, t);
    v.load(src(N1 - 1) + o.vec, t);
    at.load(src(N1 - 1) + o.at, t);
    if constexpr (FOLD) u.load(src(N1 - 1) + o.u, t);
    T.load(src(N1 - 1) + o.t, t);
    __syncthreads();
    for (int n = N1; n >= 0; --n) {
      // Beside phase 1: phase 3's operands.
      q.store(tQ, t);
      q.load(src(n - 1) + o.q, t);
      if constexpr (FOLD) {
        a.store(tA[0], t);
        a.load(src(n - 1) + o.a, t);
      }
      v.store(vecs[(n + 1) & 1], t);
      v.load(src(n - 2) + o.vec, t);
      lds_barrier();
      // Beside phase 2: the next chunk's operands of phase 1.
      at.store(tAt, t);
      at.load(src(n - 2) + o.at, t);
      if constexpr (FOLD) {
        u.store(tU, t);
        u.load(src(n - 2) + o.u, t);
      } else {
        a.store(tA[(n + 1) & 1], t);
        a.load(src(n - 2) + o.a, t);
      }
      lds_barrier();
      // Beside phase 3: the next chunk's T.
      T.store(tT, t);
      T.load(src(n - 2) + o.t, t);
      lds_barrier();
    }
    return;
  }
  const int ct = tile * C + team, col = 16 * ct + m16;
  const bool live = col < d.V;
  const int cl = min(col, d.V - 1);
  const TG* dyp = static_cast<const TG*>(p.dy);

  f32x4 S[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int rb = tw + 4 * i;
    S[i] = zero4();
    if (p.ds_final) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * rb + 4 * g4 + r;
        const float x = p.ds_final[(size_t(bh) * d.K + min(row, d.K - 1)) * d.V + cl];
        S[i][r] = live && row < d.K ? x : 0.f;
      }
    }
    if (rb < KB) st4(&Sx[team][rb * kBlk + 4 * lane], S[i]);
  }
  f32x4 py;
  auto fetch = [&](int n) {
    const int rl = min(kC, d.S - n * kC);
    const size_t row0 = (size_t(b) * d.S + size_t(n) * kC) * d.H + h;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = 16 * tb + 4 * g4 + r;
      const float x = ld(dyp, (row0 + size_t(min(t, rl - 1)) * d.H) * d.V + cl);
      py[r] = live && t < rl ? x : 0.f;
    }
  };
  fetch(d.N - 1);
  st4(&YVx[(d.N - 1) & 1][team][tb * kBlk + 4 * lane], py);
  __syncthreads();
  for (int n = d.N - 1; n >= 0; --n) {
    const size_t cid = chunk(n);
    const float *la = tA[FOLD ? 0 : n & 1], *lu = FOLD ? tU : la, *vec = vecs[n & 1];
    const float* Yx = YVx[n & 1][team];
    float* Vx = YVx[(n + 1) & 1][team];
    fetch(max(n - 1, 0));
    if (ct < VB)
#pragma unroll
      for (int i = 0; i < NR; ++i)
        if (tw + 4 * i < KB)
          stw(p.ds_after + ((cid * KB + tw + 4 * i) * VB + ct) * kBlk + 4 * lane, S[i]);
    f32x4 dv = zero4(), av = zero4();
#pragma unroll
    for (int cb = 0; cb < KB; ++cb)
      dv = mm(ld4(&lu[(tb * KB + cb) * kBlk + fo]), ld4(&Sx[team][cb * kBlk + 4 * lane]),
              dv);
    // A transposed block's operand: its four words in column order.
    auto tr = [&](const float* x) { return f32x4{x[to[0]], x[to[1]], x[to[2]], x[to[3]]}; };
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j >= tb)
        av = mm(tr(&tAt[tri_blk(j, tb) * kBlk]), ld4(&Yx[j * kBlk + 4 * lane]), av);
    {
      const f32x4 gk = ld4(&vec[128 + 16 * tb + 4 * g4]);
#pragma unroll
      for (int r = 0; r < 4; ++r) dv[r] = av[r] + (FOLD ? dv[r] : gk[r] * dv[r]);
    }
    st4(&Vx[tb * kBlk + 4 * lane], dv);
    if (ct < VB) stw(p.dvn + ((cid * 4 + tb) * VB + ct) * kBlk + 4 * lane, dv);
    lds_barrier();
    f32x4 z = zero4();
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j >= tb)
        z = mm(tr(&tT[tri_blk(j, tb) * kBlk]), ld4(&Vx[j * kBlk + 4 * lane]), z);
    st4(&Zx[team][tb * kBlk + 4 * lane], z);
    if (ct < VB) stw(p.z + ((cid * 4 + tb) * VB + ct) * kBlk + 4 * lane, z);
    lds_barrier();
#pragma unroll
    for (int i = 0; i < NR; ++i)
      if (tw + 4 * i < KB) {
        const f32x4 e = ld4(&vec[256 + 16 * (tw + 4 * i) + 4 * g4]);
#pragma unroll
        for (int r = 0; r < 4; ++r) S[i][r] *= e[r];
      }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f32x4 y = ld4(&Yx[j * kBlk + 4 * lane]), zj = ld4(&Zx[team][j * kBlk + 4 * lane]);
      const f32x4 xe = ld4(&vec[16 * j + 4 * g4]), ys = ld4(&vec[64 + 16 * j + 4 * g4]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        y[r] *= FOLD ? 1.f : ys[r];
        zj[r] *= FOLD ? -1.f : -xe[r];
      }
#pragma unroll
      for (int i = 0; i < NR; ++i)
        if (tw + 4 * i < KB) {
          const int at = (j * KB + tw + 4 * i) * kBlk;
          S[i] = mm(tr(&tQ[at]), y, S[i]);
          S[i] = mm(tr(&la[at]), zj, S[i]);
        }
    }
#pragma unroll
    for (int i = 0; i < NR; ++i)
      if (tw + 4 * i < KB) st4(&Sx[team][(tw + 4 * i) * kBlk + 4 * lane], S[i]);
    st4(&Vx[tb * kBlk + 4 * lane], py);  // the next chunk's dY
    lds_barrier();
  }
#pragma unroll
  for (int i = 0; i < NR; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * (tw + 4 * i) + 4 * g4 + r;
      if (live && row < d.K) p.dstate[(size_t(bh) * d.K + row) * d.V + col] = S[i][r];
    }
}

// ---------------------------------------------------------------------------
// chunk-local gradients
// ---------------------------------------------------------------------------
// One workgroup per chunk-head. Phase B walks the value axis 16 columns at a
// time, double-buffered through LDS (one barrier a step): wave w owns key
// channels 16w … 16w+15 and sums V'·dSᵀ, dY·S₀ᵀ and Z·S₀ᵀ for all 64 tokens,
// 48 accumulator registers; the ten lower blocks of dY·V'ᵀ and dV'·Xᵀ are
// dealt over the waves. Then the score backward (chunk_bwd_tail).
template <int KB, bool PCG, bool EK, class TQ, class TG>
__global__ __launch_bounds__(64 * (KB < 4 ? 4 : KB)) void f32_chunk_bwd_kernel(FParams p) {
  constexpr bool kFold = PCG || EK;
  constexpr Lay o = lay(KB, kFold);
  constexpr int NW = KB < 4 ? 4 : KB;
  constexpr int kTiles = 20 + 2 * KB;  // X, V', dV', Z, dY (4 blocks each), S₀, dS
  constexpr int kPlain = 12 + 2 * KB;  // all but dY and Z
  constexpr int NPT = (kPlain + NW - 1) / NW;
  constexpr int NP = (10 + NW - 1) / NW;
  constexpr int kStage = 2 * kTiles * kBlk;
  constexpr int kLds = kStage > 5 * kTri ? kStage : 5 * kTri;
  __shared__ __attribute__((aligned(16))) float lds[kLds];
  __shared__ float sG[kC], red[2][NW][kC];

  const Dims& d = p.d;
  const int cid = blockIdx.x;
  const int h = cid % d.H, n = (cid / d.H) % d.N, b = cid / (d.H * d.N);
  const int VB = (d.V + 15) / 16;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m16 = lane & 15, g4 = lane >> 4;
  const int fo = (g4 * 16 + (m16 ^ g4)) * 4;
  int to[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) to[r] = blk(4 * g4 + r, m16);
  const int rl = min(kC, d.S - n * kC);
  const size_t row0 = (size_t(b) * d.S + size_t(n) * kC) * d.H + h;
  const float* ws = p.ws + size_t(cid) * o.per;
  const TQ* vp = static_cast<const TQ*>(p.v);
  const TG* dyp = static_cast<const TG*>(p.dy);

  // --- phase B ---------------------------------------------------------------
  // Waves 0 … 3 load token block `wave` of dY and of Z, with v and the write
  // gate beside Z; the other blocks are dealt over all waves, one scalar
  // address each.
  f32x4 pf[NPT], py, pz;
  float vz[4], wz[4], dwr[4] = {0.f, 0.f, 0.f, 0.f};
  const float* src[NPT];
#pragma unroll
  for (int i = 0; i < NPT; ++i) {
    const int t = min((wave + 4) % NW + NW * i, kPlain - 1);
    if (t < 12) {
      src[i] = (t < 4 ? p.xs : t < 8 ? p.vn : p.dvn) + (size_t(cid) * 4 + (t & 3)) * VB * kBlk;
    } else {
      const int sb = t - 12;
      src[i] = (sb < KB ? p.states : p.ds_after) +
               (size_t(cid) * KB + (sb < KB ? sb : sb - KB)) * VB * kBlk;
    }
  }
  const float* zsrc = p.z + (size_t(cid) * 4 + (wave & 3)) * VB * kBlk;
  size_t at4[4];  // this lane's rows of dY, v and d_v (waves 0 … 3)
#pragma unroll
  for (int r = 0; r < 4; ++r)
    at4[r] = (row0 + size_t(min(16 * (wave & 3) + 4 * g4 + r, rl - 1)) * d.H) * d.V;
  auto load = [&](int vt) {
#pragma unroll
    for (int i = 0; i < NPT; ++i) pf[i] = ldw(src[i] + size_t(vt) * kBlk + 4 * lane);
    if (wave < 4) {
      const int col = 16 * vt + m16, cl = min(col, d.V - 1);
      pz = ldw(zsrc + size_t(vt) * kBlk + 4 * lane);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        py[r] = ld(dyp, at4[r] + cl);
        vz[r] = ld(vp, at4[r] + cl);
        if (d.ww != 1) wz[r] = p.write[at4[r] + cl];
      }
    }
  };
  if (wave < 4 && d.ww == 1)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      wz[r] = p.write[row0 + size_t(min(16 * wave + 4 * g4 + r, rl - 1)) * d.H];
  // To LDS with rows and columns swapped (a lane's four values are rows), and
  // from Z the gradients of v and the write gate.
  auto stage = [&](float* buf, int vt) {
#pragma unroll
    for (int i = 0; i < NPT; ++i) {
      const int t = (wave + 4) % NW + NW * i;
      if (t >= kPlain) continue;
      // X, V', dV' at blocks 0 … 11; Z and dY at 12 … 19; S₀ and dS after.
      float* dst = buf + (t < 12 ? t : t + 8) * kBlk;
#pragma unroll
      for (int r = 0; r < 4; ++r) dst[to[r]] = pf[i][r];
    }
    if (wave < 4) {
      const int col = 16 * vt + m16;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool ok = 16 * wave + 4 * g4 + r < rl && col < d.V;
        buf[(12 + wave) * kBlk + to[r]] = pz[r];
        buf[(16 + wave) * kBlk + to[r]] = ok ? py[r] : 0.f;
        const float dw = pz[r] * vz[r];
        if (ok) {
          st(static_cast<TG*>(p.dv), at4[r] + col, pz[r] * wz[r]);
          if (d.ww != 1) p.dwrite[at4[r] + col] = dw;
        }
        dwr[r] += ok ? dw : 0.f;
      }
    }
  };
  f32x4 dkc[4], dqr[4], dkg[4], dat[NP], dtt[NP];
  float degl = 0.f;
#pragma unroll
  for (int t = 0; t < 4; ++t) dkc[t] = dqr[t] = dkg[t] = zero4();
#pragma unroll
  for (int u = 0; u < NP; ++u) dat[u] = dtt[u] = zero4();
  load(0);
  for (int vt = 0; vt < VB; ++vt) {
    float* buf = lds + (vt & 1) * kTiles * kBlk;
    stage(buf, vt);
    lds_barrier();
    if (vt + 1 < VB) load(vt + 1);
    if (wave < KB) {
      const f32x4 s0 = ld4(&buf[(20 + wave) * kBlk + fo]);
      const f32x4 ds = ld4(&buf[(20 + KB + wave) * kBlk + fo]);
#pragma unroll
      for (int r = 0; r < 4; ++r) degl += s0[r] * ds[r];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        dkc[t] = mm(ld4(&buf[(4 + t) * kBlk + fo]), ds, dkc[t]);
        dqr[t] = mm(ld4(&buf[(16 + t) * kBlk + fo]), s0, dqr[t]);
        dkg[t] = mm(ld4(&buf[(12 + t) * kBlk + fo]), s0, dkg[t]);
      }
    }
#pragma unroll
    for (int u = 0; u < NP; ++u) {
      const int pr = wave + NW * u;
      if (pr >= 10) continue;
      const int ti = pr < 1 ? 0 : pr < 3 ? 1 : pr < 6 ? 2 : 3, tj = pr - tri_blk(ti, 0);
      dat[u] = mm(ld4(&buf[(16 + ti) * kBlk + fo]), ld4(&buf[(4 + tj) * kBlk + fo]), dat[u]);
      dtt[u] = mm(ld4(&buf[(8 + ti) * kBlk + fo]), ld4(&buf[tj * kBlk + fo]), dtt[u]);
    }
  }
  if (d.ww == 1 && wave < 4) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float x = dwr[r];
#pragma unroll
      for (int s = 1; s < 16; s *= 2) x += __shfl_xor(x, s, 64);
      const int tok = 16 * wave + 4 * g4 + r;
      if (m16 == 0 && tok < rl) p.dwrite[row0 + size_t(tok) * d.H] = x;
    }
  }
  if (!PCG && tid < kC) sG[tid] = ws[o.vec + 192 + tid];
  __syncthreads();

  float *lT = lds;
  for (int i = tid; i < kTri / 4; i += 64 * NW) st4(&lT[4 * i], ldw(ws + o.t + 4 * i));
  const ChunkTail x{d, row0, rl, p.erase, p.g, p.derase, p.dg};
  chunk_bwd_tail<KB, NW, PCG, EK>(x, DirectRows<TQ, TG>{x, p.q, p.k, p.dq, p.dk}, lds, red, sG,
                                  dkc, dqr, dkg, dat, dtt, degl);
}

hipError_t launch_rev(const FParams& p, int grad_dtype, hipStream_t stream) {
  const Dims& d = p.d;
  const int teams = scan_teams(d);
  const dim3 grid(scan_blocks(d, teams)), block(256 * teams + 256);
  const bool g16 = grad_dtype == DN_BF16, fold = folds(d);
  ProfScope ps("dn_f32_rev_scan", stream);
#define DN_R(KB, C, F)                                                                       \
  do {                                                                                       \
    if (g16)                                                                                 \
      hipLaunchKernelGGL((f32_rev_scan_kernel<KB, C, F, bf16>), grid, block, 0, stream, p);  \
    else                                                                                     \
      hipLaunchKernelGGL((f32_rev_scan_kernel<KB, C, F, float>), grid, block, 0, stream, p); \
  } while (0)
#define DN_RK(KB)                                                           \
  do {                                                                      \
    if (teams == 1) { if (fold) DN_R(KB, 1, true); else DN_R(KB, 1, false); } \
    else { if (fold) DN_R(KB, 2, true); else DN_R(KB, 2, false); }          \
  } while (0)
  switch (key_blocks(d.K)) {
    case 2: DN_RK(2); break;
    case 4: DN_RK(4); break;
    case 6: DN_RK(6); break;
    default: DN_RK(8); break;
  }
#undef DN_RK
#undef DN_R
  return hipGetLastError();
}

hipError_t launch_chunk_bwd(const FParams& p, int qkv_dtype, int grad_dtype, hipStream_t stream) {
  const Dims& d = p.d;
  const bool pcg = d.dw > 1, ek = d.ew > 1;
  const bool b16 = qkv_dtype == DN_BF16, g16 = grad_dtype == DN_BF16;
  const int kb = key_blocks(d.K);
  const dim3 grid(unsigned(chunk_heads(d))), block(64 * (kb < 4 ? 4 : kb));
  ProfScope ps("dn_f32_chunk_bwd", stream);
#define DN_C(KB, PC, EK, TQ, TG) \
  hipLaunchKernelGGL((f32_chunk_bwd_kernel<KB, PC, EK, TQ, TG>), grid, block, 0, stream, p)
#define DN_CT(KB, PC, EK)                                                                \
  do {                                                                                   \
    if (b16) { if (g16) DN_C(KB, PC, EK, bf16, bf16); else DN_C(KB, PC, EK, bf16, float); }  \
    else { if (g16) DN_C(KB, PC, EK, float, bf16); else DN_C(KB, PC, EK, float, float); }    \
  } while (0)
#define DN_CG(KB)                                                             \
  do {                                                                        \
    if (pcg) { if (ek) DN_CT(KB, true, true); else DN_CT(KB, true, false); }  \
    else { if (ek) DN_CT(KB, false, true); else DN_CT(KB, false, false); }    \
  } while (0)
  switch (kb) {
    case 2: DN_CG(2); break;
    case 4: DN_CG(4); break;
    case 6: DN_CG(6); break;
    default: DN_CG(8); break;
  }
#undef DN_CG
#undef DN_CT
#undef DN_C
  return hipGetLastError();
}

// The backward's buffers after the tiles.
struct BwdSizes {
  size_t state, rows;  // bytes of one [G][KB][VB] and one [G][4][VB] block array
};
BwdSizes bwd_sizes(const Dims& d) {
  const size_t blocks = chunk_heads(d) * size_t((d.V + 15) / 16) * kBlk;
  return {bytes_of(blocks * key_blocks(d.K)), bytes_of(blocks * 4)};
}

}  // namespace

size_t f32_bwd_workspace(const Dims& d) {
  const BwdSizes s = bwd_sizes(d);
  return f32_fwd_workspace(d) + 2 * s.state + 4 * s.rows +
         bytes_of(size_t(d.B) * d.H * d.K * d.V);  // the recompute's final state (unused)
}

hipError_t f32_bwd(const Dims& d, int qkv_dtype, int grad_dtype, const void* dy,
                   const float* dstate_final, const void* q, const void* k, const void* v,
                   const float* erase, const float* write, const float* g, const float* state_in,
                   void* dq, void* dk, void* dv, float* derase, float* dwrite, float* dg,
                   float* dstate, void* ws, hipStream_t stream) {
  FParams p = f32_params(d, qkv_dtype, q, k, v, erase, write, g, state_in, ws);
  const BwdSizes s = bwd_sizes(d);
  char* base = static_cast<char*>(ws) + f32_fwd_workspace(d);
  auto take = [&](size_t bytes) {
    float* at = reinterpret_cast<float*>(base);
    base += bytes;
    return at;
  };
  p.states = take(s.state);
  p.ds_after = take(s.state);
  p.xs = take(s.rows);
  p.vn = take(s.rows);
  p.dvn = take(s.rows);
  p.z = take(s.rows);
  p.s_out = take(0);
  p.dy = dy;
  p.ds_final = dstate_final;
  p.dstate = dstate;
  p.dq = dq;
  p.dk = dk;
  p.dv = dv;
  p.derase = derase;
  p.dwrite = dwrite;
  p.dg = dg;
  hipError_t e = f32_intra(p, qkv_dtype, stream);
  if (e != hipSuccess) return e;
  // The two scans need nothing from each other: the reverse one runs on the
  // calling stream's second stream.
  e = side_by_side(
      stream, [&](hipStream_t side) { return launch_rev(p, grad_dtype, side); },
      [&] { return f32_scan(p, qkv_dtype, DN_F32, true, stream); });
  if (e != hipSuccess) return e;
  return launch_chunk_bwd(p, qkv_dtype, grad_dtype, stream);
}

}  // namespace dn
