// The chunk scans with a team of four waves per 16 value columns (bf16 MFMA,
// fp32 state): the forward and the backward's states scan (team_scan_kernel),
// and the reverse scan (team_rev_kernel). Same inputs, workspace tiles and
// arithmetic as mfma_scan_kernel and mfma_rev_scan_kernel, whose waves each
// walk the chunks alone with all state rows of their 16 columns.
//
// A wave of a team takes one 16-token block of a chunk's products and every
// fourth 16-row block of the state; the state, X and V' cross the team through
// LDS as bf16 operand words. Four more waves only stage: a chunk's 50 KB of
// tiles take the CU's vector memory path about 800 cycles to deliver, and
// waves that issued those loads and LDS writes between their products spent
// half of a chunk on them (C = 1, cycles of 5225: 1540 issuing, 1170 staging).
//
// Bound by the chain of a chunk: three exchanges through LDS, each a write, a
// barrier and a read behind a dozen MFMAs, and LDS busy for 1350 of about 3300
// cycles. us a chunk at head_k_dim 128, one round of 16 chunks (a launch's
// start and end in them): lone waves, two to a workgroup (32 columns) 3.2,
// per-channel gates 3.4; a team (16 columns) 1.7 and 1.85, two (32 columns) 2.05
// and 2.25; the reverse scan 3.7 and 1.8, 2.2. Over longer sequences 1.5 for a
// team (24 chunks, 36 us) and 1.9 for two (256 chunks, 488).
//
// K·S_hi and K·S_lo are summed apart, as are T·X's three products, so that a
// chunk's chain is half as long; with the lone kernels' order of sums the y of
// B=4 S=16384 H=16 differs by 1.6e-4 (last bits that turn over the rounding of
// V' to bf16), and either is 3.1e-3 from float64.
// B=1 S=1531 H=16 dk 128 dv 256: forward 82 -> 44 us; B=4 S=16384 H=16
// dk=dv=128: 910 -> 659.
#pragma once

#include "mfma_scan.hpp"

namespace dn {
namespace {

// Operand tiles in LDS are 16 × 32 blocks (row, contraction index) of 64
// 16-byte words in the MFMA lanes' order: word (m, g), row m and indices
// 8g … 8g+7, at slot 16g + (m ^ x), x = g + 4kk for k-step kk of a tile whose
// global rows are read along the row: the XOR then spreads eight lanes of a
// staging write over the banks. A fragment read covers 256 bytes per 16 lanes;
// its phases pair rows {0–3, 12–15} of one g with {4–11} of the next, so x may
// differ within a phase in its two low bits only.
__device__ inline int team_slot(int m, int g, int kk) { return 16 * g + (m ^ (g + 4 * kk)); }
// The triangular tiles' blocks, whose staging lanes take four words of a row.
__device__ inline int tri_slot(int m, int g) { return 16 * g + (m ^ (2 * g)); }

// What the teams exchange is written by accumulator lanes (column n, rows
// 4g … 4g+3 of row block rb) and read as whole fragments (word (n, g') of
// k-step kk): four rows are half a word.
__device__ inline int half_word(int rb, int lane) {
  const int n = lane & 15, g = lane >> 4;
  return (((rb >> 1) * 64 + 16 * (2 * (rb & 1) + (g >> 1)) + n) << 1) + (g & 1);
}
__device__ inline uint2 pack4(const f32x4& a) {
  return make_uint2(pk_bf16(a[0], a[1]), pk_bf16(a[2], a[3]));
}
__device__ inline uint2 pack4_lo(const f32x4& a, const uint2& h) {
  return make_uint2(pk_bf16(a[0] - lo_f(h.x), a[1] - hi_f(h.x)),
                    pk_bf16(a[2] - lo_f(h.y), a[3] - hi_f(h.y)));
}

// Forward (ST = false) and states scan (ST). C teams per workgroup.
// Tiles by the phase that last reads them, each staged for the next chunk as
// soon as that phase's barrier has passed:
//   A (phase 1)       Q; per channel kg, kg lo, qg
//   B (phase 2)       T, T lo
//   D (phase 3)       K, attn; per channel Kcᵀ, attn: in two buffers
// SEG: the segmented scan's mode (MfmaParams::seg): the sequence is cut into
// seg_p segments of seg_n chunks (the last ones may be shorter, or empty).
template <int K, class TY, int C, bool PC, bool ST, int SEG = 0>
__global__ __launch_bounds__(256 * C + 256) void team_scan_kernel(MfmaParams p) {
  constexpr int KK = K / 32, RB = K / 16, NR = RB / 4;  // state row blocks per wave
  static_assert(RB % 4 == 0, "every wave owns NR row blocks");
  constexpr int kRow = 64 * K / 8, kTile = kTriSteps * 64;  // 16-byte words of a tile
  constexpr bool kY = !ST && SEG != 1;                      // y is written
  constexpr int kA = PC ? (kY ? 3 : 2) : (kY ? 1 : 0);      // K-wide tiles of class A
  constexpr int NA = kA * kRow, NB = 2 * kTile, ND = kRow + (kY ? kTile : 0);
  constexpr int PA = NA / 256, PB = NB / 256, PD = (ND + 255) / 256;
  static_assert(NA % 256 == 0 && NB % 256 == 0 && kRow % 256 == 0, "staging rounds");
  constexpr bool kPacked = !PC && tri_packed(K, ST);
  static_assert(SEG == 0 || !ST, "the states scan is not segmented");
  __shared__ uint4 tA[NA > 0 ? NA : 1], tB[NB], tD[2][ND];
  __shared__ uint4 Sx[C][2][KK * 64];       // S hi, lo
  __shared__ uint4 Xx[C][2][128];           // X hi, lo
  __shared__ uint4 Vx[C][PC ? 1 : 2][128];  // V', and e^{G_last−G}⊙V'
  __shared__ __attribute__((aligned(16))) float gt[2][PC ? 1 : 4 * kL];  // xe, w, ys, gk
  __shared__ __attribute__((aligned(16))) float ge[2][PC ? K : 1];       // e^{G_last}

  const int P = SEG ? p.seg_p : 1, VB = (SEG == 1 ? p.V + K : p.V) / 16;
  const int ntile = VB / C, BH = p.B * P * p.H;
  const int group = blockIdx.x / (8 * ntile), within = blockIdx.x % (8 * ntile);
  const int tile = within / 8, bh = group * 8 + within % 8;
  if (bh >= BH) return;
  const int seq = bh / p.H, h = bh % p.H, b = seq / P, seg = seq % P;
  // This segment's chunks n0 … n1−1; an empty one keeps to valid addresses.
  const int n0 = min(SEG ? seg * p.seg_n : 0, p.N), n1 = SEG ? min(n0 + p.seg_n, p.N) : p.N;
  const int first = min(n0, p.N - 1), last = max(n1 - 1, first);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m16 = lane & 15, g4 = lane >> 4;
  auto chunk_of = [&](int n) { return (size_t(b) * p.N + n) * p.H + h; };
  auto rows_of = [&](int n) { return (size_t(b) * p.S + size_t(n) * kL) * p.H + h; };

  if (wave >= 4 * C) {
    // --- staging waves -------------------------------------------------------
    // Global words in order (16 or 8 lanes along a row) at 32-bit offsets from
    // per-chunk bases; rows past the sequence end are clamped to its last row
    // (their gates are zero).
    const int st = tid - 256 * C;  // 0 … 255
    uint4 ra[PA > 0 ? PA : 1], rb[PB], rd[PD];
    float pg = 0.f, pl, pe = 0.f, pr = 0.f;
    auto word = [](const uint16_t* base, uint32_t elems) {
      return *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(base) + 2u * elems);
    };
    // K-wide rows of q or k: word u of the chunk's [64][K].
    auto rows_word = [&](const uint16_t* base, int u, int rl) {
      const int row = min(u / (K / 8), rl - 1), c8 = u % (K / 8);
      return word(base, uint32_t(row * p.H * K + 8 * c8));
    };
    auto wide_slot = [&](int u) {  // [64][K] word u
      const int row = u / (K / 8), c8 = u % (K / 8);
      return ((row >> 4) * KK + (c8 >> 2)) * 64 + team_slot(row & 15, c8 & 3, c8 >> 2);
    };
    auto tri_word = [&](const uint16_t* base, int u) {  // six lower blocks of a full tile
      const int s6 = u >> 6, row = 16 * tril_tb(s6) + ((u >> 2) & 15);
      return word(base, uint32_t(row * kL + 32 * tril_kk(s6) + 8 * (u & 3)));
    };
    auto tri_at = [&](int u) { return (u & ~63) + tri_slot((u >> 2) & 15, u & 3); };
    auto load_a = [&](int n, int i0, int i1) {
      const size_t cid = chunk_of(n);
#pragma unroll
      for (int i = 0; i < PA; ++i) {
        if (i < i0 || i >= i1) continue;
        const int which = 256 * i / kRow, u = 256 * i + st - which * kRow;
        if constexpr (PC) {
          const uint16_t* base = which == 0 ? p.Kg : which == 1 ? p.Kglo : p.Qg;
          ra[i] = word(base + cid * kL * K, 8u * uint32_t(u));
        } else {
          ra[i] = rows_word(p.q + rows_of(n) * K, u, min(kL, p.S - n * kL));
        }
      }
    };
    auto put_a = [&](int i0, int i1) {
#pragma unroll
      for (int i = 0; i < PA; ++i) {
        if (i < i0 || i >= i1) continue;
        const int which = 256 * i / kRow, u = 256 * i + st - which * kRow;
        tA[which * kRow + wide_slot(u)] = ra[i];
      }
    };
    auto load_b = [&](int n) {
      const size_t cid = chunk_of(n);
#pragma unroll
      for (int i = 0; i < PB; ++i) {
        const int w = 256 * i + st;
        if constexpr (kPacked) {
          rb[i] = word(p.T + cid * kTriTrio, 8u * uint32_t(w));
        } else {
          const bool lo = 256 * i + 64 * (wave - 4 * C) >= kTile;  // a wave's words are in one tile
          rb[i] = tri_word((lo ? p.Tlo : p.T) + cid * kL * kL, w - (lo ? kTile : 0));
        }
      }
    };
    auto put_b = [&] {
#pragma unroll
      for (int i = 0; i < PB; ++i) {
        tB[tri_at(256 * i + st)] = rb[i];
      }
    };
    auto load_d = [&](int n) {
      const size_t cid = chunk_of(n);
      const int rl = min(kL, p.S - n * kL);
      const size_t row0 = rows_of(n);
#pragma unroll
      for (int i = 0; i < PD; ++i) {
        const int u = 256 * i + st;
        if (256 * i < kRow) {
          rd[i] = PC ? word(p.KcT + cid * K * kL, 8u * uint32_t(u)) : rows_word(p.k + row0 * K, u, rl);
        } else {
          const int w = min(u - kRow, kTile - 1);
          rd[i] = kPacked ? word(p.T + cid * kTriTrio, 8u * uint32_t(2 * kTile + w))
                          : tri_word(p.attn + cid * kL * kL, w);
        }
      }
      if constexpr (PC) {
        pl = p.egl[cid * K + st % K];
      } else {
        // Thread st: token st mod 64's gates.
        pg = p.gc[cid * kL + lane];
        pl = p.gc[cid * kL + kL - 1];
        const size_t row = row0 + size_t(min(lane, rl - 1)) * p.H;
        pe = p.erase[row];
        pr = p.write[row];
      }
    };
    // (The values are masked here: a select beside a load waits for it.)
    auto put_d = [&](int n, int buf) {
#pragma unroll
      for (int i = 0; i < PD; ++i) {
        const int u = 256 * i + st;
        if (256 * i < kRow) {
          // Kcᵀ is [K][64]: two k-steps.
          const int at = PC ? ((u >> 7) * 2 + ((u >> 2) & 1)) * 64 +
                                  team_slot((u >> 3) & 15, u & 3, (u >> 2) & 1)
                            : wide_slot(u);
          tD[buf][at] = rd[i];
        } else if (u < ND) {
          tD[buf][kRow + tri_at(u - kRow)] = rd[i];
        }
      }
      if constexpr (PC) {
        if (st < K) ge[buf][st] = pl;
      } else {
        const float eg = __expf(pg);
        const bool ok = lane < p.S - n * kL;
        const int kind = st >> 6;
        gt[buf][st] = kind == 0   ? (ok ? pe : 0.f) * eg
                      : kind == 1 ? (ok ? pr : 0.f)
                      : kind == 2 ? p.scale * eg
                                  : __expf(pl - pg);
        if (st == 0) ge[buf][0] = __expf(pl);
      }
    };
    // Class A in two halves, so that neither phase 2 nor phase 3 waits for its
    // writes (48 KB a chunk with per-channel gates).
    constexpr int HA = (PA + 1) / 2;
    load_a(first, 0, PA);
    load_b(first);
    load_d(first);
    put_a(0, PA);
    put_b();
    put_d(first, 0);
    load_d(min(first + 1, last));
    load_a(min(first + 1, last), 0, PA);
    load_b(min(first + 1, last));
    lds_barrier();
    for (int n = n0; n < n1; ++n) {
      const int nn = min(n + 2, last);
      put_d(min(n + 1, last), (n + 1 - n0) & 1);
      load_d(nn);
      lds_barrier();
      put_a(0, HA);
      load_a(nn, 0, HA);
      lds_barrier();
      put_b();
      load_b(nn);
      put_a(HA, PA);
      load_a(nn, HA, PA);
      lds_barrier();
    }
    return;
  }

  // --- the teams ---------------------------------------------------------------
  const int team = wave >> 2, tw = wave & 3;
  // Odd teams take the token blocks in reverse: the triangular products of
  // the waves that share a SIMD then add up alike.
  const int tb = (team & 1) ? 3 - tw : tw;
  const int ct = tile * C + team;
  const int jl = 16 * ct + m16;
  // A transition column (SEG 1): column jl − V of the identity; the v it reads
  // weighs nothing.
  const bool trans = SEG == 1 && 16 * ct >= p.V;
  const int jv = trans ? m16 : jl;

  f32x4 S[NR];
  auto put_state = [&] {
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int at = half_word(tw + 4 * i, lane);
      const uint2 hi = pack4(S[i]);
      reinterpret_cast<uint2*>(Sx[team][0])[at] = hi;
      reinterpret_cast<uint2*>(Sx[team][1])[at] = pack4_lo(S[i], hi);
    }
  };
#pragma unroll
  for (int i = 0; i < NR; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * (tw + 4 * i) + 4 * g4 + r;
      S[i][r] = SEG == 1 ? (trans && row == jl - p.V ? 1.f : 0.f)
                         : p.s_in[(size_t(bh) * K + row) * p.V + jl];
    }
  const int HV = p.H * p.V;
  uint16_t vr[4];
  float wr[PC ? 4 : 1];
  auto load_v = [&](int n) {
    const int rl = min(kL, p.S - n * kL);
    const size_t row0 = rows_of(n);
    const uint16_t* vb = p.v + row0 * p.V;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      vr[r] = vb[uint32_t(min(16 * tb + 4 * g4 + r, rl - 1) * HV + jv)];
    if constexpr (PC) {
      const float* wb = p.write + row0 * p.ww + (p.ww == 1 ? 0 : jv);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        wr[r] = wb[size_t(min(16 * tb + 4 * g4 + r, rl - 1)) * (p.H * p.ww)];
    }
  };
  auto as8 = [](const uint4& x) { return __builtin_bit_cast(bf16x8, x); };
  const int at4 = half_word(tb, lane);
  const int kmax = tb >> 1;  // the last k-step of this wave's rows of T and attn

  load_v(first);
  put_state();
  lds_barrier();
  for (int n = n0; n < n1; ++n) {
    const int cur = (n - n0) & 1, nn = min(n + 1, last);
    if constexpr (ST) {
      float* dst = p.states + chunk_of(n) * K * p.V + jl;
#pragma unroll
      for (int i = 0; i < NR; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          dst[size_t(16 * (tw + 4 * i) + 4 * g4 + r) * p.V] = S[i][r];
    }
    // Phase 1: X = w⊙v − (e⊙e^G)⊙(K·S) of this wave's tokens; yᵀ = Sᵀ·Qᵀ.
    f32x4 X = {0.f, 0.f, 0.f, 0.f}, X2 = X, yt = X;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      const int at = (tb * KK + kk) * 64 + team_slot(m16, g4, kk);
      const bf16x8 sh = as8(Sx[team][0][kk * 64 + lane]), sl = as8(Sx[team][1][kk * 64 + lane]);
      const bf16x8 kf = as8(PC ? tA[at] : tD[cur][at]);
      X = mfma16(kf, sh, X);
      X2 = mfma16(kf, sl, X2);
      if constexpr (PC) X2 = mfma16(as8(tA[kRow + at]), sh, X2);
      if constexpr (kY) yt = mfma16(sh, as8(tA[(PC ? 2 * kRow : 0) + at]), yt);
    }
    float4 gk;
    if constexpr (!PC) {
      const float4 xe = *reinterpret_cast<const float4*>(&gt[cur][16 * tb + 4 * g4]);
      float4 w4 = *reinterpret_cast<const float4*>(&gt[cur][64 + 16 * tb + 4 * g4]);
      if (trans) w4 = make_float4(0.f, 0.f, 0.f, 0.f);
      const float ysc = gt[cur][128 + 16 * tb + m16];
      gk = *reinterpret_cast<const float4*>(&gt[cur][192 + 16 * tb + 4 * g4]);
      X = {w4.x * lo_f(vr[0]) - xe.x * (X[0] + X2[0]), w4.y * lo_f(vr[1]) - xe.y * (X[1] + X2[1]),
           w4.z * lo_f(vr[2]) - xe.z * (X[2] + X2[2]), w4.w * lo_f(vr[3]) - xe.w * (X[3] + X2[3])};
#pragma unroll
      for (int r = 0; r < 4; ++r) yt[r] *= ysc;
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float w = !trans && 16 * tb + 4 * g4 + r < p.S - n * kL ? wr[r] : 0.f;
        X[r] = w * lo_f(vr[r]) - (X[r] + X2[r]);
      }
    }
    {
      const uint2 hi = pack4(X);
      reinterpret_cast<uint2*>(Xx[team][0])[at4] = hi;
      reinterpret_cast<uint2*>(Xx[team][1])[at4] = pack4_lo(X, hi);
    }
    load_v(nn);
    // What the next phase reads besides X waits for no barrier.
    bf16x8 th[2], tlo[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int at = tril_step(tb, min(kk, kmax)) * 64 + tri_slot(m16, g4);
      th[kk] = as8(tB[at]);
      tlo[kk] = as8(tB[kTile + at]);
    }
    lds_barrier();
    // Phase 2: V' = T·X, hi + lo parts of both.
    f32x4 Va = {0.f, 0.f, 0.f, 0.f}, Vb = Va, Vc = Va;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      if (kk > kmax) continue;
      const bf16x8 xh = as8(Xx[team][0][kk * 64 + lane]), xl = as8(Xx[team][1][kk * 64 + lane]);
      Va = mfma16(th[kk], xh, Va);
      Vb = mfma16(tlo[kk], xh, Vb);
      Vc = mfma16(th[kk], xl, Vc);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) Va[r] += Vb[r] + Vc[r];
    reinterpret_cast<uint2*>(Vx[team][0])[at4] = pack4(Va);
    if constexpr (!PC) {
      const f32x4 sc = {gk.x * Va[0], gk.y * Va[1], gk.z * Va[2], gk.w * Va[3]};
      reinterpret_cast<uint2*>(Vx[team][PC ? 0 : 1])[at4] = pack4(sc);
    }
    // Kᵀ of state rows 16rb … and tokens 32kk …, from the K tile through the
    // LDS transpose read: lane 4j + c of each 16-lane group supplies channels
    // 4c … 4c+3 of token 8g + j (then 8g + 4 + j); lane i receives channel i.
    auto kt = [&](int rb, int kk) {
      typedef short v4s __attribute__((ext_vector_type(4)));
      typedef __attribute__((address_space(3))) v4s lds_v4s;
      const int c0 = 16 * (rb & 1) + 4 * (m16 & 3), ck = rb >> 1;
      const int t0 = 8 * (g4 & 1) + (m16 >> 2), tbk = 2 * kk + (g4 >> 1);
      const uint4* blk = &tD[cur][(tbk * KK + ck) * 64];
      const uint16_t* a = reinterpret_cast<const uint16_t*>(
                              &blk[team_slot(t0, c0 >> 3, ck)]) + (c0 & 7);
      const uint16_t* c = reinterpret_cast<const uint16_t*>(
                              &blk[team_slot(t0 + 4, c0 >> 3, ck)]) + (c0 & 7);
      const v4s x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)a);
      const v4s y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)c);
      const uint2 ux = __builtin_bit_cast(uint2, x), uy = __builtin_bit_cast(uint2, y);
      return __builtin_bit_cast(bf16x8, make_uint4(ux.x, ux.y, uy.x, uy.y));
    };
    bf16x8 uf[NR][2], af[2];
    float4 eg[NR];
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int rb = tw + 4 * i;
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
        uf[i][kk] = PC ? as8(tD[cur][(rb * 2 + kk) * 64 + team_slot(m16, g4, kk)])
                       : kt(rb, kk);
      if constexpr (PC)
        eg[i] = *reinterpret_cast<const float4*>(&ge[cur][16 * rb + 4 * g4]);
      else
        eg[i] = make_float4(ge[cur][0], ge[cur][0], ge[cur][0], ge[cur][0]);
    }
    if constexpr (kY)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
        af[kk] = as8(tD[cur][kRow + tril_step(tb, min(kk, kmax)) * 64 + tri_slot(m16, g4)]);
    lds_barrier();
    // Phase 3: S ← e^{G_last}⊙S + (e^{G_last−G}⊙K)ᵀ·V'; yᵀ += V'ᵀ·attnᵀ.
#pragma unroll
    for (int i = 0; i < NR; ++i)
      S[i] = {S[i][0] * eg[i].x, S[i][1] * eg[i].y, S[i][2] * eg[i].z, S[i][3] * eg[i].w};
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const bf16x8 vc = as8(Vx[team][PC ? 0 : 1][kk * 64 + lane]);
#pragma unroll
      for (int i = 0; i < NR; ++i) S[i] = mfma16(uf[i][kk], vc, S[i]);
    }
    if constexpr (kY)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
        if (kk <= kmax) yt = mfma16(as8(Vx[team][0][kk * 64 + lane]), af[kk], yt);
    put_state();
    if constexpr (kY) {
      TY* yb = static_cast<TY*>(p.y) + rows_of(n) * p.V;
      const int t = 16 * tb + m16;
      if (t < p.S - n * kL) {
        TY* dst = yb + uint32_t(t * HV + 16 * ct + 4 * g4);
        if constexpr (sizeof(TY) == 2)
          *reinterpret_cast<uint2*>(dst) = pack4(yt);
        else
          *reinterpret_cast<float4*>(dst) = make_float4(yt[0], yt[1], yt[2], yt[3]);
      }
    }
    lds_barrier();
  }
  float* out = p.s_out + size_t(bh) * K * p.V + jl;
  int ld = p.V;
  if constexpr (SEG == 1) {
    out = trans ? p.seg_m + size_t(bh) * K * K + (jl - p.V) : p.seg_h + size_t(bh) * K * p.V + jl;
    ld = trans ? K : p.V;
  } else if constexpr (SEG == 2) {
    if (seg != P - 1) return;  // only the last segment's end state leaves the call
    out = p.seg_final + (size_t(b) * p.H + h) * K * p.V + jl;
  }
#pragma unroll
  for (int i = 0; i < NR; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      out[size_t(16 * (tw + 4 * i) + 4 * g4 + r) * ld] = S[i][r];
}

// Reverse scan. ds_after in row-major [G][K][V]. Tiles as in the forward:
//   A (phase 1) Kc, attnᵀ;  B (phase 2) Tᵀ, Tᵀ lo;  D (phase 3) Qgᵀ, Kgᵀ, in
// two buffers. dY (phases 1 and 3) is staged by the teams.
template <int K, class TG, int C>
__global__ __launch_bounds__(256 * C + 256) void team_rev_kernel(RevParams p) {
  constexpr int KK = K / 32, RB = K / 16, NR = RB / 4;
  static_assert(RB % 4 == 0, "every wave owns NR row blocks");
  constexpr int kRow = 64 * K / 8, kTile = 6 * 64;
  constexpr int NA = kRow + kTile, NB = 2 * kTile, ND = 2 * kRow;
  constexpr int PA = (NA + 255) / 256, PB = NB / 256, PD = ND / 256;
  static_assert(NB % 256 == 0 && kRow % 256 == 0, "staging rounds");
  __shared__ uint4 tA[NA], tB[NB], tD[2][ND];
  __shared__ uint4 Sx[C][2][KK * 64];  // dS hi, lo
  __shared__ uint4 Yx[2][C][128];      // dY
  __shared__ uint4 Vx[C][2][128];      // dV' hi, lo
  __shared__ uint4 Zx[C][128];         // −Z
  __shared__ __attribute__((aligned(16))) float ge[2][K];

  const int ntile = p.V / (16 * C), BH = p.B * p.H;
  const int group = blockIdx.x / (8 * ntile), within = blockIdx.x % (8 * ntile);
  const int tile = within / 8, bh = group * 8 + within % 8;
  if (bh >= BH) return;
  const int b = bh / p.H, h = bh % p.H;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m16 = lane & 15, g4 = lane >> 4;
  auto chunk_of = [&](int n) { return (size_t(b) * p.N + n) * p.H + h; };

  if (wave >= 4 * C) {
    const int st = tid - 256 * C;
    uint4 ra[PA], rb[PB], rd[PD];
    float pe;
    auto word = [](const uint16_t* base, uint32_t elems) {
      return *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(base) + 2u * elems);
    };
    auto tri_word = [&](const uint16_t* base, int u) {  // six upper blocks of a full tile
      const int s6 = u >> 6;
      return word(base, uint32_t((16 * triu_tb(s6) + ((u >> 2) & 15)) * kL + 32 * triu_kk(s6) +
                                 8 * (u & 3)));
    };
    auto tri_at = [&](int u) { return (u & ~63) + tri_slot((u >> 2) & 15, u & 3); };
    auto load_a = [&](int n) {
      const size_t cid = chunk_of(n);
#pragma unroll
      for (int i = 0; i < PA; ++i) {
        const int u = 256 * i + st;
        ra[i] = 256 * i < kRow ? word(p.bt.Kc + cid * kL * K, 8u * uint32_t(u))
                               : tri_word(p.bt.AtT + cid * kL * kL, min(u - kRow, kTile - 1));
      }
    };
    auto put_a = [&] {
#pragma unroll
      for (int i = 0; i < PA; ++i) {
        const int u = 256 * i + st;
        if (256 * i < kRow) {
          const int row = u / (K / 8), c8 = u % (K / 8);
          tA[((row >> 4) * KK + (c8 >> 2)) * 64 + team_slot(row & 15, c8 & 3, c8 >> 2)] =
              ra[i];
        } else if (u < NA) {
          tA[kRow + tri_at(u - kRow)] = ra[i];
        }
      }
    };
    auto load_b = [&](int n) {
      const size_t cid = chunk_of(n);
#pragma unroll
      for (int i = 0; i < PB; ++i) {
        const bool lo = 256 * i + 64 * (wave - 4 * C) >= kTile;
        rb[i] = tri_word((lo ? p.bt.Ttl : p.bt.Tt) + cid * kL * kL,
                         256 * i + st - (lo ? kTile : 0));
      }
    };
    auto put_b = [&] {
#pragma unroll
      for (int i = 0; i < PB; ++i) {
        tB[tri_at(256 * i + st)] = rb[i];
      }
    };
    auto load_d = [&](int n) {
      const size_t cid = chunk_of(n);
#pragma unroll
      for (int i = 0; i < PD; ++i)
        rd[i] = word((256 * i < kRow ? p.bt.QgT : p.bt.KgT) + cid * K * kL,
                     8u * uint32_t(256 * i % kRow + st));
      pe = p.bt.egl[cid * K + st % K];
    };
    auto put_d = [&](int buf) {
#pragma unroll
      for (int i = 0; i < PD; ++i) {
        const int u = 256 * i % kRow + st;  // [K][64]
        tD[buf][(256 * i < kRow ? 0 : kRow) + ((u >> 7) * 2 + ((u >> 2) & 1)) * 64 +
                team_slot((u >> 3) & 15, u & 3, (u >> 2) & 1)] = rd[i];
      }
      if (st < K) ge[buf][st] = pe;
    };
    const int top = p.N - 1;
    load_a(top);
    load_b(top);
    load_d(top);
    put_a();
    put_b();
    put_d(0);
    load_d(max(top - 1, 0));
    load_a(max(top - 1, 0));
    load_b(max(top - 1, 0));
    lds_barrier();
    for (int it = 0; it < p.N; ++it) {
      const int nn = max(top - it - 2, 0);
      put_d((it + 1) & 1);
      load_d(nn);
      lds_barrier();
      put_a();
      load_a(nn);
      lds_barrier();
      put_b();
      load_b(nn);
      lds_barrier();
    }
    return;
  }

  const int team = wave >> 2, tw = wave & 3;
  const int tb = (team & 1) ? 3 - tw : tw;
  const int ct = tile * C + team;
  const int jl = 16 * ct + m16;
  const int at4 = half_word(tb, lane), kmin = tb >> 1;

  f32x4 S[NR];
  auto put_state = [&] {
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int at = half_word(tw + 4 * i, lane);
      const uint2 hi = pack4(S[i]);
      reinterpret_cast<uint2*>(Sx[team][0])[at] = hi;
      reinterpret_cast<uint2*>(Sx[team][1])[at] = pack4_lo(S[i], hi);
    }
  };
  if (p.dstate_final) {
#pragma unroll
    for (int i = 0; i < NR; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        S[i][r] = p.dstate_final[(size_t(bh) * K + 16 * (tw + 4 * i) + 4 * g4 + r) * p.V + jl];
  } else {
#pragma unroll
    for (int i = 0; i < NR; ++i) S[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  float py[4];
  auto load_y = [&](int n) {
    const int rl = min(kL, p.S - n * kL);
    const size_t row0 = (size_t(b) * p.S + size_t(n) * kL) * p.H + h;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      py[r] = ld(static_cast<const TG*>(p.dy),
                 (row0 + size_t(min(16 * tb + 4 * g4 + r, rl - 1)) * p.H) * p.V + jl);
  };
  auto put_y = [&](int n, int buf) {
    const int rl = p.S - n * kL - 16 * tb - 4 * g4;  // valid rows from this lane's first
    reinterpret_cast<uint2*>(Yx[buf][team])[at4] =
        pack4(f32x4{rl > 0 ? py[0] : 0.f, rl > 1 ? py[1] : 0.f, rl > 2 ? py[2] : 0.f,
                    rl > 3 ? py[3] : 0.f});
  };
  auto as8 = [](const uint4& x) { return __builtin_bit_cast(bf16x8, x); };

  load_y(p.N - 1);
  put_y(p.N - 1, 0);
  load_y(max(p.N - 2, 0));
  put_state();
  lds_barrier();
  for (int it = 0; it < p.N; ++it) {
    const int n = p.N - 1 - it, cur = it & 1;
    float* dst = p.ds_after + chunk_of(n) * K * p.V + jl;
#pragma unroll
    for (int i = 0; i < NR; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        dst[size_t(16 * (tw + 4 * i) + 4 * g4 + r) * p.V] = S[i][r];
    // Phase 1: dV' = attnᵀ·dY + Kc·dS of this wave's tokens.
    f32x4 a = {0.f, 0.f, 0.f, 0.f}, c = a, e = a;
    bf16x8 yf[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) yf[kk] = as8(Yx[cur][team][kk * 64 + lane]);
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      const bf16x8 kf = as8(tA[(tb * KK + kk) * 64 + team_slot(m16, g4, kk)]);
      a = mfma16(kf, as8(Sx[team][0][kk * 64 + lane]), a);
      c = mfma16(kf, as8(Sx[team][1][kk * 64 + lane]), c);
    }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
      if (kk >= kmin)
        e = mfma16(as8(tA[kRow + triu_step(tb, kk) * 64 + tri_slot(m16, g4)]), yf[kk],
                   e);
#pragma unroll
    for (int r = 0; r < 4; ++r) a[r] = e[r] + (a[r] + c[r]);
    {
      const uint2 hi = pack4(a);
      reinterpret_cast<uint2*>(Vx[team][0])[at4] = hi;
      reinterpret_cast<uint2*>(Vx[team][1])[at4] = pack4_lo(a, hi);
    }
    put_y(max(n - 1, 0), cur ^ 1);
    load_y(max(n - 2, 0));
    bf16x8 th[2], tlo[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int w = triu_step(tb, max(kk, kmin)) * 64 + tri_slot(m16, g4);
      th[kk] = as8(tB[w]);
      tlo[kk] = as8(tB[kTile + w]);
    }
    lds_barrier();
    // Phase 2: Z = Tᵀ·dV', hi + lo parts of both.
    f32x4 z = {0.f, 0.f, 0.f, 0.f}, z2 = z, z3 = z;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      if (kk < kmin) continue;
      const bf16x8 vh = as8(Vx[team][0][kk * 64 + lane]);
      z = mfma16(th[kk], vh, z);
      z2 = mfma16(tlo[kk], vh, z2);
      z3 = mfma16(th[kk], as8(Vx[team][1][kk * 64 + lane]), z3);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) z[r] = -(z[r] + (z2[r] + z3[r]));
    reinterpret_cast<uint2*>(Zx[team])[at4] = pack4(z);
    // dS ← e^{G_last}⊙dS + Qgᵀ·dY, which waits for no barrier.
    bf16x8 kg[NR][2];
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int rb = tw + 4 * i;
      const float4 g = *reinterpret_cast<const float4*>(&ge[cur][16 * rb + 4 * g4]);
      S[i] = {S[i][0] * g.x, S[i][1] * g.y, S[i][2] * g.z, S[i][3] * g.w};
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const int w = (rb * 2 + kk) * 64 + team_slot(m16, g4, kk);
        S[i] = mfma16(as8(tD[cur][w]), yf[kk], S[i]);
        kg[i][kk] = as8(tD[cur][kRow + w]);
      }
    }
    lds_barrier();
    // Phase 3: dS ← dS − Kgᵀ·Z.
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const bf16x8 zf = as8(Zx[team][kk * 64 + lane]);
#pragma unroll
      for (int i = 0; i < NR; ++i) S[i] = mfma16(kg[i][kk], zf, S[i]);
    }
    put_state();
    lds_barrier();
  }
#pragma unroll
  for (int i = 0; i < NR; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      p.dstate[(size_t(bh) * K + 16 * (tw + 4 * i) + 4 * g4 + r) * p.V + jl] = S[i][r];
}

}  // namespace
}  // namespace dn
