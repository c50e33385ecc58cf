// Launches of the four-wave-team scans (mfma_team.hpp).
#include "dn_common.hpp"
#include "mfma_team.hpp"

namespace dn {

hipError_t launch_team_scan(const MfmaParams& p, int K, bool pc, bool states, bool yb, int teams,
                            hipStream_t stream) {
  const int ntile = (p.seg == 1 ? p.V + K : p.V) / (16 * teams);  // V and K: multiples of 64
  const int seqs = p.B * (p.seg ? p.seg_p : 1) * p.H;
  const dim3 grid(unsigned(((seqs + 7) / 8) * 8 * ntile)), block(256 * teams + 256);
#define DN_T(KD, TY, C, PCV, STV, SG) \
  hipLaunchKernelGGL((team_scan_kernel<KD, TY, C, PCV, STV, SG>), grid, block, 0, stream, p)
#define DN_TY(KD, C, PCV)                                                  \
  do {                                                                     \
    if (states) DN_T(KD, float, C, PCV, true, 0);                          \
    else if (p.seg == 1) DN_T(KD, float, C, PCV, false, 1);                \
    else if (p.seg == 2) {                                                 \
      if (yb) DN_T(KD, bf16, C, PCV, false, 2);                            \
      else DN_T(KD, float, C, PCV, false, 2);                              \
    } else if (yb) DN_T(KD, bf16, C, PCV, false, 0);                       \
    else DN_T(KD, float, C, PCV, false, 0);                                \
  } while (0)
#define DN_TP(KD, C) \
  do { if (pc) DN_TY(KD, C, true); else DN_TY(KD, C, false); } while (0)
#define DN_TC(KD)                  \
  do {                             \
    if (teams == 1) DN_TP(KD, 1);  \
    else DN_TP(KD, 2);             \
  } while (0)
  if (K == 128) DN_TC(128); else DN_TC(64);
#undef DN_TC
#undef DN_TP
#undef DN_TY
#undef DN_T
  return hipGetLastError();
}

hipError_t launch_team_rev(const RevParams& p, int K, bool grad_bf16, int teams,
                           hipStream_t stream) {
  const int ntile = p.V / (16 * teams);
  const dim3 grid(unsigned(((p.B * p.H + 7) / 8) * 8 * ntile)), block(256 * teams + 256);
#define DN_R(KD, C)                                                                       \
  do {                                                                                    \
    if (grad_bf16)                                                                        \
      hipLaunchKernelGGL((team_rev_kernel<KD, bf16, C>), grid, block, 0, stream, p);      \
    else                                                                                  \
      hipLaunchKernelGGL((team_rev_kernel<KD, float, C>), grid, block, 0, stream, p);     \
  } while (0)
  if (K == 128) { if (teams == 1) DN_R(128, 1); else DN_R(128, 2); }
  else { if (teams == 1) DN_R(64, 1); else DN_R(64, 2); }
#undef DN_R
  return hipGetLastError();
}

}  // namespace dn
