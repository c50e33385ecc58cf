"""The scans' workgroup width (scan_waves) at head counts either side of where
a wider workgroup saves a round: the bf16 MFMA forward and backward against
the fp32 kernels, at the bf16 path's bar."""

import numpy as np
import pytest
import torch

from conftest import random_raw, rel_err
from gpu_util import announce, np_of, pkg, to_gpu

pytestmark = pytest.mark.gpu

MFMA, GENERIC = pkg.abi.DN_ALGO_MFMA, pkg.abi.DN_ALGO_GENERIC


# H heads of V columns on 256 CUs: forward widths 2 | 4 | 8 with H·V/32, H·V/64
# and H·V/128 workgroups; the backward's pair of scans reaches each at half.
@pytest.mark.parametrize("H,K,V,channel", [(32, 128, 256, False), (33, 128, 256, False),
                                           (65, 128, 256, False), (17, 128, 256, False),
                                           (65, 64, 64, False), (33, 128, 256, True),
                                           (66, 64, 128, True)])
def test_scan_width(rng, H, K, V, channel):
    announce(f"scan width H {H} K {K} V {V} channel {channel}")
    args = to_gpu(random_raw(rng, 1, 70, H, K, V, channel=channel), torch.bfloat16)
    dy = torch.tensor(rng.standard_normal((1, 70, H, V)), device=args[0].device).bfloat16()
    scale = 1.0 / np.sqrt(K)
    fwd, bwd = {}, {}
    for algo in (MFMA, GENERIC):
        fwd[algo] = pkg.delta_chunk_recalculated(*args, True, 64, scale, algo=algo)
        g = pkg.combined_backward(dy, None, *args, 64, scale, algo=algo)
        bwd[algo] = (g.d_q_bshk, g.d_k_bshk, g.d_v_bshv, g.d_erase_bshK, g.d_write_bshV,
                     g.d_g_bshK, g.d_state_bhkv)
    torch.cuda.synchronize()
    for got, want in zip(fwd[MFMA] + bwd[MFMA], fwd[GENERIC] + bwd[GENERIC]):
        assert rel_err(np_of(got), np_of(want)) < 2e-2
