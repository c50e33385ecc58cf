"""How the scans cover the device (scan_shape): one or two four-wave teams, or
4 or 8 lone waves, to a workgroup, at head counts either side of where the
choice turns, and the team scans' segments where they are uneven or empty. The
bf16 MFMA forward and backward against the fp32 kernels, at the bf16 path's
bar."""

import numpy as np
import pytest
import torch

from conftest import random_raw, rel_err
from gpu_util import announce, np_of, pkg, to_gpu

pytestmark = pytest.mark.gpu

MFMA, GENERIC = pkg.abi.DN_ALGO_MFMA, pkg.abi.DN_ALGO_GENERIC


# On 256 CUs, H·V/16 teams: forward one team a workgroup to 256 of them, two to
# 512, then 4 and 8 lone waves; the backward's pair of scans turns at half.
# (tests/cpp/test_launches.cpp asserts which of them a call launches.) 330 tokens
# are six chunks: every buffer of a scan is filled again.
@pytest.mark.parametrize("H,K,V,gates", [
    (3, 128, 64, "none"), (7, 128, 256, "head"), (17, 128, 256, "head"), (32, 128, 256, "head"),
    (33, 128, 256, "head"), (65, 128, 256, "head"), (5, 64, 192, "none"), (65, 64, 64, "head"),
    (9, 128, 128, "channel"), (33, 128, 256, "channel"), (66, 64, 128, "channel"),
    (129, 64, 128, "head"), (128, 64, 192, "channel")])
@pytest.mark.parametrize("S", [1, 70, 330])
def test_scan_width(rng, H, K, V, gates, S):
    announce(f"scan width H {H} K {K} V {V} {gates} S {S}")
    raw = random_raw(rng, 1, S, H, K, V, gated=gates != "none", channel=gates == "channel")
    args = to_gpu(raw, torch.bfloat16)
    dy = torch.tensor(rng.standard_normal((1, S, H, V)), device=args[0].device).bfloat16()
    ds = torch.tensor(rng.standard_normal((1, H, K, V)), device=args[0].device).float()
    scale = 1.0 / np.sqrt(K)
    out = {}
    for algo in (MFMA, GENERIC):
        y, s = pkg.delta_chunk_recalculated(*args, gates != "none", 64, scale, algo=algo)
        g = pkg.combined_backward(dy, ds, *args, 64, scale, algo=algo)
        out[algo] = [y, s, g.d_q_bshk, g.d_k_bshk, g.d_v_bshv, g.d_erase_bshK, g.d_write_bshV,
                     g.d_g_bshK, g.d_state_bhkv]
    torch.cuda.synchronize()
    # A single token's d_g is a difference of q ⊙ d_q and k ⊙ d_k (bf16 terms).
    least = max(rel_base(out[GENERIC][2], args[0]), rel_base(out[GENERIC][3], args[1]))
    for i, (got, want) in enumerate(zip(out[MFMA], out[GENERIC])):
        if want is not None:
            scale_ = max(np.abs(np_of(want)).max(), least if i == 7 else 0.0)
            assert np.abs(np_of(got) - np_of(want)).max() / scale_ < 2e-2, i


def rel_base(grad, x):
    return float(np.abs(np_of(grad) * np_of(x)).max())


@pytest.mark.parametrize("N,K,V,gates", [(50, 128, 64, "head"), (45, 64, 128, "head"),
                                         (41, 128, 64, "channel"), (37, 64, 64, "none"),
                                         (161, 128, 64, "head")])  # the last segment is empty
def test_uneven_segments(rng, N, K, V, gates):
    announce(f"uneven segments N {N} K {K} V {V} {gates}")
    args = to_gpu(random_raw(rng, 1, 64 * N, 1, K, V, gated=gates != "none",
                             channel=gates == "channel"), torch.bfloat16)
    run = lambda algo: pkg.delta_chunk_recalculated(*args, gates != "none", 64, 1.0 / np.sqrt(K),
                                                    algo=algo, y_dtype=torch.float32)
    want = run(GENERIC)
    torch.cuda.synchronize()
    pkg.abi.profile_enable(True)
    got = run(MFMA)
    torch.cuda.synchronize()
    names = pkg.abi.profile_read()
    pkg.abi.profile_enable(False)
    assert "dn_mfma_seg_carry" in names, names
    for a, b in zip(got, want):
        assert rel_err(np_of(a), np_of(b)) < 2e-2
