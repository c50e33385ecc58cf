"""The chunk-local backward (csrc/chunk_bwd_local.hip) at its edges: one value
step of 32 columns more or less than two, ragged and single-token chunks, each
gate width, fp32 and bf16 gradients, no forget gate, a write gate that is
aligned to its elements only, and the shapes either side of the ones that
chunk_bwd_mfma.hip keeps. Against the fp32 kernels, which end in the same code
(csrc/chunk_bwd_tail.hpp), and the float64 oracle, at the bf16 path's bar (attnᵀ
and the decayed keys are single bf16 factors, 2^-9 of a term each)."""

import numpy as np
import pytest
import torch

from conftest import random_raw
from gpu_util import announce, as_oracle_inputs, np_of, pkg, to_gpu
from oracle import oracle as O

pytestmark = pytest.mark.gpu

MFMA, GENERIC = pkg.abi.DN_ALGO_MFMA, pkg.abi.DN_ALGO_GENERIC


# S, K, V, widths of erase and write (0: 1 each, per-head decay; -1: no decay)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("S,K,V,widths", [
    (1, 128, 64, 0), (63, 64, 192, 0), (65, 128, 128, -1), (130, 128, 256, 0), (64, 64, 128, 0),
    (130, 64, 64, (64, 64)), (63, 128, 192, (1, 192)), (1, 64, 128, (64, 1)),
    (65, 128, 64, (1, 1)), (200, 128, 64, (128, 64)), (127, 64, 256, -1)])
def test_chunk_bwd_local(rng, S, K, V, widths, dtype):
    announce(f"chunk-local backward S {S} K {K} V {V} {widths} {dtype}")
    B, H = 2, 3
    raw = random_raw(rng, B, S, H, K, V, gated=widths != -1, channel=not isinstance(widths, int))
    if not isinstance(widths, int):
        raw[3], raw[4] = raw[3][..., :widths[0]], raw[4][..., :widths[1]]
    args = to_gpu(raw, torch.bfloat16)
    flat = torch.empty(args[4].numel() + 1, device=args[4].device)
    flat[1:] = args[4].flatten()
    args[4] = flat[1:].view(args[4].shape)
    dy = torch.tensor(rng.standard_normal((B, S, H, V)), device=args[0].device).to(dtype)
    ds = torch.tensor(rng.standard_normal((B, H, K, V)), device=args[0].device).float()
    out = {}
    for algo in (MFMA, GENERIC):
        g = pkg.combined_backward(dy, ds, *args, 64, 1.0 / np.sqrt(K), algo=algo)
        out[algo] = [g.d_q_bshk, g.d_k_bshk, g.d_v_bshv, g.d_erase_bshK, g.d_write_bshV,
                     g.d_g_bshK, g.d_state_bhkv]
    torch.cuda.synchronize()
    # d_g is a difference of q ⊙ d_q and k ⊙ d_k terms.
    least = max(float(np.abs(np_of(out[GENERIC][i]) * np_of(args[i])).max()) for i in (0, 1))
    fp32 = [None if t is None else np_of(t) for t in out[GENERIC]]
    exact = O.chunk_bwd(np_of(dy), np_of(ds), *as_oracle_inputs(args), chunk_len=64)
    for i, got in enumerate(out[MFMA]):
        for want in (fp32[i], exact[i]):
            if want is not None:
                scale = max(np.abs(want).max(), least if i == 5 else 0.0)
                assert np.abs(np_of(got) - want).max() / scale < 2e-2, i


@pytest.mark.parametrize("K,V,gates", [(128, 192, "head"), (64, 192, "none"), (64, 64, "channel"),
                                       (128, 64, "channel")])
def test_v_four_bytes_past_a_boundary(rng, K, V, gates):
    """v is owed 4 bytes of alignment: a view that starts there takes the same
    kernels to the same bits."""
    announce(f"v at a four-byte offset K {K} V {V} {gates}")
    raw = random_raw(rng, 1, 70, 2, K, V, gated=gates != "none", channel=gates == "channel")
    args = to_gpu(raw, torch.bfloat16)
    dy = torch.tensor(rng.standard_normal(raw[2].shape), device=args[0].device).bfloat16()
    flat = torch.empty(args[2].numel() + 2, dtype=torch.bfloat16, device=args[0].device)
    flat[2:] = args[2].flatten()
    off = list(args)
    off[2] = flat[2:].view(args[2].shape)
    assert off[2].data_ptr() % 8 == 4
    for a, b in zip(*[vars(pkg.combined_backward(dy, None, *x, 64, 1.0 / np.sqrt(K), algo=MFMA)).values()
                      for x in (args, off)]):
        assert (a is None and b is None) or torch.equal(a, b)


@pytest.mark.parametrize("K,gates", [(128, "head"), (64, "channel"), (128, "channel")])
def test_infinite_value_of_the_last_token(rng, K, gates):
    """The erase gates before a token do not meet its value, whatever that is:
    their gradients are those of a finite one, to the bit."""
    announce(f"chunk-local backward: an infinite value K {K} {gates}")
    S, V = 128, 64
    args = to_gpu(random_raw(rng, 1, S, 2, K, V, channel=gates == "channel"), torch.bfloat16)
    dy = torch.tensor(rng.standard_normal((1, S, 2, V)), device=args[0].device).bfloat16()
    out = []
    for value in (1.0, float("inf")):
        args[2][:, -1, :, 3] = value
        out.append(pkg.combined_backward(dy, None, *args, 64, 1.0 / np.sqrt(K),
                                         algo=MFMA).d_erase_bshK[:, :-1])
    assert bool(torch.isfinite(out[1]).all()) and torch.equal(*out)
