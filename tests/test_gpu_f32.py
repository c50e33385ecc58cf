"""What DN_ALGO_GENERIC names, against the float64 oracle: the fp32 matrix-core
chunk kernels (csrc/chunk_f32.hpp; head_k_dim up to 128, chunks of 64) at the
edges of their tiles (key blocks of 32, value columns of 16 in one- and two-team
workgroups, a chunk's 64 tokens), and the kernels of any shape
(csrc/chunk_generic.hip) in what is left to them.

Bar: an output is a sum of products over at most K keys and two triangles of
64 tokens, each rounded to 2^-24 of the running sum; twice that worst case,
normwise."""

import numpy as np
import pytest
import torch

from conftest import random_raw, rel_err
from gpu_util import DEV, announce, as_oracle_inputs, np_of, pkg, to_gpu
from oracle import oracle as O

pytestmark = pytest.mark.gpu

GENERIC = pkg.abi.DN_ALGO_GENERIC


def bar(K):
    return 2 * (K + 2 * 64) * 2.0 ** -24


def inputs(rng, B, S, H, K, V, erase, write, decay):
    """Gates by width: 1, the head's (None: no forget gate)."""
    q, k, v, e, w, g, s = random_raw(rng, B, S, H, K, V, channel=True)
    cut = lambda x, width: x[..., :1].copy() if width == 1 else x
    return [q, k, v, cut(e, erase), cut(w, write), None if decay is None else cut(g, decay), s]


# B, S, H, K, V, chunk_len, widths of erase, write and decay
CASES = [
    (1, 1, 1, 1, 1, 64, (1, 1, 1)),
    (1, 64, 1, 32, 16, 64, (1, 1, None)),
    (2, 65, 3, 33, 17, 64, (33, 1, 1)),
    (1, 63, 2, 64, 5, 64, (1, 5, 64)),
    (2, 130, 1, 100, 48, 64, (100, 48, 100)),
    (1, 128, 2, 128, 40, 64, (1, 1, 1)),
    (1, 96, 2, 128, 130, 64, (128, 130, 128)),
    (3, 70, 1, 96, 33, 100, (1, 33, 1)),
    (1, 200, 2, 66, 32, 64, (66, 1, None)),
    # 288 column tiles: more than the device's CUs, so two-team workgroups
    (9, 66, 16, 64, 24, 64, (1, 1, 1)),
    (9, 66, 16, 128, 24, 64, (128, 24, 128)),
    # ... and chunks enough for every buffer to be filled a second and third time
    (9, 330, 16, 64, 24, 64, (1, 1, 1)),
    (9, 330, 16, 32, 40, 64, (32, 1, 32)),
    (1, 330, 2, 128, 24, 64, (1, 24, 128)),
]

# The kernels of any shape, where the others do not go: head_k_dim above 128,
# a per-channel forget gate in other chunks than 64, short chunks.
ANY_SHAPE = [
    (1, 70, 2, 129, 20, 64, (1, 1, 1)),
    (1, 130, 1, 192, 40, 64, (192, 40, 192)),
    (2, 65, 1, 256, 64, 64, (1, 64, None)),
    (1, 33, 2, 300, 17, 100, (300, 1, 1)),
    (1, 90, 2, 64, 24, 40, (1, 1, 64)),
    (1, 200, 2, 66, 32, 32, (66, 1, None)),
]


def profiled(f, kernels="dn_f32"):
    pkg.abi.profile_enable(True)
    out = f()
    torch.cuda.synchronize()
    names = pkg.abi.profile_read()
    pkg.abi.profile_enable(False)
    assert names and all(n.startswith(kernels) for n in names), names
    return out


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("case", CASES)
def test_f32_forward_and_backward_match_oracle(rng, case, dtype):
    match_oracle(rng, case, dtype, "dn_f32")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("case", ANY_SHAPE)
def test_any_shape_forward_and_backward_match_oracle(rng, case, dtype):
    match_oracle(rng, case, dtype, "dn_generic")


def match_oracle(rng, case, dtype, kernels):
    B, S, H, K, V, L, (ew, ww, dw) = case
    announce(f"{kernels} kernels {case} {dtype}")
    args = inputs(rng, B, S, H, K, V, ew, ww, dw)
    g_args = to_gpu(args, dtype)
    ref = as_oracle_inputs(g_args)
    scale = 1.0 / np.sqrt(K)
    y, s = profiled(lambda: pkg.delta_chunk_recalculated(
        *g_args, dw is not None, L, scale, algo=GENERIC, y_dtype=torch.float32), kernels)
    want_y, want_s = O.chunk_fwd(*ref, chunk_len=L)
    assert rel_err(np_of(y), want_y) < bar(K)
    assert rel_err(np_of(s), want_s) < bar(K)
    dy = torch.tensor(rng.standard_normal((B, S, H, V)), dtype=torch.float32, device=DEV)
    ds = torch.tensor(rng.standard_normal((B, H, K, V)), dtype=torch.float32, device=DEV)
    got = profiled(lambda: pkg.combined_backward(dy, ds, *g_args, L, scale, algo=GENERIC), kernels)
    want = O.chunk_bwd(np_of(dy), np_of(ds), *ref, chunk_len=L)
    names = ("d_q_bshk", "d_k_bshk", "d_v_bshv", "d_erase_bshK", "d_write_bshV", "d_g_bshK",
             "d_state_bhkv")
    # d_g sums q ⊙ d_q and k ⊙ d_k with both signs (at one token of one channel
    # the sum is 1e-3 of its terms): its rounding is that of the terms.
    term = max(float(np.abs(want[i] * ref[i]).max()) for i in (0, 1))
    for name, x in zip(names, want):
        if x is not None:
            least = term if name == "d_g_bshK" else 0.0
            err = np.abs(np_of(getattr(got, name)) - x).max() / max(np.abs(x).max(), least)
            assert err < bar(K), name


def test_f32_kernels_do_not_enlarge_a_workspace(rng):
    """One chunk of 65 tokens of a small head: two 64-token chunks' tiles would
    need more scratch than a caller held for it, so it keeps its kernels."""
    args = to_gpu(inputs(rng, 1, 65, 1, 4, 4, 1, 1, 1))
    y, s = torch.empty_like(args[2]), torch.empty_like(args[6])
    held = [pkg.abi.lib().dn_chunk_fwd_workspace_bytes(
        pkg.abi.chunk_fwd_args(*args, y, s, L, 0.5, algo=GENERIC)) for L in (65, 64)]
    assert 0 < held[0] < held[1]
    for L, kernels in ((65, "dn_generic"), (64, "dn_f32")):
        profiled(lambda: pkg.delta_chunk_recalculated(*args, True, L, 0.5, algo=GENERIC), kernels)


@pytest.mark.parametrize("K", [32, 128])
@pytest.mark.parametrize("L", [16, 32])
def test_short_chunks_are_as_accurate_as_their_length(rng, L, K):
    """The state is cleared by a log gate of -3e4 at the last token of every
    second short chunk, which leaves no sum that the gate enters beside others;
    carried on in a longer chunk, a cumulative gate of -3e4 (2^-9 its last bit)
    would cost the tokens after it three digits."""
    B, S, H, V = 1, 200, 2, 24
    announce(f"short chunks L {L} K {K}")
    args = inputs(rng, B, S, H, K, V, 1, 1, 1)
    args[5][:, L - 1::2 * L] = -3e4
    g_args = to_gpu(args)
    ref = as_oracle_inputs(g_args)
    y, s = pkg.delta_chunk_recalculated(*g_args, True, L, 0.5, algo=GENERIC)
    want = O.chunk_fwd(*ref, chunk_len=L, scale=0.5)
    assert rel_err(np_of(y), want[0]) < bar(K) and rel_err(np_of(s), want[1]) < bar(K)
    dy = torch.tensor(rng.standard_normal((B, S, H, V)), dtype=torch.float32, device=DEV)
    got = pkg.combined_backward(dy, None, *g_args, L, 0.5, algo=GENERIC)
    want = O.chunk_bwd(np_of(dy), np.zeros(want[1].shape), *ref, chunk_len=L, scale=0.5)
    for i, name in enumerate(("d_q_bshk", "d_k_bshk", "d_v_bshv", "d_erase_bshK",
                              "d_write_bshV")):
        assert rel_err(np_of(getattr(got, name)), want[i]) < bar(K), name


@pytest.mark.parametrize("widths", [(1, 1, 1), (64, 24, 64)])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_erase_gate_that_is_not_finite(rng, value, widths):
    """The gradients of v and the write gate from a token on do not meet its
    erase gate, whatever that is: they are those of a finite one, to the bit."""
    announce(f"f32 kernels: erase gate {value} {widths}")
    S, K, V, t = 100, 64, 24, 20
    args = to_gpu(inputs(rng, 1, S, 2, K, V, *widths))
    dy = torch.tensor(rng.standard_normal((1, S, 2, V)), dtype=torch.float32, device=DEV)
    out = []
    for e in (0.5, value):
        args[3][:, t, 0, 0] = e
        g = profiled(lambda: pkg.combined_backward(dy, None, *args, 64, 0.5, algo=GENERIC))
        out.append((g.d_v_bshv[:, t:], g.d_write_bshV[:, t:]))
    for want, got in zip(*out):
        assert bool(torch.isfinite(got).all()) and torch.equal(want, got)


@pytest.mark.parametrize("V,widths", [(40, (1, 1, 1)), (24, (64, 24, 64))])
def test_workspace_at_a_four_byte_boundary(rng, V, widths):
    """The generic path's workspace is owed the alignment of its floats: one
    that starts four bytes past a boundary holds the same bits."""
    announce(f"f32 kernels: workspace off a 16-byte boundary V {V} {widths}")
    B, S, H, K = 1, 130, 2, 64
    args = to_gpu(inputs(rng, B, S, H, K, V, *widths))
    dy = torch.tensor(rng.standard_normal((B, S, H, V)), dtype=torch.float32, device=DEV)
    lib, out = pkg.abi.lib(), []
    for off in (0, 4):
        y, s = torch.empty_like(args[2]), torch.empty_like(args[6])
        grads = [torch.empty_like(t) for t in args]
        fwd = pkg.abi.chunk_fwd_args(*args, y, s, 64, 0.5, algo=GENERIC)
        bwd = pkg.abi.chunk_bwd_args(dy, None, *args, grads, 64, 0.5, algo=GENERIC)
        for a, size, run in ((fwd, lib.dn_chunk_fwd_workspace_bytes, pkg.abi.run_chunk_fwd),
                             (bwd, lib.dn_chunk_bwd_workspace_bytes, pkg.abi.run_chunk_bwd)):
            ws = torch.empty(size(a) + off, dtype=torch.uint8, device=DEV)
            a.workspace, a.workspace_bytes = ws.data_ptr() + off, size(a)
            profiled(lambda: run(a))
        out.append([y, s] + grads)
    assert all(torch.equal(a, b) for a, b in zip(*out))
