"""Gradients through one of the two outputs: the other's cotangent reaches the
backward as nothing at all, and has to act as zeros; on the default stream and
on another one."""

import numpy as np
import pytest
import torch

from conftest import random_raw
from gpu_util import announce, pkg, to_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,K,S", [(torch.float32, 64, 70), (torch.bfloat16, 128, 130),
                                       (torch.bfloat16, 256, 64)])
@pytest.mark.parametrize("used", ["y", "state"])
def test_one_output(rng, dtype, K, S, used):
    announce(f"gradients through {used} {dtype} K {K} S {S}")
    args = to_gpu(random_raw(rng, 2, S, 2, K, 128), dtype)
    leaves = [a.requires_grad_() for a in args]
    y, s = pkg.DeltaInput(*leaves).run()
    dy, ds = torch.randn_like(y), torch.randn_like(s)
    if used == "y":
        want = torch.autograd.grad([y, s], leaves, [dy, torch.zeros_like(s)], retain_graph=True)
    else:
        want = torch.autograd.grad([y, s], leaves, [torch.zeros_like(y), ds], retain_graph=True)
    torch.cuda.synchronize()
    for stream in (torch.cuda.current_stream(), torch.cuda.Stream()):
        with torch.cuda.stream(stream):
            y, s = pkg.DeltaInput(*leaves).run()
            got = torch.autograd.grad(*((y, leaves, dy) if used == "y" else (s, leaves, ds)))
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            # (atomic sums differ in their order)
            bar = 2.0 ** (-7 if a.dtype == torch.bfloat16 else -12)
            assert (a - b).abs().max() <= bar * b.abs().max()
            assert np.isfinite(float(a.float().sum()))
