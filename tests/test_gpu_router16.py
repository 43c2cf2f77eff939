"""The router with 16 tokens per workgroup (fp32, and bf16 with 64 experts, up
to 16 tokens per CU): the logits, indices and gates of the 64-token kernel bit
for bit (which mep_route_dispatch runs for these shapes), at token counts
around a workgroup and the switch, hidden sizes around the blocks in flight,
and every kind of k against the oracle's rule."""
import numpy as np
import pytest
import torch

from helpers import banner, to_np
from miniep_amd import ops
from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _inputs(n, H, E, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(n, H, generator=g).to(dtype).to(DEV)
    w = (torch.randn(E, H, generator=g) * 0.02).to(dtype).to(DEV)
    w[E // 2] = w[1]                                    # exactly tied logits
    return x, w


@pytest.mark.parametrize("n,H,E,dtype", [
    (1, 1024, 32, torch.float32), (15, 256, 16, torch.float32), (17, 1280, 32, torch.float32),
    (512, 512, 64, torch.float32), (4096, 256, 32, torch.float32), (4097, 256, 32, torch.float32),
    (16, 256, 64, torch.bfloat16), (33, 768, 64, torch.bfloat16), (1000, 2048, 64, torch.bfloat16),
    (4096, 1024, 64, torch.bfloat16), (4097, 1024, 64, torch.bfloat16)])
def test_router16_equals_64_token_kernel(n, H, E, dtype):
    banner(f"router16 n={n} H={H} E={E} {dtype}")
    x, w = _inputs(n, H, E, dtype, n + H)
    idx, gate, logits = ops.router_topk(x, w, 8, return_logits=True)
    idx2, gate2, _, logits2 = ops.route_dispatch(x, w, 8, return_logits=True)
    assert torch.equal(logits, logits2) and torch.equal(idx, idx2) and torch.equal(gate, gate2)


@pytest.mark.parametrize("E,k,dtype", [(16, 1, torch.float32), (16, 16, torch.float32), (32, 5, torch.float32),
                                       (64, 64, torch.float32), (64, 3, torch.bfloat16), (64, 64, torch.bfloat16)])
def test_router16_any_k(E, k, dtype):
    banner(f"router16 E={E} k={k} {dtype}")
    x, w = _inputs(45, 512, E, dtype, E + k)
    idx, gate, logits = ops.router_topk(x, w, k, return_logits=True)
    assert torch.equal(logits, ops.router_topk(x, w, 8, return_logits=True)[2])
    ridx, rgate = O.topk_softmax(to_np(logits), k, gate_bf16=dtype == torch.bfloat16)
    assert np.array_equal(to_np(idx), ridx)
    assert np.abs(to_np(gate) - rgate).max() <= (2 ** -8 if dtype == torch.bfloat16 else 2e-6)
