"""The mid-size experts launch (some tens to a few hundred rows per expert,
both GEMMs in one launch): the bits of the two separate launches on every
row, at row counts around the edges of its 16-row fragments, half chunks and
chunks, with few and many experts, and a wait that gives up."""
import numpy as np
import pytest
import torch

from helpers import banner
from miniep_amd import _lib, ops, workloads
from test_gpu_experts import _topk_with_counts, _two_launches, _world1
from test_gpu_giveup import _cells, _first_rows, _queue_words_zero, _raises_hip, force_giveup

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF = torch.bfloat16


def _case(counts, k, H, I, seed):
    E, n = len(counts), sum(counts) // k
    topk = _topk_with_counts(counts, k, n, seed)
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(n, H, generator=g).to(BF).to(DEV)
    w_in, w_out = workloads.expert_weights(g, E, H, I)
    table, n_rep, g2l = _world1(E)
    d = ops.dispatch(topk.to(DEV), None, E, table, n_rep, False, None, 0, g2l, E)
    return x, d, w_in.to(BF).to(DEV), w_out.to(BF).to(DEV)


@pytest.mark.parametrize("name,counts,k,H,I", [
    # 64-row chunks: empty experts, 1 row, around fragments, halves and chunks
    ("edges64", [0, 1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 96, 97, 128, 129, 13], 4, 1024, 512),
    # 128-row chunks: an average of 64 rows and more, enough column blocks
    ("edges128", [64, 1, 127, 128, 129, 63, 65, 16] * 4, 4, 512, 1024),
    ("k256", [40, 100, 7, 210, 11, 0, 64, 80], 2, 256, 256),       # the shortest K loops, no rotation of whole quarters
    ("one_expert", [300], 1, 1024, 512),                            # fewer chunks than XCDs
    ("e64_wide", [5] * 63 + [197], 2, 2048, 1024),
    ("hot", [1000, 8, 8, 8, 8, 8, 4, 4], 1, 1024, 512),
])
def test_mid_launch_equals_two_launches(name, counts, k, H, I):
    banner(f"mid-size experts launch: {name}")
    x, d, wi, wo = _case(counts, k, H, I, len(counts))
    n = x.shape[0]
    assert n * k > 256
    results = []
    for rep in range(2):                                            # a second input through the same buffers
        xr = x if rep == 0 else x.flip(0).contiguous()
        y1 = torch.full((n * k, H), 7.0, dtype=BF, device=DEV)
        y2 = y1.clone()
        ops.grouped_swiglu(xr, d, wi, wo, y1)
        _two_launches(xr, d, wi, wo, y2)
        ops.experts_check()
        assert torch.equal(y1, y2), rep
        _queue_words_zero()
        results.append(y1)
    assert not torch.equal(*results)


def test_mid_launch_slots_and_masks():
    """Weight slots, and masked tokens whose cells stay untouched."""
    banner("mid-size experts launch: slots, masks")
    g = torch.Generator().manual_seed(5)
    E, k, n, H, I = 32, 8, 150, 1024, 512
    topk = torch.rand(n, E, generator=g).topk(k, -1).indices
    valid = torch.rand(n, generator=g) < 0.7
    x = torch.randn(n, H, generator=g).to(BF).to(DEV)
    w_in, w_out = (w.to(BF).to(DEV) for w in workloads.expert_weights(g, E, H, I))
    table, n_rep, g2l = _world1(E)
    d = ops.dispatch(topk.to(DEV), valid.to(DEV), E, table, n_rep, False, None, 0, g2l, E)
    y1 = torch.full((n * k, H), 7.0, dtype=BF, device=DEV)
    y2, y3 = y1.clone(), y1.clone()
    ops.grouped_swiglu(x, d, w_in, w_out, y1)
    _two_launches(x, d, w_in, w_out, y2)
    slot = torch.randperm(E, generator=g)
    inv = torch.argsort(slot).to(DEV)
    ops.grouped_swiglu(x, d, w_in[inv].contiguous(), w_out[inv].contiguous(), y3, w_slot=slot.to(torch.int32).to(DEV))
    ops.experts_check()
    assert torch.equal(y1, y2) and torch.equal(y1, y3)
    assert bool((y1[(~valid).repeat_interleave(k).to(DEV)] == 7.0).all())


def test_mid_launch_giveup():
    """Chunk 0's GEMM-2 workgroups wait for a count that cannot come: NaN in
    its 64 rows' cells, the flag, the schedule words at zero, the next call
    exact."""
    banner("mid-size experts launch: give-up")
    x, d, wi, wo = _case([70, 30, 40, 0, 50, 60, 33, 37], 1, 1024, 512, 3)
    y0 = torch.full((320, 1024), 7.0, dtype=BF, device=DEV)
    ops.grouped_swiglu(x, d, wi, wo, y0)
    y1 = torch.full_like(y0, 7.0)
    with force_giveup(_lib.GIVEUP_CHUNK):
        ops.grouped_swiglu(x, d, wi, wo, y1)
        torch.cuda.synchronize()
    _raises_hip(ops.experts_check, "gave up waiting")
    bad = np.zeros(320, bool)
    bad[_cells(d, _first_rows(d, 64))] = True
    bad = torch.from_numpy(bad).to(DEV)
    assert int(bad.sum()) == 64 and bool(torch.isnan(y1[bad].float()).all())
    assert torch.equal(y1[~bad], y0[~bad])
    _queue_words_zero()
    y2 = torch.full_like(y0, 7.0)
    ops.grouped_swiglu(x, d, wi, wo, y2)
    ops.experts_check()
    assert torch.equal(y2, y0)
