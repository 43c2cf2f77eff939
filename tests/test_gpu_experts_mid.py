"""The mid-size experts launch (some tens to a few hundred rows per expert in
bf16, any in fp32; both GEMMs in one launch): the bits of the two separate launches on every
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


def _case(counts, k, H, I, seed, dtype=BF):
    E, n = len(counts), sum(counts) // k
    topk = _topk_with_counts(counts, k, n, seed)
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(n, H, generator=g).to(dtype).to(DEV)
    w_in, w_out = workloads.expert_weights(g, E, H, I)
    table, n_rep, g2l = _world1(E)
    d = ops.dispatch(topk.to(DEV), None, E, table, n_rep, False, None, 0, g2l, E)
    return x, d, w_in.to(dtype).to(DEV), w_out.to(dtype).to(DEV)


@pytest.mark.parametrize("name,counts,k,H,I", [
    # fp32 (names "f32..."): 32-row chunks, the shortest K loop (128 floats); 64-row chunks with short last ones
    ("f32_edges32", [0, 1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 3], 2, 256, 128),
    ("f32_one_row", [1], 1, 1024, 512),
    ("f32_edges64", [64, 1, 127, 128, 129, 63, 65, 16, 33, 31, 96, 97] * 2, 2, 512, 2048),
    # 64-row chunks: empty experts, 1 row, around fragments, halves and chunks
    ("edges64", [0, 1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 96, 97, 128, 129, 13], 4, 1024, 512),
    # 128-row chunks: an average of 64 rows and more, enough column blocks
    ("edges128", [64, 1, 127, 128, 129, 63, 65, 16] * 4, 4, 512, 1024),
    ("k256", [40, 100, 7, 210, 11, 0, 64, 80], 2, 256, 256),       # the shortest K loops, no rotation of whole quarters
    # the shortest K loop with every rotation of it, 64- and 128-row chunks, several chunks of an expert
    ("k256_rot64", [130, 1, 65, 64, 200, 0, 96, 84], 2, 1024, 256),
    ("k256_rot64_wide", [40, 100, 7, 210, 11, 0, 64, 80], 2, 2048, 256),
    ("k256_rot128", [64, 1, 127, 128, 129, 63, 257, 16] * 8, 5, 1024, 256),
    ("one_expert", [300], 1, 1024, 512),                            # fewer chunks than XCDs
    ("e64_wide", [5] * 63 + [197], 2, 2048, 1024),
    ("hot", [1000, 8, 8, 8, 8, 8, 4, 4], 1, 1024, 512),
])
def test_mid_launch_equals_two_launches(name, counts, k, H, I):
    banner(f"mid-size experts launch: {name}")
    f32 = name.startswith("f32")
    x, d, wi, wo = _case(counts, k, H, I, len(counts), torch.float32 if f32 else BF)
    n = x.shape[0]
    assert f32 or n * k > 256
    results = []
    for rep in range(2):                                            # a second input through the same buffers
        xr = x if rep == 0 else -x.flip(0).contiguous()
        y1 = torch.full((n * k, H), 7.0, dtype=x.dtype, device=DEV)
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


def test_f32_small_schedule_buffer():
    """fp32 calls with a schedule buffer below mep_experts_queue_ints keep the
    two launches, which take any: same bits."""
    banner("experts fp32: small schedule buffer")
    x, d, wi, wo = _case([40, 3, 0, 21], 1, 256, 128, 9, torch.float32)
    L = _lib.lib()
    n, H, I = x.shape[0], 256, 128
    want = ops.grouped_swiglu(x, d, wi, wo)
    got = torch.empty_like(want)
    ws = torch.empty(L.mep_experts_workspace_size(n, I, _lib.DTYPE_F32), dtype=torch.uint8, device=DEV)
    tq = torch.zeros(64, dtype=torch.int32, device=DEV)
    rc = L.mep_grouped_swiglu(x.data_ptr(), n, 1, d.perm.data_ptr(), d.offsets.data_ptr(), 4, n, wi.data_ptr(),
                              wo.data_ptr(), H, I, _lib.DTYPE_F32, got.data_ptr(), ws.data_ptr(), ws.numel(),
                              tq.data_ptr(), tq.numel(), torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and torch.equal(got, want) and int(tq.abs().sum()) == 0
