"""The kernels around the MoE block (ops.add_norm, ops.attention) against the
same steps in fp64, and the model's native forward against its torch
statement."""
import pytest
import torch

from miniep_amd import HipMoEBackend, ops
from miniep_amd.model import (GraniteMoeModel, KVCache, ModelConfig, RotaryTable, build_hip_model,
                              random_weights)

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,H", [(1, 1024), (5, 1000), (33, 2048), (3, 4096), (2, 8), (7, 2056)])
def test_add_norm(n, H, dtype):
    """Row widths below, at and above a lane's chunk counts.  h_out's two
    roundings are torch's own; x is within one rounding of the fp64 norm."""
    g = torch.Generator().manual_seed(n * H)
    h, d = (torch.randn(n, H, generator=g).to(dtype).to(DEV) for _ in range(2))
    w = (1 + 0.1 * torch.randn(H, generator=g)).to(dtype).to(DEV)
    for delta in (d, None):
        h2, x = ops.add_norm(h, w, 1e-6, delta, 0.22)
        want_h = h if delta is None else h + delta * 0.22
        assert torch.equal(h2, want_h)
        hd = want_h.double()
        want = w.double() * hd * torch.rsqrt(hd.pow(2).mean(-1, keepdim=True) + 1e-6)
        # fp32: the mean of H squares (H/64 + 6 adds), rsqrt and two products; bf16 adds its rounding
        eps = 2.0 ** -8 if dtype == torch.bfloat16 else (H / 64 + 12) * 2.0 ** -24
        assert ((x.double() - want).abs() <= eps * want.abs() + 1e-30).all()


def _rope64(t, rope, pos):
    cos, sin = rope.cos[pos].double(), rope.sin[pos].double()       # (t, d)
    half = t.shape[-1] // 2
    return t * cos + torch.cat([-t[..., half:], t[..., :half]], -1) * sin


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,T,start,hq,hk", [
    (1, 1, 0, 16, 8), (3, 1, 63, 16, 8), (2, 1, 64, 4, 4), (1, 1, 255, 8, 2), (2, 1, 2047, 16, 8), (1, 1, 2500, 8, 2),
    (2, 2, 0, 16, 8), (1, 17, 0, 4, 4), (2, 64, 5, 8, 2), (1, 65, 0, 16, 8), (2, 130, 70, 16, 8)])
def test_attention(B, T, start, hq, hk, dtype):
    """Decode (one token: the new position alone, chunks of 2048 scores and
    one past them) and prefill (partial and whole blocks of 64 queries and
    keys, cached positions in front), 1, 2 and 4 query heads per kv head;
    positions of the cache past the call stay as they are."""
    d, max_len = 64, start + T + 3
    cfg = ModelConfig(num_attention_heads=hq, num_key_value_heads=hk, hidden_size=64 * hq)
    rope = RotaryTable(cfg, DEV)
    g = torch.Generator().manual_seed(B + T + start)
    q, k, v = (torch.randn(B * T, h * d, generator=g).to(dtype).to(DEV) for h in (hq, hk, hk))
    cache = torch.randn(2, B, hk, max_len, d, generator=g).to(DEV)
    kc, vc = cache[0].clone(), cache[1].clone()
    out = ops.attention(q, k, v, rope.cos, rope.sin, B, start, kc, vc, 0.05)

    pos = torch.arange(start, start + T, device=DEV)
    qd, kd, vd = (t.double().view(B, T, -1, d).transpose(1, 2) for t in (q, k, v))
    qd, kd = _rope64(qd, rope, pos), _rope64(kd, rope, pos)
    want_k, want_v = cache[0].double(), cache[1].double()
    want_k[:, :, start:start + T], want_v[:, :, start:start + T] = kd, vd
    assert torch.equal(vc.double(), want_v)
    assert (kc.double() - want_k).abs().max() <= 3 * 2.0 ** -24 * want_k.abs().max()
    S = start + T
    kk, vv = (t[:, :, :S].repeat_interleave(hq // hk, 1) for t in (want_k, want_v))
    s = (qd @ kk.transpose(2, 3).contiguous()) * 0.05
    s = s.masked_fill(torch.arange(S, device=DEV) > pos[:, None], -torch.inf)
    want = (torch.softmax(s, -1) @ vv).transpose(1, 2).reshape(B * T, hq * d)
    # a score is a sum of 64 products (error below 64 ulp of the largest), so a
    # probability is off by that times the score, and the values' sum adds S/64 + 16 roundings
    tol = (64 * float(s[s.isfinite()].abs().max()) + S / 64 + 32) * 2.0 ** -24 * float(vv.abs().max())
    err = (out.double() - want).abs()
    if dtype == torch.bfloat16:
        err = err - 2.0 ** -8 * want.abs()
    assert float(err.max()) <= tol


@pytest.mark.parametrize("T,dead", [(1, 2048), (1, 2100), (1, 3), (70, 64), (70, 130), (70, 1)])
def test_attention_scores_of_minus_infinity(T, dead):
    """Cached keys whose scores are -inf weigh 0, also where they fill the first
    chunk (decode) or block (prefill) of keys."""
    B, hq, hk, d, start = 2, 8, 4, 64, dead + 5
    cfg = ModelConfig(num_attention_heads=hq, num_key_value_heads=hk, hidden_size=64 * hq)
    rope = RotaryTable(cfg, DEV)
    g = torch.Generator().manual_seed(dead + T)
    q = torch.full((B * T, hq * d), 1.0, device=DEV)
    k, v = (torch.randn(B * T, hk * d, generator=g).to(DEV) for _ in range(2))
    cache = torch.randn(2, B, hk, start + T, d, generator=g).to(DEV)
    pos = torch.arange(start, start + T, device=DEV)
    # a dead key is 0 but for its element 63, where every rotated query is positive
    turned = _rope64(q.double().view(B, T, hq, d).transpose(1, 2), rope, pos)
    cache[0][:, :, :dead] = 0.0
    cache[0][:, :, :dead, 63] = -torch.inf
    assert bool((turned[..., 63] > 0).all())
    out = ops.attention(q, k, v, rope.cos, rope.sin, B, start, cache[0].clone(), cache[1].clone(), 0.05)
    kc, vc = cache[0].double(), cache[1].double()
    kc[:, :, start:] = _rope64(k.double().view(B, T, hk, d).transpose(1, 2), rope, pos)
    vc[:, :, start:] = v.double().view(B, T, hk, d).transpose(1, 2)
    kk, vv = (t.repeat_interleave(hq // hk, 1) for t in (kc, vc))
    s = (turned @ kk.transpose(2, 3).contiguous()) * 0.05
    s = s.masked_fill(torch.arange(start + T, device=DEV) > pos[:, None], -torch.inf)
    assert bool((s[..., :dead] == -torch.inf).all())
    want = (torch.softmax(s, -1) @ vv).transpose(1, 2).reshape(B * T, hq * d)
    tol = (64 * float(s[s.isfinite()].abs().max()) + (start + T) / 64 + 32) * 2.0 ** -24 * float(vv.abs().max())
    assert float((out.double() - want).abs().max()) <= tol         # (NaN fails it)


def _count_native(m):
    """The calls of m's forward on the HIP kernels, appended as they are made."""
    calls, inner = [], m._forward_native

    def forward(*a, **kw):
        calls.append(a[0].shape)
        return inner(*a, **kw)
    m._forward_native = forward
    return calls


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_native_forward_equals_torch_statement(dtype):
    """Prefill, a decode step and a second chunk through one cache, and the
    cacheless forward, against the same model made to run its torch statement
    (an explicit causal mask).  One layer of rounding differences in bf16,
    fp32 sums otherwise."""
    cfg = ModelConfig(num_hidden_layers=2, vocab_size=997)
    w = random_weights(cfg, seed=3, dtype=dtype, device=DEV)
    m = build_hip_model(cfg, w)
    ids = torch.randint(0, cfg.vocab_size, (3, 45), generator=torch.Generator().manual_seed(1)).to(DEV)

    def causal(t, s):
        return torch.arange(s, device=DEV) <= torch.arange(s - t, s, device=DEV)[:, None]

    tol = 2e-2 if dtype == torch.bfloat16 else 2e-5
    native = _count_native(m)
    a, b = (KVCache(cfg, 3, 50, DEV) for _ in range(2))
    for lo, hi in ((0, 30), (30, 31), (31, 45)):
        got = m(ids[:, lo:hi], cache=a)
        want = m(ids[:, lo:hi], cache=b, attn_mask=causal(hi - lo, hi))
        assert a.length == b.length == hi and got.shape == want.shape
        assert native.pop() == (3, hi - lo) and not native           # the first call ran on them, the second did not
        assert float((got - want).norm() / want.norm()) <= tol
    at = torch.tensor([3, -1, 44], device=DEV)
    got, want = m(ids, logits_at=at), m(ids, logits_at=at, attn_mask=causal(45, 45))
    assert native == [(3, 45)]
    assert got.shape == (3, 1, cfg.vocab_size) and float((got - want).norm() / want.norm()) <= tol


@pytest.mark.parametrize("what", ["KVCache.write", "RotaryTable.rotate", "_block", "_attention", "set on the object",
                                  "set on the class"])
def test_overridden_parts_are_called(what, monkeypatch):
    """A program's own cache write, rotation, block or attention (a subclass's,
    or one put in place of ours) is called for every layer of a prefill and of a
    decode step, with the results of the native forward up to rounding."""
    cfg = ModelConfig(num_hidden_layers=2, vocab_size=997)
    m = build_hip_model(cfg, random_weights(cfg, seed=3, dtype=torch.bfloat16, device=DEV))
    ids = torch.randint(0, cfg.vocab_size, (2, 41), generator=torch.Generator().manual_seed(1)).to(DEV)
    plain = KVCache(cfg, 2, 50, DEV)
    want = [m(ids[:, :40], cache=plain), m(ids[:, 40:], cache=plain)]
    calls = []

    def counted(fn):
        def call(*a, **kw):
            calls.append(fn)
            return fn(*a, **kw)
        return call

    cache, per_layer = KVCache(cfg, 2, 50, DEV), 1
    if what == "KVCache.write":
        cache = type("Cache", (KVCache,), {"write": counted(KVCache.write)})(cfg, 2, 50, DEV)
    elif what == "RotaryTable.rotate":
        m.rope, per_layer = type("Rope", (RotaryTable,), {"rotate": counted(RotaryTable.rotate)})(cfg, DEV), 2
    elif what == "set on the object":
        cache.write = counted(cache.write)
    elif what == "set on the class":
        monkeypatch.setattr(KVCache, "write", counted(KVCache.write))
    else:
        m = type("Model", (GraniteMoeModel,), {what: counted(getattr(GraniteMoeModel, what))})(
            cfg, m.w, m.router, m.moe, fuse_router=True)
    native = _count_native(m)
    got = [m(ids[:, :40], cache=cache), m(ids[:, 40:], cache=cache)]
    assert not native and len(calls) == 2 * cfg.num_hidden_layers * per_layer
    for a, b in zip(got, want):
        assert float((a - b).norm() / b.norm()) <= 2e-2


def test_forward_under_autocast():
    """An fp32 model under autocast, whose products are then bf16: accepted, the
    result that of the torch statement."""
    cfg = ModelConfig(num_hidden_layers=2, vocab_size=997)
    m = build_hip_model(cfg, random_weights(cfg, seed=3, dtype=torch.float32, device=DEV))
    ids = torch.randint(0, cfg.vocab_size, (2, 40), generator=torch.Generator().manual_seed(1)).to(DEV)
    mask = torch.arange(40, device=DEV) <= torch.arange(40, device=DEV)[:, None]
    native = _count_native(m)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        got, want = m(ids), m(ids, attn_mask=mask)
    assert torch.equal(got, want) and not native


@pytest.mark.parametrize("model,backend,layers", [(torch.float32, torch.bfloat16, (0, 1)),
                                                  (torch.float32, torch.bfloat16, (0,)), (torch.bfloat16, torch.float32, (1,))])
def test_backends_of_another_dtype_and_shape(model, backend, layers):
    """Backends whose experts (and output) are of another dtype than the model,
    in the last layer only where the sum outgrows the weights' dtype, and one
    that returns (batch, tokens, hidden): as the torch statement has them."""
    cfg = ModelConfig(num_hidden_layers=2, vocab_size=997)
    w = random_weights(cfg, seed=3, dtype=model, device=DEV)
    m = build_hip_model(cfg, w)
    for i in layers:
        be = m.moe[i]
        m.moe[i] = HipMoEBackend(be.w_in.to(backend), be.w_out.to(backend))
    inner = m.moe[1].route_and_call
    m.moe[1].route_and_call = lambda *a, **kw: (inner(*a, **kw)[0].view(2, -1, cfg.hidden_size),)
    ids = torch.randint(0, cfg.vocab_size, (2, 41), generator=torch.Generator().manual_seed(1)).to(DEV)
    native = _count_native(m)
    a, b = KVCache(cfg, 2, 50, DEV), KVCache(cfg, 2, 50, DEV)
    for lo, hi in ((0, 40), (40, 41)):
        mask = torch.arange(hi, device=DEV) <= torch.arange(lo, hi, device=DEV)[:, None]
        got, want = m(ids[:, lo:hi], cache=a), m(ids[:, lo:hi], cache=b, attn_mask=mask)
        assert got.shape == want.shape and native.pop() == (2, hi - lo) and not native
        assert float((got - want).norm() / want.norm()) <= 2e-2


def test_backend_with_strided_output():
    """A backend whose (batch, tokens, hidden) lies tokens first in memory."""
    cfg = ModelConfig(num_hidden_layers=2, vocab_size=997)
    m = build_hip_model(cfg, random_weights(cfg, seed=3, dtype=torch.bfloat16, device=DEV))
    ids = torch.randint(0, cfg.vocab_size, (2, 40), generator=torch.Generator().manual_seed(1)).to(DEV)
    want = m(ids)
    inner = m.moe[0].route_and_call

    def tokens_first(*a, **kw):
        out = inner(*a, **kw)[0].view(2, 40, cfg.hidden_size)
        return (out.transpose(0, 1).contiguous().transpose(0, 1),)
    m.moe[0].route_and_call = tokens_first
    native = _count_native(m)
    assert torch.equal(m(ids), want) and native == [(2, 40)]


def test_native_forward_with_unaligned_tensors():
    """A backend that returns a view off the 16-byte grid, and such a cache:
    accepted, with the results of aligned ones (the cache goes through the torch
    statement, so to its rounding)."""
    cfg = ModelConfig(num_hidden_layers=2, vocab_size=997)
    m = build_hip_model(cfg, random_weights(cfg, seed=3, dtype=torch.bfloat16, device=DEV))
    ids = torch.randint(0, cfg.vocab_size, (2, 40), generator=torch.Generator().manual_seed(1)).to(DEV)
    want = m(ids)

    def off_grid(t):
        flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
        flat[1:] = t.reshape(-1)
        return flat[1:].view(t.shape)

    native = _count_native(m)
    cache = KVCache(cfg, 2, 40, DEV)
    cache.k = [off_grid(t) for t in cache.k]
    assert float((m(ids, cache=cache) - want).norm() / want.norm()) <= 2e-2
    assert not native
    inner = m.moe[0].route_and_call
    m.moe[0].route_and_call = lambda *a, **kw: (off_grid(inner(*a, **kw)[0]),)
    assert torch.equal(m(ids), want) and native == [(2, 40)]


def _norm64(h, w):
    return w.double() * h.double() * torch.rsqrt(h.double().pow(2).mean(-1, keepdim=True) + 1e-6)


@pytest.mark.parametrize("n,H,vocab", [(1, 1024, 16), (16, 1024, 49155), (17, 2048, 1000), (32, 1024, 8193)])
def test_norm_head(n, H, vocab):
    """One and two row fragments, partial column tiles, one tile and many per
    workgroup.  x is bf16 and equal to add_norm's, so the logits are fp32 sums
    of exact products: H roundings at most, of sums below |x| |w|."""
    g = torch.Generator().manual_seed(n + vocab)
    h, d = (torch.randn(n, H, generator=g).bfloat16().to(DEV) for _ in range(2))
    norm = (1 + 0.1 * torch.randn(H, generator=g)).bfloat16().to(DEV)
    w = (torch.randn(vocab, H, generator=g) * 0.02).bfloat16().to(DEV)
    for delta in (d, None):
        got = ops.norm_head(h, delta, 0.22, norm, 1e-6, w, 6.0)
        _, x = ops.add_norm(h, norm, 1e-6, delta, 0.22)
        want = x.double() @ w.double().T.contiguous() / 6.0
        # the norm's mean is summed in another order than add_norm's: a few x elements round the other way
        tol = H * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T.contiguous()) / 6.0
        flip = 2.0 ** -8 * float(x.abs().max()) * float(w.abs().max()) / 6.0
        assert ((got.double() - want).abs() <= tol + 4 * flip).all()


@pytest.mark.parametrize("B,T,start,H,hq,hk", [(1, 1, 0, 1024, 16, 8), (8, 1, 40, 1024, 16, 8), (17, 1, 3, 1024, 16, 16),
                                               (32, 1, 9, 2048, 16, 4), (3, 7, 5, 1024, 32, 8), (2, 16, 0, 2048, 32, 16)])
def test_attention_block(B, T, start, H, hq, hk):
    """mep_attention_block against the same steps as separate calls (add_norm,
    F.linear, attention): every tensor between the steps is bf16, so the two
    differ by one bf16 rounding here and there (sums in another order)."""
    d, n = 64, B * T
    cfg = ModelConfig(num_attention_heads=hq, num_key_value_heads=hk, hidden_size=64 * hq)
    rope = RotaryTable(cfg, DEV)
    g = torch.Generator().manual_seed(B * T + H)

    def mat(*shape, sd=0.02):
        return (torch.randn(*shape, generator=g) * sd).bfloat16().to(DEV)

    h, moe = mat(n, H, sd=1), mat(n, H, sd=1)
    n1, n2 = mat(H, sd=1), mat(H, sd=1)
    wq, wk, wv, wo = mat(hq * d, H), mat(hk * d, H), mat(hk * d, H), mat(H, hq * d)
    cache = torch.randn(2, B, hk, start + T, d, generator=g).to(DEV)
    ws = ops.attention_block_workspace(n, H, hq, hk, d, DEV)
    for delta in (moe, None):
        kc, vc = cache[0].clone(), cache[1].clone()
        got_h, got_x = ops.attention_block(h, delta, 0.22, n1, n2, 1e-6, (wq, wk, wv, wo), rope.cos, rope.sin, B, start,
                                           kc, vc, 0.015625, ws)
        kr, vr = cache[0].clone(), cache[1].clone()
        h1, x = ops.add_norm(h, n1, 1e-6, delta, 0.22)
        q, k, v = (torch.nn.functional.linear(x, w) for w in (wq, wk, wv))
        o = ops.attention(q, k, v, rope.cos, rope.sin, B, start, kr, vr, 0.015625)
        want_h, want_x = ops.add_norm(h1, n2, 1e-6, torch.nn.functional.linear(o, wo), 0.22)
        for a, b, most in ((kc, kr, 2.0 ** -7), (vc, vr, 2.0 ** -7), (got_h, want_h, 2.0 ** -7), (got_x, want_x, 2.0 ** -6)):
            a, b = a.double(), b.double()
            # one bf16 step of the element (or of the rotation's other half), seldom
            assert ((a - b).abs() <= most * b.abs() + 2.0 ** -7 * b.abs().mean()).float().mean() > 0.999
            assert float((a - b).norm() / b.norm()) <= 2e-3


@pytest.mark.parametrize("n,K,cols", [
    (1, 256, (128,)), (33, 1024, (1024, 512, 512)), (64, 1024, (128, 128)), (65, 384, (128, 256, 128)),
    (130, 512, (256,)), (1024, 1024, (1024, 512, 512)), (1025, 1024, (1024, 512, 512)), (4097, 256, (512, 128))])
def test_linear(n, K, cols):
    """Tiles of 64 and of 128 rows, partial last tiles, one to three matrices,
    the shortest K.  Products of bf16 are exact in fp32: K roundings at most of
    sums below |x| |w|, then one to bf16."""
    g = torch.Generator().manual_seed(n + K)
    x = torch.randn(n, K, generator=g).bfloat16().to(DEV)
    ws = [(torch.randn(c, K, generator=g) * 0.02).bfloat16().to(DEV) for c in cols]
    for w, got in zip(ws, ops.linear(x, ws)):
        want = x.double() @ w.double().T.contiguous()
        tol = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T.contiguous())
        assert ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + tol).all()
