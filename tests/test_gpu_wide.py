"""Many-row passes (csrc/wide.hip) and the backend operations on them against
the oracle and 64-bit torch: prompts through the
drafter (fuse and forward) at the edges of the row tiles (16, 128) and of a pass
(1024), few rows over a long context (the keys split over blocks), head sizes with and without the flash attention, both cache types, a
sliding window, two layers.

Tolerances, max |got - want| / max |want|: 1e-5 with an fp32 cache (fp32
products, sums in another order); 1e-3 with a bf16 cache, where a key or value
at a rounding boundary lands one bf16 step (2^-8) off in a sum over many.
"""
import numpy as np
import pytest
import torch

from oracle import core

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.abs(np.asarray(a, np.float64) - np.asarray(b, np.float64)).max() / np.abs(b).max())


@pytest.mark.parametrize("rows,ctx,kv,layers,window,head_dim,heads", [
    (9, 700, torch.float32, 1, None, 128, 4),
    (12, 500, torch.bfloat16, 1, 300, 128, 8),
    (17, 5, torch.float32, 1, None, 128, 4),
    (33, 0, torch.bfloat16, 1, None, 128, 4),
    (40, 70, torch.float32, 2, None, 128, 4),
    (65, 3, torch.bfloat16, 1, 20, 128, 8),
    (128, 0, torch.float32, 1, None, 128, 2),
    (129, 100, torch.float32, 1, 64, 128, 4),
    (35, 9, torch.float32, 1, None, 64, 4),
    (333, 31, torch.bfloat16, 1, None, 128, 4),
    (1030, 2, torch.float32, 1, None, 128, 2),
])
def test_prompt_matches_oracle(cuda, rows, ctx, kv, layers, window, head_dim, heads):
    from woodcock_amd.config import DrafterConfig
    from woodcock_amd.drafter import Drafter
    from woodcock_amd.synthetic import random_drafter, to_bits

    cfg = DrafterConfig(hidden_size=256, num_layers=layers, num_heads=heads, num_kv_heads=2, head_dim=head_dim,
                        intermediate_size=416, vocab_size=500, target_hidden_size=96, window=window)
    w = random_drafter(cfg, seed=rows, device=cuda, std=0.05)
    d = Drafter(cfg, dict(w), cuda, kv)
    od = core.Drafter(cfg.as_dict(), {k: to_bits(v) for k, v in w.items()})
    cap = ctx + rows + 7
    cache, oc = d.make_cache(cap), od.make_cache(cap, kv_bf16=kv == torch.bfloat16)
    g = torch.Generator(device=cuda).manual_seed(rows)
    for li, c in enumerate(cache):
        c.keys[0, :, :ctx] = torch.randn(c.keys[0, :, :ctx].shape, generator=g, device=cuda).to(kv)
        c.values[0, :, :ctx] = torch.randn(c.values[0, :, :ctx].shape, generator=g, device=cuda).to(kv)
        c.keys[0, :, ctx + rows:] = float("nan")  # slots past the prompt are never read
        c.values[0, :, ctx + rows:] = float("nan")
        c.offset = ctx
        oc.k[li][:] = to_bits(c.keys[0]) if kv == torch.bfloat16 else c.keys[0].cpu().numpy()
        oc.v[li][:] = to_bits(c.values[0]) if kv == torch.bfloat16 else c.values[0].cpu().numpy()
    oc.offset = ctx
    taps = [torch.randn(rows, cfg.target_hidden_size, generator=g, device=cuda) for _ in range(3)]
    tok = torch.randint(0, cfg.vocab_size, (rows,), generator=g, device=cuda)
    tol = 1e-5 if kv == torch.float32 else 1e-3
    feat = d.fuse(taps)
    want = od.fuse([t.cpu().numpy() for t in taps])
    assert _rel(feat.cpu().numpy(), want) < 1e-5
    hid, out = d(tok, feat, cache)
    ohid, oout = od.forward(tok.cpu().numpy(), feat.cpu().numpy(), oc)
    assert _rel(hid.cpu().numpy(), ohid) < tol
    assert _rel(out.cpu().numpy(), oout) < tol
    assert cache[0].offset == oc.offset == ctx + rows
    for li, c in enumerate(cache):
        for got, ref in ((c.keys, oc.keys_f32(li)), (c.values, oc.values_f32(li))):
            assert _rel(got[0, :, :ctx + rows].float().cpu().numpy(), ref[:, :ctx + rows]) < max(tol, 4e-3 * (tol > 1e-4))
            assert torch.isnan(got[0, :, ctx + rows:]).all()


@pytest.mark.parametrize("rows", [17, 48, 130])
def test_fuse_gathers_rows_and_bf16_taps(cuda, rows):
    """Gathered, clamped tap rows and bf16 taps give what the gathered fp32 taps give."""
    import ctypes as C

    from woodcock_amd import _lib
    from woodcock_amd.config import DrafterConfig
    from woodcock_amd.drafter import Drafter
    from woodcock_amd.runtime import ptr, stream_ptr
    from woodcock_amd.synthetic import random_drafter

    cfg = DrafterConfig(hidden_size=256, num_layers=1, num_heads=2, num_kv_heads=2, head_dim=128,
                        intermediate_size=416, vocab_size=500, target_hidden_size=96)
    d = Drafter(cfg, random_drafter(cfg, seed=rows, device=cuda), cuda)
    g = torch.Generator(device=cuda).manual_seed(rows)
    taps = [torch.randn(40, 96, generator=g, device=cuda).bfloat16() for _ in range(3)]
    idx = torch.randint(-3, 45, (rows,), generator=g, device=cuda, dtype=torch.int32)
    got = torch.empty(rows, 256, device=cuda)
    tp = (C.c_void_p * 3)(*[t.data_ptr() for t in taps])
    _lib.call("wc_drafter_fuse", C.byref(d.dims), C.byref(d.wstruct), tp, _lib.WC_BF16, 96, ptr(idx), 40, rows, None,
              ptr(got), 256, ptr(d.ws), stream_ptr())
    want = d.fuse([t[idx.long().clamp(0, 39)].float() for t in taps])
    assert torch.equal(got, want)


@pytest.mark.parametrize("wdt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("L,K,N", [(1, 8, 3), (1, 2056, 4100), (2, 520, 7), (3, 512, 33), (7, 4104, 129), (8, 64, 5000),
                                   (9, 32, 1), (16, 96, 50), (17, 2048, 1030), (33, 544, 64), (65, 256, 8200),
                                   (130, 2048, 2048), (600, 128, 6145)])
def test_linear_shapes(cuda, wdt, L, K, N):
    """Row counts around the vector / matrix-core boundary (8 | 9), odd widths and
    outputs, tiles past the last row and column; sums in fp32 against 64 bits."""
    from woodcock_amd import ops

    g = torch.Generator(device=cuda).manual_seed(L * K + N)
    x = torch.randn(L, K, generator=g, device=cuda)
    W = torch.randn(N, K, generator=g, device=cuda).to(wdt)
    y0 = torch.randn(L, N, generator=g, device=cuda)
    want = x.double() @ W.double().T
    # |error| <= a few roundings of the largest partial sum, ~ sqrt(K) for unit inputs
    tol = 8 * 2.0 ** -24 * K ** 0.5 * 4
    pad = torch.full((L * N + 64,), 7.0, device=cuda)
    y = pad[:L * N].view(L, N)
    ops.linear(x, W, y=y)
    assert (y.double() - want).abs().max() < tol * 4
    assert (pad[L * N:] == 7).all()
    acc = y0.clone()
    ops.linear(x, W, y=acc, accumulate=True)
    assert (acc.double() - (y0.double() + want)).abs().max() < tol * 5


@pytest.mark.parametrize("L", [4, 40])
def test_linear_infinities_and_nan(cuda, L):
    """An infinite or NaN entry reaches exactly the outputs it reaches in fp32."""
    from woodcock_amd import ops

    g = torch.Generator(device=cuda).manual_seed(L)
    x = torch.randint(1, 4, (L, 64), generator=g, device=cuda).float()
    W = torch.randint(1, 4, (96, 64), generator=g, device=cuda).bfloat16()
    x[1, 5] = float("inf")
    x[2, 7] = float("nan")
    W[3, 9] = float("-inf")
    got, want = ops.linear(x, W), (x.double() @ W.double().T).float()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.isnan(want).any()
    assert torch.equal(got[~torch.isnan(want)], want[~torch.isnan(want)])


@pytest.mark.parametrize("L,T,H,Hk,masked", [(1, 1, 4, 2, False), (1, 65, 8, 8, False), (3, 257, 4, 1, True),
                                             (20, 33, 8, 2, True), (64, 64, 16, 8, True), (128, 129, 16, 8, True),
                                             (200, 1000, 8, 4, True), (300, 70, 4, 4, False)])
def test_attention_shapes(cuda, L, T, H, Hk, masked):
    """Both head_dim 128 kernels around their limits, masks of unaligned row
    lengths with rows that see one key only, values past the last key untouched."""
    from woodcock_amd import ops

    g = torch.Generator(device=cuda).manual_seed(L * T)
    q = torch.randn(L, H, 128, generator=g, device=cuda)
    K = torch.randn(T + 3, Hk, 128, generator=g, device=cuda)
    V = torch.randn(T + 3, Hk, 128, generator=g, device=cuda)
    K[T:], V[T:] = float("nan"), float("nan")
    K, V = K[:T], V[:T]
    m = None
    if masked:
        m = torch.rand(L, T, generator=g, device=cuda) < 0.5
        m[:, 0] |= ~m.any(dim=1)
        m[0] = False
        m[0, T - 1] = True
    got = ops.attention(q, K, V, m, 0.09)
    kd, vd = (t.double().transpose(0, 1).repeat_interleave(H // Hk, 0) for t in (K, V))
    z = q.double().transpose(0, 1) @ kd.transpose(1, 2).contiguous() * 0.09
    if m is not None:
        z = z.masked_fill(~m[None], -float("inf"))
    want = (torch.softmax(z, dim=2) @ vd).transpose(0, 1)
    # weights of relative error ~ |z| 2^-23 (|z| < 6) against values of unit size
    assert (got.double() - want).abs().max() < 1e-5
