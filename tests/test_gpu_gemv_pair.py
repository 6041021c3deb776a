"""The few-row gate / up pair with one block per CU (csrc/gemvp.hip) through a
drafter forward, against the oracle: one to five half tiles of 8 features per
block with a ragged last block, k steps that divide evenly over the eight waves
or leave waves short or idle, 2..8 rows, row-major and fragment-major weights.

Tolerance 1e-5 of the largest value with an fp32 cache: fp32 products summed in
another order (K <= 2560 terms: sqrt(K) 2^-24 = 3e-6 of the sum's own scale).
"""
import numpy as np
import pytest
import torch

from oracle import core

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,inter,rows,frag", [
    (256, 2048, 2, False),   # one half tile per block, one step per wave
    (1056, 2064, 5, True),   # 258 half tiles: two per block; 33 steps: the last wave has none
    (512, 5104, 4, True),    # 638: three per block, the last block short
    (2048, 6144, 8, False),
    (2560, 6400, 4, True),   # 800: four per block, ten steps per wave
    (2048, 9736, 3, False),  # 1217: five per block
])
def test_pair_matches_oracle(cuda, hidden, inter, rows, frag):
    from woodcock_amd import _lib
    from woodcock_amd.config import DrafterConfig
    from woodcock_amd.drafter import Drafter
    from woodcock_amd.runtime import ptr, stream_ptr
    from woodcock_amd.synthetic import random_drafter, to_bits

    cfg = DrafterConfig(hidden_size=hidden, num_layers=1, num_heads=2, num_kv_heads=1, head_dim=128,
                        intermediate_size=inter, vocab_size=64, target_hidden_size=96)
    w = random_drafter(cfg, seed=inter, device=cuda, std=0.03)
    d = Drafter(cfg, dict(w), cuda, torch.float32)
    keep = []
    if frag:
        for name in ("gate", "up"):
            m = w[f"layers.0.mlp.{name}_proj.weight"]
            keep.append(torch.empty_like(m))
            _lib.call("wc_weights_frag", ptr(m), inter, hidden, ptr(keep[-1]), stream_ptr())
            setattr(d.wstruct.layers[0], f"{name}_frag", ptr(keep[-1]))
    od = core.Drafter(cfg.as_dict(), {k: to_bits(v) for k, v in w.items()})
    cache, oc = d.make_cache(64), od.make_cache(64)
    g = torch.Generator(device=cuda).manual_seed(rows)
    feat = torch.randn(rows, hidden, generator=g, device=cuda)
    tok = torch.randint(0, cfg.vocab_size, (rows,), generator=g, device=cuda)
    hid, out = d(tok, feat, cache)
    ohid, oout = od.forward(tok.cpu().numpy(), feat.cpu().numpy(), oc)
    for got, want in ((hid, ohid), (out, oout)):
        assert np.abs(got.cpu().numpy().astype(np.float64) - want).max() <= 1e-5 * np.abs(want).max()
