"""The matrix-core chunked prefill for fp32 caches and head dims other than 128
(prefill_tiled.hip), at the edges of its tiles: 32 and 128 pairs per workgroup, 32, 64 and 128
keys per tile, every head-dim instantiation with and without padded dims.

Tolerance: bf16 rounds the output once (at most 2^-8 of it: 8 bits) and holds the weights to 2^-17, so the sums
are within 2^-17 * max|v| < 5e-5 plus fp32 summation: 1e-4. fp32: 2e-5, as for every kernel.
"""
import numpy as np
import pytest
import torch

from _util import ATOL, make_case, to_np
from modelcore_amd.kernels.flash_attn import flash_attn
from oracle import kv_oracle as ko

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)

CASES = [
    # seqlens, T_new, H, H_kv, D, T_max, window
    ([0, 31], 32, 2, 2, 16, 80, -1),            # one whole block of 32 pairs; padded dims
    ([32, 95], 33, 2, 2, 32, 160, -1),          # a second block of one pair
    ([127, 128], 7, 9, 3, 40, 160, -1),         # G = 3: 21 pairs
    ([100, 0, 57], 65, 4, 4, 64, 200, 31),      # a window inside a tile
    ([200], 130, 10, 2, 72, 340, 200),          # G = 5, blocks that start inside a position
    ([0, 64, 129], 43, 6, 2, 96, 200, -1),
    ([63, 1], 64, 4, 1, 128, 130, 0),           # fp32 only takes this kernel; window 0
    ([40], 50, 3, 3, 136, 100, -1),
    ([1000, 17], 20, 4, 4, 192, 1030, 300),
    ([5, 400], 70, 8, 2, 256, 480, -1),
    ([300], 3, 64, 1, 64, 310, -1),             # G = 64
    # At least 512 workgroups of 128 pairs: the waves share the tiles instead of the pairs.
    ([0, 31, 64, 65, 90, 127, 1, 2], 33, 64, 64, 64, 170, -1),
    ([0, 31, 64, 65, 90, 127, 1, 2], 33, 64, 64, 40, 170, 50),
    ([90, 3], 130, 128, 128, 32, 230, -1),
    ([50, 0, 3, 7], 33, 512, 128, 96, 90, -1),  # G = 4: a second block of 4 pairs
    ([50, 0, 3, 7], 33, 128, 128, 128, 90, -1),
]


def _gpu(c):
    return {k: v.to(DEV) for k, v in c.items()}


def _run(c, window):
    g = _gpu(c)
    return flash_attn.flash_attn_with_kvcache(g["q"], g["k_cache"], g["v_cache"], k=g["k"], v=g["v"],
                                              cache_seqlens=g["cache_seqlens"], causal=True,
                                              window_size=(window, 0))


def _oracle(c, window):
    return ko.flash_attn_with_kvcache(*(to_np(c[n]) for n in ("q", "k_cache", "v_cache", "k", "v")),
                                      c["cache_seqlens"].tolist(), window)[0]


def _close(out, ref, dtype):
    err = np.abs(to_np(out) - ref)
    bound = ATOL[dtype] if dtype == torch.float32 else np.abs(ref) * 2.0 ** -8 + 1e-4
    assert np.all(err <= bound), float((err - bound).max())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("seqlens,T_new,H,H_kv,D,T_max,window", CASES)
def test_tile_edges_match_the_oracle(dtype, seqlens, T_new, H, H_kv, D, T_max, window):
    if dtype == torch.bfloat16 and D == 128:
        pytest.skip("bf16 at head_dim 128 runs prefill_mfma.hip")
    print("case: tiled", dtype, seqlens, T_new, H, H_kv, D, T_max, window, flush=True)
    c = make_case(seqlens, T_new, H, H_kv, D, T_max, dtype, seed=41)
    _close(_run(c, window), _oracle(c, window), dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads", [2, 128], ids=["keys-over-waves", "pairs-over-waves"])
def test_infinities_and_nan_reach_only_the_pairs_that_see_them(dtype, heads):
    """Values past a query's position are multiplied by a weight of zero on the matrix cores: a
    pair they would spoil is redone over its own keys. An infinite V gives an infinite output, as
    a plain sum does."""
    print("case: tiled non-finite", dtype, heads, flush=True)
    seqlens, T_new, D, T_max, window = [40, 7, 0, 3], 40, 64, 100, 25
    c = make_case(seqlens, T_new, heads, heads, D, T_max, dtype, seed=42)
    ref = _oracle(c, window)
    plain = _run(c, window)
    c["v"][0, 30, :, 5] = float("nan")    # position 70: seen by queries 30.. of row 0
    c["v"][1, 20, :, 9] = float("inf")    # position 27: seen by queries 20.. of row 1
    c["k"][2, 35, :, 0] = float("nan")    # a masked key of queries 0..34 of row 2
    c["v_cache"][3, 90:] = float("nan")   # past every query of row 3
    out = _run(c, window)
    _close(out[0, :30], ref[0, :30], dtype)
    assert torch.isnan(out[0, 30:, :, 5]).all()
    assert torch.isfinite(out[0, 30:, :, 6:]).all()
    _close(out[1, :20], ref[1, :20], dtype)
    assert torch.isposinf(out[1, 20:, :, 9]).all()
    _close(out[1, 20:, :, 10:], ref[1, 20:, :, 10:], dtype)
    _close(out[2, :35], ref[2, :35], dtype)
    assert torch.equal(out[3], plain[3])
