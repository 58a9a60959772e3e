"""The general single-token decode (decode_splitk.hip) at the edges of its splits and chunks, its
own append, and the bf16 / head_dim 128 decode's merge over very many segments, against the float64
oracle within the dtype's tolerance. The appended caches are compared bit for bit."""
import numpy as np
import pytest
import torch

from _util import ATOL, bits, make_case, max_abs, to_np
from modelcore_amd.kernels.flash_attn import flash_attn
from oracle import kv_oracle as ko

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


def _run(c, window, append=True):
    g = {k: v.to(DEV) for k, v in c.items()}
    out = flash_attn.flash_attn_with_kvcache(g["q"], g["k_cache"], g["v_cache"],
                                             k=g["k"] if append else None,
                                             v=g["v"] if append else None,
                                             cache_seqlens=g["cache_seqlens"], causal=True,
                                             window_size=(window, 0))
    torch.cuda.synchronize()
    return out, g


def _oracle(c, window, append=True):
    q, kc, vc = to_np(c["q"]), to_np(c["k_cache"]), to_np(c["v_cache"])
    k, v = (to_np(c["k"]), to_np(c["v"])) if append else (None, None)
    return ko.flash_attn_with_kvcache(q, kc, vc, k, v, c["cache_seqlens"].tolist(), window)[0]


CASES = [
    # seqlens, H, H_kv, D, T_max, window
    ([0, 62, 63, 64, 65, 127, 128], 4, 2, 128, 300, -1),     # fp32: 64-key splits
    ([0, 127, 128, 255, 256, 257], 6, 6, 64, 300, -1),       # fp32: 128; bf16: one split of 256
    ([511, 512, 767, 3], 16, 2, 64, 800, -1),                # G = 8: two keys a chunk
    ([700, 64, 33], 12, 4, 96, 800, 63),                     # padded dims, a window of one split
    ([500, 1], 16, 1, 256, 600, 300),                        # G = 16: two head chunks append once
    ([31, 32, 33], 3, 3, 16, 40, -1),
    ([90, 10], 4, 4, 8, 100, -1),                            # half of each key's two lanes
    ([(7 * i) % 400 for i in range(260)], 8, 8, 8, 400, -1),  # 2080 workgroups of up to 512 keys
    # 64 rows of four splits each at most, most of them shorter
    ([(37 * i) % 1024 for i in range(64)], 16, 16, 16, 1024, -1),
    ([1023] + [i % 5 for i in range(63)], 32, 16, 16, 1024, -1),
]


@pytest.mark.parametrize("append", [True, False], ids=["append", "no-append"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("seqlens,H,H_kv,D,T_max,window", CASES)
def test_split_edges_match_the_oracle(dtype, seqlens, H, H_kv, D, T_max, window, append):
    print("case: splits", dtype, seqlens[:8], H, H_kv, D, T_max, window, append, flush=True)
    c = make_case(seqlens, 1, H, H_kv, D, T_max, dtype, seed=51)
    out, g = _run(c, window, append)
    assert max_abs(to_np(out), _oracle(c, window, append)) <= ATOL[dtype]
    want = (bits(c["k_cache"]), bits(c["v_cache"]))
    if append:
        want = ko.append(*want, bits(c["k"]), bits(c["v"]), seqlens)
    assert np.array_equal(bits(g["k_cache"]), want[0]) and np.array_equal(bits(g["v_cache"]), want[1])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_values_past_the_split_and_infinities(dtype):
    """Stale keys past a row's end are never used; an infinite last value gives an infinite
    output although the chunk's missing keys re-read it; rows outside the cache get NaN."""
    print("case: splits, non-finite", dtype, flush=True)
    seqlens = [70, 200, 299, 300]
    c = make_case([70, 200, 299, 0], 1, 4, 2, 64, 300, dtype, seed=52)
    ref = _oracle(c, -1)
    c["cache_seqlens"] = torch.tensor(seqlens, dtype=torch.int32)
    c["k_cache"][0, 71:] = float("nan")
    c["v_cache"][0, 71:] = float("nan")
    c["v"][1, 0, 0, 7] = float("inf")
    out, g = _run(c, -1)
    assert max_abs(to_np(out[0]), ref[0]) <= ATOL[dtype]
    assert torch.isposinf(out[1, 0, :2, 7]).all() and torch.isfinite(out[1, 0, 2:]).all()
    assert max_abs(to_np(out[1, 0, :, 8:]), ref[1, 0, :, 8:]) <= ATOL[dtype]
    assert torch.isnan(out[3]).all()
    assert torch.equal(g["k_cache"][3].cpu(), c["k_cache"][3])


@pytest.mark.parametrize("seqlens,H,H_kv,T_max,window", [
    ([16000], 32, 8, 16400, -1),       # 128 segments a unit
    ([2500], 4, 1, 2600, -1),          # one unit over the launch, idle KV rows
    ([900, 2000, 5], 10, 2, 2100, 1500),
    ([-1, 3000], 8, 4, 3100, -1),      # a row outside the cache beside one of many segments
])
def test_merge_of_very_many_segments(seqlens, H, H_kv, T_max, window):
    dtype = torch.bfloat16
    print("case: wide merge", seqlens, H, H_kv, T_max, window, flush=True)
    c = make_case([max(s, 0) for s in seqlens], 1, H, H_kv, 128, T_max, dtype, seed=53)
    ref = _oracle(c, window)
    c["cache_seqlens"] = torch.tensor(seqlens, dtype=torch.int32)
    out, _ = _run(c, window)
    ok = [i for i, s in enumerate(seqlens) if s >= 0]
    assert max_abs(to_np(out[ok]), ref[ok]) <= ATOL[dtype]
    assert torch.isnan(out[[i for i, s in enumerate(seqlens) if s < 0]]).all()
    sl = c["cache_seqlens"].to(DEV)
    g = {k: v.to(DEV) for k, v in c.items()}
    moved = flash_attn.flash_attn_with_kvcache(g["q"], g["k_cache"], g["v_cache"], k=g["k"], v=g["v"],
                                               cache_seqlens=sl, causal=True,
                                               window_size=(window, 0), advance=2)
    assert torch.equal(moved[ok], out[ok])
    assert torch.equal(sl.cpu(), c["cache_seqlens"] + 2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T_max,length", [(1024, 512), (2048, 1024), (4096, 2048)])
def test_long_splits_of_large_grids(dtype, T_max, length):
    """4096 (row, KV head)s of two splits: three rows at a split's edges against the oracle."""
    print("case: long splits", dtype, T_max, length, flush=True)
    B, H, D = 64, 64, 16 // dtype.itemsize
    seqlens = [(97 * b) % T_max for b in range(B)]
    seqlens[:4] = [length - 1, length, T_max - 1, length // 2]
    g = torch.Generator(device=DEV).manual_seed(54)
    c = {n: torch.randn(B, T, H, D, generator=g, device=DEV).to(dtype)
         for n, T in (("q", 1), ("k", 1), ("v", 1), ("k_cache", T_max), ("v_cache", T_max))}
    c["cache_seqlens"] = torch.tensor(seqlens, dtype=torch.int32, device=DEV)
    rows = {n: t[:4].clone() for n, t in c.items()}
    out, _ = _run(c, -1)
    assert max_abs(to_np(out[:4]), _oracle(rows, -1)) <= ATOL[dtype]
    assert torch.isfinite(out).all()


def test_a_cache_of_more_positions_than_a_grid_has_blocks_of_2048():
    print("case: 135M positions", flush=True)
    T_max, D = 135_000_000, 8
    c = {n: torch.zeros(1, T, 1, D, dtype=torch.bfloat16, device=DEV)
         for n, T in (("q", 1), ("k", 1), ("v", 1), ("k_cache", T_max), ("v_cache", T_max))}
    g = torch.Generator(device=DEV).manual_seed(55)
    for n in ("q", "k", "v"):
        c[n].normal_(generator=g)
    for n in ("k_cache", "v_cache"):
        c[n][:, :5000].normal_(generator=g)
    c["cache_seqlens"] = torch.tensor([4999], dtype=torch.int32, device=DEV)
    small = {n: t[:, :5000].clone() if n.endswith("cache") else t for n, t in c.items()}
    out, _ = _run(c, -1)
    assert max_abs(to_np(out), _oracle(small, -1)) <= ATOL[torch.bfloat16]


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 256), (torch.float32, 128), (torch.float32, 256)])
@pytest.mark.parametrize("T_max", [1025, 1300], ids=["odd", "even"])
def test_paired_splits_of_wide_rows(dtype, D, T_max):
    """2048 workgroups or more of 512-byte or 1 KB rows: two splits of a head beside each other, an
    odd and an even number of them."""
    print("case: paired splits", dtype, D, T_max, flush=True)
    B, H, H_kv = 64, 16, 8
    seqlens = [(129 * b) % T_max for b in range(B)]
    seqlens[:5] = [255, 256, 511, T_max - 1, 0]
    g = torch.Generator(device=DEV).manual_seed(56)
    c = {n: torch.randn(B, T, h, D, generator=g, device=DEV).to(dtype)
         for n, T, h in (("q", 1, H), ("k", 1, H_kv), ("v", 1, H_kv), ("k_cache", T_max, H_kv),
                         ("v_cache", T_max, H_kv))}
    c["cache_seqlens"] = torch.tensor(seqlens, dtype=torch.int32, device=DEV)
    pick = [0, 1, 2, 3, 4, 13, 63]
    rows = {n: t[pick].clone() for n, t in c.items()}
    out, _ = _run(c, -1)
    assert max_abs(to_np(out[pick]), _oracle(rows, -1)) <= ATOL[dtype]
    assert torch.isfinite(out).all()
