"""The matrix-core chunked prefill for fp32 caches and head dims other than 128
(prefill_tiled.hip), and the key ranges of calls with few query blocks (prefill_split.h), at the
edges of its tiles: 32 and 128 pairs per workgroup, 32, 64 and 128 keys per tile, every head-dim
instantiation with and without padded dims.

Tolerance: bf16 rounds the output once (at most 2^-8 of it: 8 bits) and holds the weights to 2^-17, so
the sums are within 2^-17 * max|v| < 5e-5 plus fp32 summation: 1e-4. fp32: 2e-5, as for every kernel.
"""
import numpy as np
import pytest
import torch

from _util import ATOL, make_case, to_np
from modelcore_amd import _ext
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
@pytest.mark.parametrize("rows,T_new,heads", [(7, 129, 19), (3, 65, 29), (5, 129, 64), (1, 33, 131)],
                         ids=["pairs-266", "keys-261", "pairs-640", "keys-262"])
def test_every_block_of_more_than_one_round_of_workgroups_is_written(dtype, rows, T_new, heads):
    """Blocks past the first 256 are dealt the other way round in steps of 8, with a rest."""
    print("case: tiled rounds", dtype, rows, T_new, heads, flush=True)
    c = make_case([11 * b for b in range(rows)], T_new, heads, heads, 32, T_new + 11 * rows, dtype,
                  seed=43)
    _close(_run(c, -1), _oracle(c, -1), dtype)


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


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D", [8, 40, 64, 96, 136, 192, 256])
@pytest.mark.parametrize("seqlens,T_new,window", [([0, 60], 70, -1), ([120, 190], 9, 64), ([600, 1100], 20, -1)],
                         ids=["steps", "window", "ranges"])
def test_redone_pairs_keep_their_other_values(dtype, D, seqlens, T_new, window):
    """Pairs that see an infinite value are redone 64 keys a step: at the steps' edges, the dims with
    the infinity and all the others."""
    print("case: redone", dtype, D, seqlens, T_new, window, flush=True)
    c = make_case(seqlens, T_new, 4, 2, D, max(seqlens) + T_new + 3, dtype, seed=51)
    dims = [1, D - 1]
    ref = _oracle(c, window)
    for b, s0 in enumerate(seqlens):  # a value that every query of the row sees
        at = s0 if window < 0 else s0 + T_new - 1 - window
        rows = c["v"][b, at - s0] if at >= s0 else c["v_cache"][b, at]
        rows[0, dims] = float("inf")
    out = _run(c, window)
    rest = [d for d in range(D) if d not in dims]
    assert torch.isposinf(out[:, :, :2][..., dims]).all()
    _close(out[..., rest], ref[..., rest], dtype)
    _close(out[:, :, 2:], ref[:, :, 2:], dtype)


@pytest.mark.parametrize("seqlens,T_new,H,H_kv,D,T_max", [
    ([40, 3], 40, 2, 2, 64, 100),         # the waves over a block's keys
    ([40, 3], 40, 512, 128, 64, 100),     # over its pairs
    ([3000, 1000], 40, 4, 2, 96, 3100),   # key ranges
    ([40, 3], 40, 2, 2, 384, 100),        # head dims above 256
    ([3000, 1000], 40, 4, 2, 128, 3100),  # bf16: prefill_mfma.hip
], ids=["keys", "pairs", "ranges", "wide", "hd128"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_a_nan_key_makes_every_output_that_sees_it_nan(dtype, seqlens, T_new, H, H_kv, D, T_max):
    """As the softmax over its scores does; the keys before it, and other KV heads, keep theirs."""
    print("case: NaN keys", dtype, seqlens, T_new, H, H_kv, D, T_max, flush=True)
    c = make_case(seqlens, T_new, H, H_kv, D, T_max, dtype, seed=46)
    good = _run(c, -1)
    G = H // H_kv
    c["k"][0, 17, 0, 1] = float("nan")                 # a new key: seen by queries 17.. of row 0
    c["k_cache"][1, 2, H_kv - 1, 0] = float("nan")     # a cached one: seen by all of row 1
    out = _run(c, -1)
    assert torch.isnan(out[0, 17:, :G]).all()
    _close(out[0, :17], to_np(good[0, :17]), dtype)
    assert torch.equal(out[0, :, G:], good[0, :, G:])
    assert torch.isnan(out[1, :, H - G:]).all()
    assert torch.equal(out[1, :, :H - G], good[1, :, :H - G])


SPLIT_CASES = [
    # seqlens, T_new, H, H_kv, D, T_max, window
    ([8000], 100, 32, 8, 128, 8200, -1),          # two blocks of queries, many ranges
    ([3000, 17], 40, 12, 12, 64, 3100, -1),       # a long row beside one that is not cut
    ([0, 900], 300, 2, 2, 128, 1300, -1),         # blocks of one to many tiles, from an empty cache
    ([2000, 1500], 30, 4, 1, 256, 2100, -1),
    ([2500], 50, 10, 2, 96, 2600, 1500),          # a window that starts inside the first range
    ([1000, 5], 70, 6, 2, 128, 4000, 700),        # a cache far longer than the rows
    ([511, 512, 513], 2, 4, 4, 72, 516, -1),      # ranges of about the least length
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("seqlens,T_new,H,H_kv,D,T_max,window", SPLIT_CASES)
def test_key_ranges_match_the_oracle(dtype, seqlens, T_new, H, H_kv, D, T_max, window):
    """bf16 at head_dim 128 keeps that kernel's tolerance (its weights are bf16)."""
    print("case: ranges", dtype, seqlens, T_new, H, H_kv, D, T_max, window, flush=True)
    scratch = _ext.lib().mcamd_attn_scratch_bytes(len(seqlens), T_new, H, H_kv, D, T_max, window,
                                                  _ext.dtype_code(dtype))
    assert scratch >= 2 * len(seqlens) * T_new * H * (D + 2) * 4  # at least two ranges
    c = make_case(seqlens, T_new, H, H_kv, D, T_max, dtype, seed=43)
    out, ref = _run(c, window), _oracle(c, window)
    if dtype == torch.bfloat16 and D == 128:
        assert np.abs(to_np(out) - ref).max() <= ATOL[dtype]
    else:
        _close(out, ref, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D", [64, 128])
def test_key_ranges_with_rows_outside_the_cache_and_non_finite_values(dtype, D):
    print("case: ranges, bad rows", dtype, D, flush=True)
    seqlens, T_new, H, H_kv, T_max = [1990, 1200, -1], 33, 4, 2, 2000
    c = make_case([1900, 1200, 0], T_new, H, H_kv, D, T_max, dtype, seed=44)
    good = _run(c, -1)
    c["cache_seqlens"] = torch.tensor(seqlens, dtype=torch.int32)
    c["v_cache"][1, 100, 0, 3] = float("inf")
    out = _run(c, -1)
    assert torch.isnan(out[0]).all() and torch.isnan(out[2]).all()
    assert torch.equal(out[1, :, 2:], good[1, :, 2:])  # the other KV head's queries
    if dtype == torch.float32 or D != 128:
        assert torch.isposinf(out[1, :, :2, 3]).all()
        assert torch.isfinite(out[1, :, :2, :3]).all() and torch.isfinite(out[1, :, :2, 4:]).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("seqlens,T_new,H,H_kv,D,T_max,window", [
    ([1990, 1200, -1, -20, 0, 2003], 33, 4, 2, 128, 2000, -1),   # rows partly and wholly outside
    ([700, 0, 63], 130, 6, 3, 128, 1100, 400),
    ([2500], 2, 32, 8, 128, 2502, -1),                           # the cache's last positions
    ([900, 5], 40, 4, 2, 96, 2000, -1),
])
def test_calls_with_key_ranges_append_bit_for_bit(dtype, seqlens, T_new, H, H_kv, D, T_max, window):
    print("case: ranges, append", dtype, seqlens, T_new, H, H_kv, D, T_max, window, flush=True)
    c = make_case([max(0, min(s, T_max - T_new)) for s in seqlens], T_new, H, H_kv, D, T_max, dtype,
                  seed=47)
    ok = [i for i, s in enumerate(seqlens) if 0 <= s <= T_max - T_new]
    ref = _oracle(c, window)
    c["cache_seqlens"] = torch.tensor(seqlens, dtype=torch.int32)
    assert _ext.lib().mcamd_attn_scratch_bytes(len(seqlens), T_new, H, H_kv, D, T_max, window,
                                               _ext.dtype_code(dtype)) > 0
    g = _gpu(c)
    out = flash_attn.flash_attn_with_kvcache(g["q"], g["k_cache"], g["v_cache"], k=g["k"], v=g["v"],
                                             cache_seqlens=g["cache_seqlens"], causal=True,
                                             window_size=(window, 0))
    assert np.abs(to_np(out[ok]) - ref[ok]).max() <= ATOL[dtype]
    assert torch.isnan(out[[i for i in range(len(seqlens)) if i not in ok]]).all()
    want = {n: c[n].clone() for n in ("k_cache", "v_cache")}
    for b, s in enumerate(seqlens):
        for t in range(T_new):
            if 0 <= s + t < T_max:
                want["k_cache"][b, s + t] = c["k"][b, t]
                want["v_cache"][b, s + t] = c["v"][b, t]
    for n in want:
        assert torch.equal(g[n].cpu(), want[n]), n


def _c_entry(g, dtype, ws, scratch_entry):
    """The C operator on copies of the case's caches; returns its output."""
    B, T_new, H, D = g["q"].shape
    T_max, H_kv = g["k_cache"].shape[1:3]
    kc, vc, out = g["k_cache"].clone(), g["v_cache"].clone(), torch.empty_like(g["q"])
    args = (g["q"].data_ptr(), g["k"].data_ptr(), g["v"].data_ptr(), kc.data_ptr(), vc.data_ptr(),
            g["cache_seqlens"].data_ptr(), out.data_ptr(), B, T_new, H, H_kv, D, T_max, kc.stride(0),
            -1, 1, _ext.dtype_code(dtype))
    tail = (ws.data_ptr() if ws is not None else None, ws.numel() if ws is not None else 0,
            _ext.stream_handle(DEV))
    lib = _ext.lib()
    if scratch_entry:
        st = lib.mcamd_flash_attn_with_kvcache_scratch(*args, 0, 0, *tail)
    else:
        st = lib.mcamd_flash_attn_with_kvcache(*args, *tail)
    _ext.check(st, "C entry")
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("dtype,D", [(torch.float32, 64), (torch.bfloat16, 128)])
def test_the_workspace_of_the_operator_is_left_alone(dtype, D):
    """mcamd_flash_attn_with_kvcache never touches its workspace in a multi-token call, whatever its
    size: a caller may share one between streams. Scratch that is too small leaves the keys whole,
    with the same bits."""
    print("case: ranges, workspace", dtype, D, flush=True)
    c = make_case([2000, 31], 20, 8, 2, D, 2100, dtype, seed=45)
    g = _gpu(c)
    need = _ext.lib().mcamd_attn_scratch_bytes(2, 20, 8, 2, D, 2100, -1, _ext.dtype_code(dtype))
    assert need > 0
    ws = torch.full((2 * need,), 7, dtype=torch.uint8, device=DEV)
    whole = _c_entry(g, dtype, None, False)
    assert torch.equal(_c_entry(g, dtype, ws, False), whole)
    assert (ws == 7).all()
    assert torch.equal(_c_entry(g, dtype, ws[:need - 16], True), whole)
    assert (ws == 7).all()
    cut = _c_entry(g, dtype, ws, True)
    assert not (ws == 7).all()
    assert torch.equal(cut, _run(c, -1))


@pytest.mark.parametrize("seqlens,T_new,H,H_kv,T_max", [([8000], 100, 32, 8, 8200), ([1500, 700], 17, 12, 4, 4000)])
def test_key_ranges_weigh_as_the_whole_walk_does(seqlens, T_new, H, H_kv, T_max):
    """bf16 weights are rounded against the maximum of a block's first tile, in every range of it, so
    cut and whole calls differ by the order of fp32 sums alone, where that moves the output's own
    rounding: by 2^-8 of a value in a few of a thousand, 2e-4 of the norm at most. Weights rounded
    against another maximum differ by about 2^-9 / sqrt(3) each way, 2e-3."""
    dtype, D = torch.bfloat16, 128
    print("case: ranges, weights", seqlens, T_new, H, H_kv, T_max, flush=True)
    c = make_case(seqlens, T_new, H, H_kv, D, T_max, dtype, seed=48)
    c["k_cache"] *= 1.2
    g = _gpu(c)
    need = _ext.lib().mcamd_attn_scratch_bytes(len(seqlens), T_new, H, H_kv, D, T_max, -1, _ext.BF16)
    assert need > 0
    whole = to_np(_c_entry(g, dtype, None, True))
    cut = to_np(_c_entry(g, dtype, torch.empty(need, dtype=torch.uint8, device=DEV), True))
    assert np.linalg.norm(cut - whole) <= 2e-4 * np.linalg.norm(whole)


def test_without_scratch_the_keys_stay_whole():
    """The C entry without a workspace gives the same call within its rounding."""
    print("case: ranges, no scratch", flush=True)
    c = make_case([2000, 31], 20, 8, 2, 64, 2100, torch.float32, seed=45)
    out = _run(c, -1)
    g = _gpu(c)
    whole = torch.empty_like(g["q"])
    st = _ext.lib().mcamd_flash_attn_with_kvcache(
        g["q"].data_ptr(), g["k"].data_ptr(), g["v"].data_ptr(), g["k_cache"].data_ptr(),
        g["v_cache"].data_ptr(), g["cache_seqlens"].data_ptr(), whole.data_ptr(), 2, 20, 8, 2, 64,
        2100, g["k_cache"].stride(0), -1, 1, _ext.F32, None, 0, _ext.stream_handle(DEV))
    _ext.check(st, "no scratch")
    _close(whole, _oracle(c, -1), torch.float32)
    _close(out, _oracle(c, -1), torch.float32)


@pytest.mark.parametrize("dtype,D", [(torch.float32, 64), (torch.bfloat16, 128)])
def test_key_ranges_on_two_streams_and_captured(dtype, D):
    """Each call has scratch of its own: calls that overlap on two streams, and a captured one replayed
    between other calls, give the bits of calls by themselves."""
    print("case: ranges, streams", dtype, D, flush=True)
    T_new, H, H_kv, T_max = 20, 8, 2, 2100
    cases = [_gpu(make_case(s, T_new, H, H_kv, D, T_max, dtype, seed=49 + i))
             for i, s in enumerate(([2000, 31], [900, 1700]))]
    assert _ext.lib().mcamd_attn_scratch_bytes(2, T_new, H, H_kv, D, T_max, -1,
                                               _ext.dtype_code(dtype)) > 0

    def call(g):
        return flash_attn.flash_attn_with_kvcache(g["q"], g["k_cache"], g["v_cache"], k=g["k"],
                                                  v=g["v"], cache_seqlens=g["cache_seqlens"],
                                                  causal=True)

    want = [call(g) for g in cases]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    got = [[], []]
    for _ in range(5):
        for i, st in enumerate(streams):
            with torch.cuda.stream(st):
                got[i].append(call(cases[i]))
    torch.cuda.synchronize()
    for i in range(2):
        for y in got[i]:
            assert torch.equal(y, want[i])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = call(cases[0])
    for _ in range(3):
        y.fill_(float("nan"))
        cases[0]["k_cache"][0, 2000:2000 + T_new] = 0  # the replay appends again
        assert torch.equal(call(cases[1]), want[1])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want[0])
        assert torch.equal(cases[0]["k_cache"][0, 2000:2000 + T_new], cases[0]["k"][0])


@pytest.mark.parametrize("dtype,D", [(torch.float32, 64), (torch.bfloat16, 64), (torch.bfloat16, 128)])
@pytest.mark.parametrize("rows,T_new,pos,H,H_kv", [(8, 512, 0, 12, 12), (12, 40, 1500, 8, 2), (60, 1, 900, 12, 12)],
                         ids=["prompts", "chunks", "decode"])
def test_a_batch_gives_its_rows_what_they_get_alone(dtype, D, rows, T_new, pos, H, H_kv):
    """How a call is cut depends on its batch (waves over keys or pairs, key ranges, split length), so
    not bit for bit: within the rounding of the two."""
    print("case: batched and alone", dtype, D, rows, T_new, pos, H, H_kv, flush=True)
    T_max = pos + T_new + 50
    seqlens = [max(0, pos - 13 * b) for b in range(rows)]
    c = make_case(seqlens, T_new, H, H_kv, D, T_max, dtype, seed=50)
    out = to_np(_run(c, -1))
    for b in (0, rows - 1):
        alone = to_np(_run({n: t[b:b + 1].contiguous() for n, t in c.items()}, -1))
        err = np.abs(out[b:b + 1] - alone)
        if dtype == torch.float32:
            assert err.max() <= 2 * ATOL[dtype]
        elif D == 64:
            assert np.all(err <= np.abs(alone) * 2.0 ** -7 + 2e-4)
        else:
            assert err.max() <= ATOL[dtype]


@pytest.mark.parametrize("dtype,D", [(torch.float32, 64), (torch.bfloat16, 64), (torch.bfloat16, 128)])
def test_a_long_prompt_in_chunks_is_the_prompt_in_one(dtype, D):
    """Past 512 keys chunks are cut into ranges, and their tiles start elsewhere than the prompt's
    blocks: the sums are the same in another order."""
    print("case: chunks of a long prompt", dtype, D, flush=True)
    T, C, H, H_kv = 1536, 128, 8, 4
    c = _gpu(make_case([0], T, H, H_kv, D, T, dtype, seed=52))
    whole = flash_attn.flash_attn_with_kvcache(c["q"], c["k_cache"], c["v_cache"], k=c["k"], v=c["v"],
                                               cache_seqlens=c["cache_seqlens"], causal=True)
    kc, vc = torch.zeros_like(c["k_cache"]), torch.zeros_like(c["v_cache"])
    pos, parts = c["cache_seqlens"].clone(), []
    for a in range(0, T, C):
        parts.append(flash_attn.flash_attn_with_kvcache(
            c["q"][:, a:a + C], kc, vc, k=c["k"][:, a:a + C], v=c["v"][:, a:a + C], cache_seqlens=pos,
            causal=True, advance=C))
    assert torch.equal(kc, c["k_cache"]) and torch.equal(vc, c["v_cache"]) and int(pos) == T
    got, ref = to_np(torch.cat(parts, 1)), to_np(whole)
    if dtype == torch.float32:
        assert np.abs(got - ref).max() <= 2 * ATOL[dtype]
    elif D == 64:
        assert np.all(np.abs(got - ref) <= np.abs(ref) * 2.0 ** -7 + 2e-4)
    else:
        assert np.abs(got - ref).max() <= ATOL[dtype]
