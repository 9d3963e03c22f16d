"""fp32 multi-row steps in tiles of rows (``AYK_FLAG_ROW_TILES``): prompts and prefill chunks.

The kernel is compared with the float64 oracle at the sizes where it can go wrong: groups that do and do
not divide a tile, tiles that span requests, contexts around its 16-position steps and its wave split,
block sizes that take one table lookup per step and those that do not, and values that are not finite
where only some rows of a tile see them. The bound is the reference contract's for fp32,
``4 * eps * max|y| + 1e-6``.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from ayaka_amd.enums import ForwardMode, KVLayoutKind
from ayaka_amd.hip import _lib
from ayaka_amd.hip import attention as hip_attention
from ayaka_amd.kvcache import RAW_CODEC, KVBuffers
from oracle import paged
from oracle.numerics import bits_to_f32, f32_to_bits
from tests import test_kv_reach as reach
from tests._support import build_scenario

EPS32 = 2.0**-23

# (rows, context) of each request
STEPS = [
    [(16, 16)],
    [(8, 8), (9, 40), (31, 31), (12, 300)],
    [(150, 150), (8, 1000), (10, 0), (33, 129)],
    [(300, 700)],
]


@pytest.mark.parametrize("head_dim", [64, 128, 256])
def test_row_tiles_read_inside_the_cache(head_dim: int) -> None:
    rng = np.random.default_rng(700 + head_dim)
    for case in range(10):
        bs = reach.BLOCK_SIZES[case % len(reach.BLOCK_SIZES)]
        kv_heads, group = [(2, 4), (3, 3), (1, 20), (4, 1)][case % 4]
        lengths = [int(n) for n in rng.integers(1, 300, size=int(rng.integers(1, 4)))]
        step = reach.Step(rng, lengths, bs, kv_heads, head_dim, False, case % 2, fp32=True)
        rows = [max(1, n // 3) for n in lengths]
        req, pos = reach._rows(step, rows)
        args = reach._common(step, kv_heads * group, len(req), req, pos)
        got = reach._walk(step, lambda lib: lib.ayk_paged_attention_v1(*args, hip_attention.ROW_TILES, None))
        reach._check(step, got, f"row tiles case {case} bs {bs}")


@pytest.mark.parametrize("head_dim", [64, 128])
def test_two_group_row_tiles_read_inside_the_cache(head_dim: int) -> None:
    rng = np.random.default_rng(706 + head_dim)
    for case, bs in enumerate(reach.BLOCK_SIZES):
        kv_heads, group = [(8, 4), (8, 3), (8, 5), (24, 1)][case % 4]
        rows = [532, 19, 26, 140]
        lengths = [600, 200, 26, -(-300 // bs) * bs]
        step = reach.Step(rng, lengths, bs, kv_heads, head_dim, False, case % 2, fp32=True)
        req, pos = reach._rows(step, rows)
        assert hip_attention.row_tile_shape(len(req), kv_heads, group, head_dim)[0] == 32
        args = reach._common(step, kv_heads * group, len(req), req, pos)
        got = reach._walk(step, lambda lib: lib.ayk_paged_attention_v1(*args, hip_attention.ROW_TILES, None))
        reach._check(step, got, f"two-group row tiles case {case} bs {bs}")


def test_the_modelled_tiles_are_the_launched_ones() -> None:
    # the launch model and the library agree on the pairs of a tile: every load of the launch is one of a
    # step that the model counts (16 positions: head_dim / 16 key and head_dim / 16 value loads per lane)
    rng = np.random.default_rng(705)
    for case in range(24):
        head_dim = (64, 128, 256)[case % 3]
        kv_heads, group = [(8, 4), (3, 3), (1, 20), (8, 8), (16, 1)][case % 5]
        lengths = [int(n) for n in rng.integers(1, 200, size=int(rng.integers(1, 60)))]
        step = reach.Step(rng, lengths, 16, kv_heads, head_dim, False, case % 2, fp32=True)
        rows = [max(1, n // (1, 2, 20)[case % 3]) for n in lengths]
        req, pos = reach._rows(step, rows)
        args = reach._common(step, kv_heads * group, len(req), req, pos)
        loads = int(reach._walk(step, lambda lib: lib.ayk_paged_attention_v1(*args, hip_attention.ROW_TILES, None))[2])
        pairs, _ = hip_attention.row_tile_shape(len(req), kv_heads, group, head_dim)
        steps = hip_attention.row_tile_walks(np.array(rows), np.array(lengths), group, pairs, 1)[1].sum()
        assert loads == steps * kv_heads * 64 * head_dim // 8, (case, pairs)
    # two groups from 2 x 256 workgroups of 32 pairs: 504 and 505 rows make 63 and 64 tiles x 8 heads
    assert hip_attention.row_tile_shape(504, 8, 4, 64)[0] == 16 and hip_attention.row_tile_shape(505, 8, 4, 64)[0] == 32


def test_attend_runs_the_launch_that_the_model_picks(monkeypatch: pytest.MonkeyPatch) -> None:
    # with the address walk on nothing launches, so the recorded call can be looked at on the CPU
    monkeypatch.setattr(hip_attention, "stream_handle", lambda device: 0)
    monkeypatch.setattr(hip_attention, "require_buffers", lambda op, buffers: None)
    monkeypatch.setattr(hip_attention, "_workspace", lambda *a: torch.zeros(1 << 24, dtype=torch.uint8))
    monkeypatch.setattr(hip_attention, "_arrivals", lambda *a: torch.zeros(1 << 12, dtype=torch.int32))
    lib = _lib.lib()

    def call(rows: list[int], lengths: list[int], mode: ForwardMode) -> tuple[str, int]:
        s = build_scenario(list(zip(rows, lengths)), heads=9, kv_heads=3, head_dim=64, block_size=16, mode=mode.value)
        meta = hip_attention.plan(mode, torch.tensor(rows), torch.tensor(lengths), torch.from_numpy(s.table), 16)
        q = torch.zeros(sum(rows), 9, 64)
        buffers = KVBuffers(torch.zeros(s.k.shape), torch.zeros(s.k.shape), KVLayoutKind.NHD, RAW_CODEC)
        assert lib.ayk_debug_kv_reach_begin(s.table.size) == 0
        try:
            hip_attention.attend(q, buffers, meta, torch.zeros_like(q), scale=0.125)
        finally:
            assert lib.ayk_debug_kv_reach_end(np.zeros(5, dtype=np.int64).ctypes.data) == 0
        (found,) = meta.plan.launches.values()
        return found.fn.__name__, found.args[-1].value

    assert call([300, 200], [300, 500], ForwardMode.MIXED) == ("ayk_paged_attention_v1", hip_attention.ROW_TILES)
    for rows, mode in (([1] * 40, ForwardMode.MIXED), ([1] * 40, ForwardMode.DECODE)):
        name, flags = call(rows, [200] * 40, mode)
        assert not flags & hip_attention.ROW_TILES, (name, mode)


def test_row_tiles_are_refused_elsewhere() -> None:
    lib = _lib.lib()

    def v1(dtype: int, flags: int, rows: object) -> int:
        return lib.ayk_paged_attention_v1(1, 1, 1, 1, 1, 4, 1, rows, rows, 1, 8, 2, 128, 10, 16, 4, 0, dtype, dtype,
                                          ctypes.c_float(1.0), 1.0, 1.0, flags, None)

    assert v1(1, hip_attention.ROW_TILES, 1) == 1 and b"unknown flags" in lib.ayk_last_error()
    assert v1(3, hip_attention.ROW_TILES, None) == 2 and b"rows with positions" in lib.ayk_last_error()
    assert v1(3, hip_attention.ROW_TILES | 32, 1) == 2


def _f32(a: np.ndarray) -> torch.Tensor:
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).to("cuda:0")


def _full_mantissas(like: np.ndarray, rng: np.random.Generator) -> np.ndarray:
    """float32 normals with all their bits where ``like`` (values of a 16-bit type) is not NaN, so that an
    operand shortened on its way to the products shows: bf16 would move a value by up to 2^-9 of it."""
    fresh = rng.standard_normal(like.shape).astype(np.float32)
    assert np.mean(fresh != bits_to_f32(f32_to_bits(fresh, "bf16"), "bf16")) > 0.99
    return np.where(np.isnan(like), like, fresh)


def _planned(steps, heads: int, kv_heads: int, head_dim: int, block_size: int, layout: str, seed: int):
    """A planned step in tiles, its caches and queries on the GPU, and the oracle's float64 output."""
    s = build_scenario(steps, heads=heads, kv_heads=kv_heads, head_dim=head_dim, block_size=block_size,
                       layout=layout, mode="mixed", seed=seed)
    rng = np.random.default_rng(seed + 1000)
    q, k, v = (_full_mantissas(a, rng) for a in (s.q, s.k, s.v))
    meta = hip_attention.plan(ForwardMode.MIXED, torch.tensor(s.rows, dtype=torch.int32, device="cuda:0"),
                              torch.tensor(s.lengths, dtype=torch.int32, device="cuda:0"),
                              torch.from_numpy(s.table.astype(np.int32)).cuda(), block_size)
    # the tiles whatever the launch model prefers: it leaves short steps to the row kernel
    meta.plan.splits[("row-tiles", kv_heads, heads // kv_heads, head_dim)] = True
    buffers = KVBuffers(_f32(k), _f32(v), KVLayoutKind.NHD if layout == "nhd" else KVLayoutKind.HND, RAW_CODEC)
    expected = paged.attention(q, k, v, s.table, np.asarray(s.lengths), scale=s.scale, layout=layout,
                               request_of_row=s.plan["request_of_row"], positions=s.plan["positions"],
                               precision=np.float64)
    return s, meta, buffers, _f32(q), expected


def _assert_matches(steps, heads: int, kv_heads: int, head_dim: int, block_size: int, layout: str,
                    seed: int) -> None:
    s, meta, buffers, q, expected = _planned(steps, heads, kv_heads, head_dim, block_size, layout, seed)
    out = torch.full_like(q, 7.0)
    for _ in range(2):  # recorded, then replayed
        hip_attention.attend(q, buffers, meta, out, scale=s.scale)
    torch.cuda.synchronize()
    got = out.double().cpu().numpy()
    bound = 4 * EPS32 * float(np.abs(expected).max()) + 1e-6
    assert np.isfinite(got).all(), steps
    assert float(np.abs(got - expected).max()) <= bound, steps


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kv_heads,head_dim", [(9, 3, 64), (32, 8, 64), (8, 2, 128), (5, 5, 128), (20, 1, 128),
                                                     (16, 8, 256), (6, 2, 256)])
@pytest.mark.parametrize("block_size,layout", [(16, "nhd"), (24, "hnd"), (5, "nhd"), (1, "hnd")])
def test_row_tiles_match_the_oracle(heads: int, kv_heads: int, head_dim: int, block_size: int, layout: str) -> None:
    for n, steps in enumerate(STEPS):
        _assert_matches(steps, heads, kv_heads, head_dim, block_size, layout, 710 + n)


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kv_heads,head_dim,block_size,layout",
                         [(32, 8, 64, 16, "nhd"), (24, 8, 64, 5, "hnd"), (32, 8, 128, 24, "hnd"), (40, 8, 128, 16, "nhd")])
def test_two_group_row_tiles_match_the_oracle(heads: int, kv_heads: int, head_dim: int, block_size: int,
                                              layout: str) -> None:
    # a border between a tile's two 16-pair groups (532 rows of 4 heads), tiles that hold two requests'
    # rows and padding rows, a ragged last tile
    steps = [(532, 560), (9, 0), (19, 200), (26, 26), (100, 250)]
    rows = sum(count for count, _ in steps)
    assert hip_attention.row_tile_shape(rows, kv_heads, heads // kv_heads, head_dim)[0] == 32
    _assert_matches(steps, heads, kv_heads, head_dim, block_size, layout, 730)


@pytest.mark.gpu
@pytest.mark.parametrize("head_dim,steps,pairs", [(64, [(40, 70)], 16), (256, [(40, 70)], 16), (64, [(600, 630)], 32),
                                                  (128, [(600, 630)], 32)])
def test_values_that_are_not_finite_reach_only_the_rows_that_see_them(head_dim: int, steps, pairs: int) -> None:
    heads, kv_heads = (32, 8) if pairs == 32 else (8, 2)
    assert hip_attention.row_tile_shape(steps[0][0], kv_heads, 4, head_dim)[0] == pairs
    s, meta, buffers, q, _ = _planned(steps, heads, kv_heads, head_dim, 16, "nhd", 720)
    clean, out = torch.empty_like(q), torch.empty_like(q)
    hip_attention.attend(q, buffers, meta, clean, scale=s.scale)
    at = 53  # the rows are positions 30 up; rows before position 53 do not see it
    block, offset = int(s.table[0][at // 16]), at % 16
    buffers.v[block, offset, 0, 3] = float("inf")
    buffers.v[block, offset, 1, 5] = float("nan")
    hip_attention.attend(q, buffers, meta, out, scale=s.scale)
    torch.cuda.synchronize()
    before = at - 30
    # a step with such a value sums its positions one by one, in another order than the clean one:
    # the contract's bound on each side of the exact result
    bound = 2 * (4 * EPS32 * float(clean.abs().max()) + 1e-6)
    assert float((out[:before] - clean[:before]).abs().nan_to_num(float("inf")).max()) <= bound
    assert torch.isinf(out[before:, :4, 3]).all() and torch.isnan(out[before:, 4:8, 5]).all()
    kept = torch.ones(head_dim, dtype=torch.bool, device="cuda:0")
    kept[3] = False
    others = (out[before:, :4] - clean[before:, :4])[:, :, kept]
    assert float(others.abs().nan_to_num(float("inf")).max()) <= bound
    assert torch.equal(out[:, 8:], clean[:, 8:])
