"""Decode and window launches at head width 256, whose matrix-core kernel holds one key and one
value buffer and refills each with the next chunk's: contexts at the edges of its 16-position
chunks and of the waves' shares of them, against the float64 oracle."""

from __future__ import annotations

import numpy as np
import pytest

from tests._support import build_scenario
from tests.test_gpu_parity import assert_parity, run_attention

pytestmark = pytest.mark.gpu

#: No context; less than, exactly and just past one chunk; one chunk per wave of 8 and one more;
#: several rounds with a ragged end.
LENGTHS = (0, 1, 15, 16, 17, 127, 128, 129, 401)


@pytest.mark.parametrize("heads", [2, 6, 16])
@pytest.mark.parametrize("launch", [dict(partitions=0, waves=1), dict(partitions=0, waves=8),
                                    dict(partitions=7, partition_size=64)])
def test_decode_chunk_edges(heads: int, launch: dict) -> None:
    s = build_scenario([(1, n) for n in LENGTHS], dtype="bf16", heads=heads, kv_heads=2, head_dim=256,
                       block_size=24, mode="decode", seed=31)
    assert_parity(run_attention(s, qk="mfma", **launch), s.expected(np.float64), "bf16", f"{heads} {launch}")


@pytest.mark.parametrize("launch", [dict(partitions=0), dict(partitions=None, partition_size=64)])
def test_window_chunk_edges(launch: dict) -> None:
    s = build_scenario([(min(n, 4), n) for n in LENGTHS if n], dtype="fp16", heads=4, kv_heads=2, head_dim=256,
                       block_size=16, layout="hnd", seed=32)
    out = run_attention(s, prefill=True, window=True, **launch)
    assert_parity(out, s.expected(np.float64), "fp16", f"windows {launch}")
