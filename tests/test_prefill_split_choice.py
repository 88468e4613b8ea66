"""The number of key splits a short chunk takes where one split would be the
rows kernel (at most 512 keys), on the host through the workspace query (256
compute units, as without a device): four for a few rows over the last 128 keys,
one where the rows make the splits' partials dearer or the keys are fewer.
"""
import pytest

from tinymetalagent_amd import runtime as R

SHAPES = {"0.5B": (14, 2, 64), "1.5B": (12, 2, 128), "3B": (16, 2, 128), "7B": (28, 4, 128)}


@pytest.mark.parametrize("shape,tokens,keys,splits", [
    ("7B", 24, 416, 4), ("7B", 32, 480, 4), ("7B", 32, 512, 4), ("7B", 64, 512, 1), ("7B", 24, 384, 1),
    ("3B", 1, 385, 4), ("3B", 48, 448, 4), ("3B", 64, 448, 1), ("3B", 128, 512, 1), ("3B", 32, 256, 1),
    ("1.5B", 32, 400, 4), ("1.5B", 64, 400, 1), ("0.5B", 1, 512, 1)])
def test_splits_of_a_short_chunk(shape, tokens, keys, splits):
    heads, kv, d = SHAPES[shape]
    n = R.load_library().te_hip_attention_prefill_vt_workspace_bytes(1, 1, tokens, keys - tokens, keys, heads, kv, d)
    assert n == (0 if splits == 1 else splits * tokens * heads * (d + 2) * 4)
