"""The next RMSNorm's operand formed inside the split-K sums, at hidden widths
around the two passes of 2048 columns that a workgroup takes: one pass full, a
second of 64 columns, the 7B width, two full, and past them (the separate
launches).  Against TE_HIP_GEMM_REDUCE_RMS=0, the same output bits: the sums
are added in the same order and the operand is split from the same values.
"""
import numpy as np
import pytest

import _synth as S

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from tinymetalagent_amd import attention as A  # noqa: E402
from tinymetalagent_amd import layers as LY  # noqa: E402


def _dev(a):
    a = np.ascontiguousarray(a)
    return torch.from_numpy(a.view(np.int16) if a.dtype == np.uint16 else a).to("cuda")


@pytest.mark.parametrize("heads,kv_heads,head_dim", [(16, 2, 128), (33, 3, 64), (28, 4, 128), (32, 2, 128),
                                                     (65, 5, 64)])
@pytest.mark.parametrize("batch", [3, 70])
def test_prefill_wide_rows_fused_norm_bits(heads, kv_heads, head_dim, batch, monkeypatch):
    layers, ffn, base = 2, 2560, 5
    ctx = base + batch
    m = S.synthetic_model(95, 2, layers, heads, kv_heads, head_dim, ffn, 64, ctx, base)
    cos, sin = A.rope_table(ctx, head_dim, 1.0e6)
    x_in = _dev(S.normal(95, "rows", (batch, m["hidden"])))
    outs = []
    for fused in ("1", "0"):
        monkeypatch.setenv("TE_HIP_GEMM_REDUCE_RMS", fused)
        kc, vc = _dev(m["key_cache"]), _dev(m["value_cache"])
        vt = A.value_t_buffer(1, layers, ctx, kv_heads, head_dim)
        A.value_transpose(vc.view(torch.float16).reshape(1, layers, ctx, kv_heads, head_dim), vt,
                          first_position=0, count=base)
        got = LY.prefill_all_layers(_dev(m["mapping"]), m["offsets"], layers, 2, x_in.clone(),
                                    _dev(m["attn_norm"]), _dev(m["ffn_norm"]), _dev(m["q_bias"]), _dev(m["k_bias"]),
                                    _dev(m["v_bias"]), cos.contiguous(), sin.contiguous(), kc, vc, vt, base, ctx,
                                    heads, kv_heads, head_dim, ffn, 1e-6)
        torch.cuda.synchronize()
        outs.append(got.cpu().numpy())
    assert np.isfinite(outs[0]).all() and np.array_equal(outs[0], outs[1])
