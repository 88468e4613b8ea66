"""A short chunk after a long cached prefix through the layer flow, whose
attention splits the keys over workgroups and whose merge writes the output
projection's operand: the operand's bits against fp32 rows and a separate
launch (TE_HIP_PREFILL_DIGITS=0), and the result against one split
(TE_HIP_PREFILL_SPLITS=1) within the attention's own error, both for the flow's
own choice and for a forced count; chunks whose preferred count the flow's
workspace holds, and chunks whose it does not.

That the keys were split shows in the result: not the bits of one split.

Bound against one split: a row's weights are rounded to fp16 against another
reference maximum per split, 2^-11 of the largest |v| at most each way, in the
projection's input; one layer keeps its relative size (the bound is 4 x 2^-11
of the largest output).
"""
import numpy as np
import pytest

import _synth as S

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from tinymetalagent_amd import attention as A  # noqa: E402
from tinymetalagent_amd import layers as LY  # noqa: E402
from tinymetalagent_amd import runtime as R  # noqa: E402

DEV = "cuda"


def _dev(a):
    a = np.ascontiguousarray(a)
    return torch.from_numpy(a.view(np.int16) if a.dtype == np.uint16 else a).to(DEV)


# forced: a count that the workspace's partials hold (max(8 rows, 20 min(rows, 64))
# hidden-wide rows); held: whether they hold the preferred one
@pytest.mark.parametrize("head_dim,batch,base,forced,held", [
    (128, 1, 3000, 19, False), (64, 33, 2500, 19, True), (128, 129, 1900, 7, True), (128, 129, 6000, 9, False),
    (128, 300, 4000, 7, False)])
def test_flow_with_key_splits(head_dim, batch, base, forced, held, monkeypatch):
    layers, heads, kv_heads, ffn = 1, 4, 2, 256
    ctx = base + batch
    one = batch * heads * (head_dim + 2) * 4  # partial bytes of a split
    cap = max(8 * batch, 20 * min(batch, 64)) * heads * head_dim * 4 // one
    preferred = R.load_library().te_hip_attention_prefill_vt_workspace_bytes(
        1, 1, batch, base, ctx, heads, kv_heads, head_dim) // one
    assert 1 < forced <= cap and preferred > 1 and (preferred <= cap) == held
    m = S.synthetic_model(95, 8, layers, heads, kv_heads, head_dim, ffn, 64, ctx, base)
    cos, sin = A.rope_table(ctx, head_dim, 1.0e6)
    x = _dev(S.normal(95, "rows", (batch, m["hidden"])))
    outs = []
    for splits, digits in ((None, "1"), (None, "0"), ("1", "1"), (str(forced), "1"), (str(forced), "0")):
        monkeypatch.setenv("TE_HIP_PREFILL_DIGITS", digits)
        if splits is None:
            monkeypatch.delenv("TE_HIP_PREFILL_SPLITS", raising=False)
        else:
            monkeypatch.setenv("TE_HIP_PREFILL_SPLITS", splits)
        kc, vc = _dev(m["key_cache"]), _dev(m["value_cache"])
        vt = A.value_t_buffer(1, layers, ctx, kv_heads, head_dim)
        A.value_transpose(vc.view(torch.float16).reshape(1, layers, ctx, kv_heads, head_dim), vt, first_position=0,
                          count=base)
        got = LY.prefill_all_layers(_dev(m["mapping"]), m["offsets"], layers, 8, x.clone(), _dev(m["attn_norm"]),
                                    _dev(m["ffn_norm"]), _dev(m["q_bias"]), _dev(m["k_bias"]), _dev(m["v_bias"]), cos,
                                    sin, kc, vc, vt, base, ctx, heads, kv_heads, head_dim, ffn, 1e-6)
        outs.append(got.cpu().numpy())
    auto, auto_rows, unsplit, cut, cut_rows = outs
    assert np.isfinite(auto).all() and np.array_equal(auto, auto_rows) and np.array_equal(cut, cut_rows)
    assert not np.array_equal(auto, unsplit) and not np.array_equal(cut, unsplit)
    bound = 4 * 2.0 ** -11 * np.abs(unsplit).max()
    print(f"d {head_dim} {batch} after {base}: {np.abs(auto - unsplit).max():.3g} "
          f"{np.abs(cut - unsplit).max():.3g} of {bound:.3g}")
    assert np.abs(auto - unsplit).max() <= bound and np.abs(cut - unsplit).max() <= bound
