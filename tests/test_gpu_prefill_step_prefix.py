"""prefill_step after a cached prefix, whose append launch also builds the V^T
of the prefix: prefixes that end inside, at and past a 32-position block, one
and several (sequence, layer) units; against the same step with a caller's V^T
(the caches and the output bit for bit) on one key split, and with k / v rows or
their biases off 16-byte alignment, which take the separate launches."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from tinymetalagent_amd import attention as A  # noqa: E402

DEV = "cuda"


@pytest.mark.parametrize("seqs,layers,heads,kv,d,tokens,base", [
    (1, 1, 14, 2, 64, 33, 1), (1, 1, 4, 2, 128, 1, 31), (2, 3, 4, 1, 64, 40, 32), (1, 2, 16, 2, 128, 130, 777),
    (1, 1, 4, 4, 64, 600, 95)])
def test_plain_step_after_a_prefix(seqs, layers, heads, kv, d, tokens, base):
    g = torch.Generator(device=DEV).manual_seed(3)

    def r(*shape):
        return torch.randn(shape, generator=g, device=DEV)

    ctx = base + tokens + 3
    q, k, v = r(seqs, layers, tokens, heads, d), r(seqs, layers, tokens, kv, d), r(seqs, layers, tokens, kv, d)
    kb, vb = r(layers, kv * d), r(layers, kv * d)
    kc, vc = r(seqs, layers, ctx, kv, d).half(), r(seqs, layers, ctx, kv, d).half()
    cos, sin = A.rope_table(ctx, d, 1e6)
    vt = A.value_t_buffer(seqs, layers, ctx, kv, d)
    A.value_transpose(vc, vt, first_position=0, count=base)
    k1, v1 = kc.clone(), vc.clone()
    want = A.prefill_step_vt(q, k, v, cos, sin, k1, v1, vt, base_position=base, k_bias=kb, v_bias=vb)
    k2, v2 = kc.clone(), vc.clone()
    got = A.prefill_step(q, k, v, cos, sin, k2, v2, base_position=base, k_bias=kb, v_bias=vb)
    assert torch.equal(k1, k2) and torch.equal(v1, v2) and torch.equal(got, want)
    # one float into a larger buffer: 4-byte aligned rows
    odd = [torch.empty(x.numel() + 1, device=DEV)[1:].view(x.shape).copy_(x) for x in (k, v, kb, vb)]
    k3, v3 = kc.clone(), vc.clone()
    got = A.prefill_step(q, *odd[:2], cos, sin, k3, v3, base_position=base, k_bias=kb, v_bias=vb)
    assert torch.equal(k1, k3) and torch.equal(v1, v3) and torch.equal(got, want)
    k3, v3 = kc.clone(), vc.clone()
    got = A.prefill_step(q, k, v, cos, sin, k3, v3, base_position=base, k_bias=odd[2], v_bias=odd[3])
    assert torch.equal(k1, k3) and torch.equal(v1, v3) and torch.equal(got, want)
