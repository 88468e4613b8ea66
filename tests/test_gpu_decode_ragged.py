"""The fused decode step over batches of ragged sequences, whose chunks are
numbered one after another over the sequences (chunks first, or the streams of
a layer and KV head first where there are few long chunks; the longest cut
finer where the lengths differ): every sequence of the batch
against the same step run on it alone (the same arithmetic over another cut of
its positions), the appended rows bit for bit, and the array-backed entry
point, which cuts a batch no finer than its array holds.

Bound: a chunk's partial sums are fp32; another cut reorders at most n sums of
values bounded by max |v|: n 2^-23 max |v|, n the positions.
"""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from tinymetalagent_amd import attention as A  # noqa: E402

DEV = "cuda"


def _inputs(seqs, layers, ctx, heads, kv, d):
    g = torch.Generator(device=DEV).manual_seed(5)

    def r(*shape):
        return torch.randn(shape, generator=g, device=DEV)

    cos, sin = A.rope_table(ctx, d, 1e6)
    return (r(seqs, layers, heads, d), r(seqs, layers, kv, d), r(seqs, layers, kv, d), cos, sin,
            r(seqs, layers, ctx, kv, d).half(), r(seqs, layers, ctx, kv, d).half())


@pytest.mark.parametrize("layers,heads,kv,d,positions", [
    (1, 14, 2, 64, [0, 31]), (3, 8, 2, 128, [32, 0, 511, 63, 64, 1000]), (2, 4, 1, 64, [700] * 8),
    (1, 2, 2, 128, [(37 * i) % 650 for i in range(64)]), (40, 16, 2, 128, [5, 3000, 255, 256, 257]),
    # streams first: one chunk each, and up to three
    (28, 8, 4, 64, [600, 598, 601, 599, 577, 575, 576, 300, 600, 544]), (28, 8, 4, 128, [1500, 900, 1503, 1501, 31]),
    # cut finer: 8 chunks of the longest
    (28, 8, 4, 64, [2000, 10, 20, 300, 50, 40, 60, 100])])
def test_ragged_batch_matches_each_sequence_alone(layers, heads, kv, d, positions):
    ctx = max(positions) + 1
    q, k, v, cos, sin, kc, vc = _inputs(len(positions), layers, ctx, heads, kv, d)
    kb, vb = kc.clone(), vc.clone()
    got = A.decode_step(q, k, v, cos, sin, kb, vb, positions=positions)
    for s, p in enumerate(positions):
        one = slice(s, s + 1)
        k1, v1 = kc[one].clone(), vc[one].clone()
        want = A.decode_step(q[one].contiguous(), k[one].contiguous(), v[one].contiguous(), cos, sin, k1, v1,
                             position=p)
        assert torch.equal(kb[one], k1) and torch.equal(vb[one], v1), (s, p)
        bound = (p + 1) * 2.0 ** -23 * float(v1[:, :, :p + 1].abs().max()) + 1e-7
        assert float((got[one] - want).abs().max()) <= bound, (s, p)


def test_array_backed_step_takes_a_batch_cut_finer_with_a_workspace():
    """8 chunks of the longest sequence would need 26 MB of partials, the array
    holds 16: the call still runs, on fewer chunks."""
    seqs, layers, heads, kv, d, ctx = 8, 28, 28, 4, 128, 2100
    positions = [2099, 100, 900, 33, 1500, 1, 640, 2048]
    q, k, v, cos, sin, kc, vc = _inputs(seqs, layers, ctx, heads, kv, d)
    kb, vb = kc.clone(), vc.clone()
    want = A.decode_step(q, k, v, cos, sin, kb, vb, positions=positions)
    out = torch.full_like(want, float("nan"))
    A.decode_step_noalloc(q, k, v, cos, sin, kc, vc, positions=positions, out=out)
    assert torch.equal(kb, kc) and torch.equal(vb, vc)
    assert float((out - want).abs().max()) <= ctx * 2.0 ** -23 * float(vc.abs().max())
