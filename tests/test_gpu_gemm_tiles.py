"""te_hip_gemm_q_f32 at the edges of its tiles: one row more or less than a
row tile (64 and 128), one column more or less than a weight tile (128), one
block, odd and partial chunks of blocks, K splits with a short last part, and
weights at 2- and 4-byte aligned addresses.

Bound per output, against the fp64 product with the dequantized weights: each
activation is the sum of two bf16 values within 2^-17 of it, the block sums and
their accumulation are fp32 (a term is rounded at most 4 times per MFMA of 16 terms
and once per block and split): (2^-17 + (k / 16 + 40) 2^-24) sum |w x|.
"""
import numpy as np
import pytest

import _synth as S

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from tinymetalagent_amd import runtime as R  # noqa: E402


@pytest.mark.parametrize("rows,n,k,split,shift", [
    (1, 1, 32, False, 0), (64, 127, 64, False, 0), (65, 128, 96, False, 0), (128, 129, 256, False, 0),
    (129, 130, 288, False, 2), (33, 256, 320, False, 4), (193, 96, 512, True, 0), (64, 300, 2080, True, 0),
    (200, 128, 2144, True, 2)])
@pytest.mark.parametrize("ggml_type", [2, 8])
def test_gemm_tile_edges(oracle_mod, ggml_type, rows, n, k, split, shift):
    lib = R.load_library()
    w = S.ggml_tensor(11, f"tw{ggml_type}{n}{k}", ggml_type, n, k, scale=0.05)
    x = S.normal(11, "tx", (rows, k))
    x[:, ::37] *= 300.0
    r = S.normal(11, "tr", (rows, n))
    wf = oracle_mod.dequantize_rows(w, ggml_type, k, n).astype(np.float64)
    exact = x.astype(np.float64) @ wf.T + r
    awx = np.abs(x).astype(np.float64) @ np.abs(wf).T + np.abs(r)
    bound = (2.0 ** -17 + (k / 16 + 40) * 2.0 ** -24) * awx
    dw = torch.zeros(w.size + 64, dtype=torch.uint8, device="cuda")
    dw[shift:shift + w.size] = torch.from_numpy(w).cuda()
    dx, dr = torch.from_numpy(x).cuda(), torch.from_numpy(r).cuda()
    # the words after the last output stay as they are
    out = torch.full((rows * n + 64,), -7.0, device="cuda")
    act = torch.empty(lib.te_hip_gemm_act_bytes(rows, k), dtype=torch.uint8, device="cuda")
    nbytes = 8 * rows * n * 4 if split else 0
    part = torch.empty(max(nbytes, 4), dtype=torch.uint8, device="cuda")
    R.check(lib.te_hip_gemm_q_f32(dw.data_ptr() + shift, ggml_type, dx.data_ptr(), None, None, 1e-6, 0, rows, n, k,
                                  out.data_ptr(), dr.data_ptr(), act.data_ptr(), part.data_ptr() if split else None,
                                  nbytes, None))
    got = out.cpu().numpy()
    assert np.all(got[rows * n:] == -7.0)
    err = np.abs(got[:rows * n].reshape(rows, n) - exact)
    print(f"type {ggml_type} {rows}x{n}x{k}: max err / bound {float((err / bound).max()):.3f}")
    assert np.all(err <= bound)


@pytest.mark.parametrize("rows,n,k", [(1, 1, 64), (31, 96, 64), (65, 129, 96), (200, 300, 512)])
def test_residual_in_place(rows, n, k):
    """The residual added in the GEMM's own stores (one K split) with out ==
    resid, as the layer flow passes it: the bits of separate buffers."""
    lib = R.load_library()
    w = torch.from_numpy(S.ggml_tensor(12, f"rw{n}{k}", 8, n, k, scale=0.05)).cuda()
    x, r = (torch.from_numpy(S.normal(12, name, shape)).cuda() for name, shape in (("rx", (rows, k)), ("rr", (rows, n))))
    act = torch.empty(lib.te_hip_gemm_act_bytes(rows, k), dtype=torch.uint8, device="cuda")

    def gemm(out, resid):
        R.check(lib.te_hip_gemm_q_f32(w.data_ptr(), 8, x.data_ptr(), None, None, 1e-6, 0, rows, n, k, out.data_ptr(),
                                      resid, act.data_ptr(), None, 0, None))
        return out

    want = gemm(torch.empty(rows, n, device="cuda"), r.data_ptr())
    plain = gemm(torch.empty(rows, n, device="cuda"), None)
    here = r.clone()
    assert torch.equal(gemm(here, here.data_ptr()), want) and torch.equal(want, r + plain)
