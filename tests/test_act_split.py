"""The prompt GEMM's activations as two bf16 values, hi = RNE(x 2^-13) and
lo = RNE(x 2^-13 - hi): |x - (hi + lo) 2^13| <= 2^-17 |x| from 2^-104 on, and
<= 2^-121 + 2^-136 below (lo is then a subnormal bf16, 2^-133 apart, and
x 2^-13 a subnormal fp32).  hi keeps 8
significant bits, so the rest is up to 2^-8 |x|, of which lo keeps 8 again.

On the host the split alone, at ties, binade edges and random values of every
exponent; on the device the kernel's, through weights that pick out one
activation each (code 1, scale 1: every product and sum is exact).
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")


def _values():
    rng = np.random.default_rng(2)
    one = np.float32(1)
    m = np.concatenate([
        rng.uniform(1, 2, 40), [1, 1 + 2 ** -7, 1 + 2 ** -8, 1 + 2 ** -9 + 2 ** -17, 1 + 2 ** -8 + 2 ** -16,
                                1 + 2 ** -8 + 2 ** -17, 2 - 2 ** -8, 2 - 2 ** -9, 2 - 2 ** -8 + 2 ** -17],
        [np.nextafter(one, np.float32(2)), np.nextafter(np.float32(2), one)]]).astype(np.float32)
    x = np.ldexp(m[None, :], np.arange(-149, 128)[:, None]).astype(np.float32).ravel()
    x = np.concatenate([x, -x, np.float32([0.0, -0.0, np.finfo(np.float32).max])])
    return np.resize(x, -(-x.size // 64) * 64).reshape(-1, 64)


def _split(x):
    t = torch.from_numpy(x) * 2.0 ** -13
    hi = t.bfloat16().float()
    return hi.double().numpy(), (t - hi).bfloat16().double().numpy()


def _error_and_bound(x, got):
    x = x.astype(np.float64)
    return np.abs(got - x), np.where(np.abs(x) >= 2.0 ** -104, 2.0 ** -17 * np.abs(x), 2.0 ** -121 + 2.0 ** -136)


def test_two_bf16_values_hold_16_bits():
    x = _values()
    hi, lo = _split(x)
    err, bound = _error_and_bound(x, (hi + lo) * 2.0 ** 13)
    assert np.isfinite(err).all() and np.all(err <= bound)
    # and no better: 1 + 2^-9 + 2^-17 is off by nearly 2^-17 of itself
    big = np.abs(x) >= 2.0 ** -104
    assert (err[big] / np.abs(x[big])).max() > 0.99 * 2.0 ** -17


@pytest.mark.gpu
def test_kernel_splits_activations_into_two_bf16_values():
    from tinymetalagent_amd import runtime as R

    lib = R.load_library()
    x = _values()
    rows, k = x.shape
    w = np.zeros((k, k // 32, 34), np.uint8)
    w[:, :, :2] = np.frombuffer(np.float16(1).tobytes(), np.uint8)
    for j in range(k):
        w[j, j // 32, 2 + j % 32] = 1
    dw, dx = torch.from_numpy(w.ravel()).cuda(), torch.from_numpy(x).cuda()
    out = torch.empty(rows, k, device="cuda")
    act = torch.empty(lib.te_hip_gemm_act_bytes(rows, k), dtype=torch.uint8, device="cuda")
    R.check(lib.te_hip_gemm_q_f32(dw.data_ptr(), 8, dx.data_ptr(), None, None, 1e-6, 0, rows, k, k, out.data_ptr(),
                                  None, act.data_ptr(), None, 0, None))
    got = out.cpu().numpy().astype(np.float64)
    hi, lo = _split(x)
    err, bound = _error_and_bound(x, got)
    print(f"max error / bound {(err / bound).max():.3f}")
    assert np.all(err <= bound)
    assert np.array_equal(got, (hi + lo) * 2.0 ** 13)
