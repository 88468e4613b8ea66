"""The fused steps' torch wrappers refuse a missing tensor or a wrong dtype with
the package's own error, before any work (no GPU: tensors on the host are
refused too, after their dtypes)."""
import pytest

torch = pytest.importorskip("torch")

from tinymetalagent_amd import attention as A  # noqa: E402
from tinymetalagent_amd.runtime import TinyEngineError  # noqa: E402


def _decode(q, k, v, kc, vc):
    return A.decode_step(q[:, :, 0], k, v, torch.zeros(4, 32), torch.zeros(4, 32), kc, vc,
                         workspace=torch.zeros(64, dtype=torch.uint8))


def _prefill(q, k, v, kc, vc):
    return A.prefill_step(q, k, v, torch.zeros(4, 32), torch.zeros(4, 32), kc, vc)


def _prefill_vt(q, k, v, kc, vc):
    return A.prefill_step_vt(q, k, v, torch.zeros(4, 32), torch.zeros(4, 32), kc, vc,
                             torch.zeros(1, 1, 2, 64, 64, dtype=torch.float16))


@pytest.mark.parametrize("step", [_decode, _prefill, _prefill_vt])
@pytest.mark.parametrize("wrong", [None, "k_new", "v_new", "value_cache", "dtype"])
def test_step_refuses_with_the_packages_error(step, wrong):
    q, k, v = torch.zeros(1, 1, 1, 4, 64), torch.zeros(1, 1, 1, 2, 64), torch.zeros(1, 1, 1, 2, 64)
    kc, vc = torch.zeros(1, 1, 4, 2, 64).half(), torch.zeros(1, 1, 4, 2, 64).half()
    if wrong == "k_new":
        k = None
    elif wrong == "v_new":
        v = None
    elif wrong == "value_cache":
        vc = None
    elif wrong == "dtype":
        k = k.double()
    with pytest.raises(TinyEngineError, match="k_new must be" if wrong == "dtype" else None):
        step(q, k, v, kc, vc)
