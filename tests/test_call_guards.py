"""Calls that must be refused before anything is launched, on the CPU: the tensors on "the GPU" are fake ones, which have a device
and sizes and no memory."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from randumb_amd import SillyLinear, _lib, ops


def _fake(*shape, dtype=torch.float32, device="cuda:0"):
    with FakeTensorMode():
        return torch.empty(*shape, dtype=dtype, device=device)


IN, OUT, K = 768, 96, 32


# ------------------------------------------------------------------------------------------------ every tensor on x's device
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("elsewhere", ["cpu", "cuda:1"])
@pytest.mark.parametrize("which", ["coefs", "scale_bias", "bias", "bias_coef", "bias_scale"])
@pytest.mark.parametrize("entry", ["one_call", "projected", "vector"])
def test_a_tensor_on_another_device_is_refused(entry, which, elsewhere, dtype):
    """A layer that was never moved, or whose bias was not: an exception, not an address of another memory in a kernel."""
    ext = _lib.extension()
    where = {n: elsewhere if n == which else "cuda:0" for n in ("coefs", "scale_bias", "bias", "bias_coef", "bias_scale")}

    def t(name, *shape):
        return torch.zeros(*shape, dtype=dtype) if where[name] == "cpu" else _fake(*shape, dtype=dtype, device=where[name])

    x = _fake(4, IN, dtype=dtype)
    c = t("coefs", K) if entry == "vector" else t("coefs", OUT, K)
    sb = t("scale_bias", 1)
    bias = (t("bias_coef", K), t("bias_scale", 1), 7) if which.startswith("bias_") else (t("bias", OUT), None, -1)
    with pytest.raises(NotImplementedError if elsewhere == "cpu" else RuntimeError, match="CPU implementation" if elsewhere == "cpu" else "cuda:1"):
        if entry == "one_call":
            ext.linear_one_call(x, c, IN, OUT, IN, 1, 3, sb, *bias)
        elif entry == "projected":
            ext.linear_projected(x, c, IN, OUT, 3, *bias, sb)
        else:
            ext.linear_vector(x, c, IN, OUT, 3, sb, *bias)


def test_embedding_with_coefficients_elsewhere_is_refused():
    with pytest.raises(NotImplementedError, match="CPU implementation"):
        _lib.extension().embed_rows(_fake(3, dtype=torch.int64), torch.zeros(K), 8, 1)
    with pytest.raises(RuntimeError, match="cuda:1"):
        _lib.extension().embed_rows(_fake(3, dtype=torch.int64), _fake(K, device="cuda:1"), 8, 1)


def test_a_layer_that_was_not_moved_is_refused():
    layer = SillyLinear(IN, OUT, [K, K], [1, 2], matrix_coef=True)
    with pytest.raises(NotImplementedError, match="CPU implementation"):
        ops.linear(_fake(4, IN), layer.weight_coef, IN, OUT, IN, 1, 1, None, None)


@pytest.mark.parametrize("name", ["scale_bias", "bias"])
def test_the_operators_refuse_a_host_scale_or_bias(name):
    from randumb_amd import hip

    kw = {name: torch.zeros(OUT if name == "bias" else 1)}
    with pytest.raises(NotImplementedError, match="CPU implementation"):
        hip.linear_fwd(_fake(4, IN), _fake(OUT, K), IN, OUT, IN, 1, 3, **kw)
