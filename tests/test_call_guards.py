"""Calls that must be refused before anything is launched, on the CPU: the tensors on "the GPU" are fake ones, which have a device
and sizes and no memory."""
import contextlib

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from randumb_amd import SillyLinear, _lib, ops


def _fake(*shape, dtype=torch.float32, device="cuda:0"):
    with FakeTensorMode():
        return torch.empty(shape, dtype=dtype, device=device)


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


@pytest.mark.parametrize("name", ["scale_bias", "bias"])
def test_the_operators_refuse_a_host_scale_or_bias(name):
    from randumb_amd import hip

    kw = {name: torch.zeros(OUT if name == "bias" else 1)}
    with pytest.raises(NotImplementedError, match="CPU implementation"):
        hip.linear_fwd(_fake(4, IN), _fake(OUT, K), IN, OUT, IN, 1, 3, **kw)


# ------------------------------------------------------------------------------------------------ sizes that are the layer's
@pytest.mark.parametrize("fused", [True, False])
@pytest.mark.parametrize("width", [IN + 256, IN - 8, 1])
def test_an_input_of_another_width_is_refused(width, fused, monkeypatch):
    """A 2-D input is passed on as it is: wider ones are not cut, narrower ones not read past their rows."""
    ran = []
    monkeypatch.setattr(ops, "linear", lambda *a: ran.append(a))
    layer = SillyLinear(IN, OUT, [K, K], [1, 2], matrix_coef=fused)
    with pytest.raises((RuntimeError, NotImplementedError)):
        layer(torch.zeros(4, width))
    with pytest.raises((RuntimeError, NotImplementedError)):
        layer(torch.zeros(2, 3, width))
    assert not ran


@pytest.mark.parametrize("entry", ["one_call", "projected", "vector"])
def test_the_entry_points_refuse_sizes_that_are_not_the_layers(entry):
    ext = _lib.extension()

    def call(x=(4, IN), coefs=(K,) if entry == "vector" else (OUT, K), scale=(1,), bias=((OUT,), None, -1)):
        x, c, sb = _fake(*x), _fake(*coefs), _fake(*scale)
        b = tuple(_fake(*v) if isinstance(v, tuple) else v for v in bias)
        if entry == "one_call":
            ext.linear_one_call(x, c, IN, OUT, IN, 1, 3, sb, *b)
        elif entry == "projected":
            ext.linear_projected(x, c, IN, OUT, 3, *b, sb)
        else:
            ext.linear_vector(x, c, IN, OUT, 3, sb, *b)

    for what, args in (("an input", {"x": (4, IN + 256)}), ("an input", {"x": (4, IN - 8)}), ("an input", {"x": ()}), ("coefficients", {"coefs": (2, OUT, K)}),
                       ("a scale", {"scale": (0,)}), ("a bias", {"bias": ((1,), None, -1)}), ("a bias", {"bias": ((OUT + 1,), None, -1)}),
                       ("bias coefficients", {"bias": ((2, K), None, 3)}), ("a bias scale", {"bias": ((K,), (0,), 3)})):
        with pytest.raises(RuntimeError, match=f"cannot take {what} of shape"):
            call(**args)


def test_the_operators_refuse_sizes_that_are_not_the_layers():
    from randumb_amd import hip

    x, c, dy = _fake(4, IN), _fake(OUT, K), _fake(4, OUT)
    one = _fake(1)
    for call in (lambda: hip.linear_fwd(_fake(4, IN + 8), c, IN, OUT, IN, 1, 3), lambda: hip.linear_fwd(x, c, IN, OUT, IN, 1, 3, bias=_fake(OUT - 1)),
                 lambda: hip.linear_bwd_dx(_fake(4, OUT - 8), c, IN, OUT, IN, 1, 3),
                 lambda: hip.linear_bwd_dcoef(dy, _fake(5, IN), K, OUT, IN, OUT, IN, 1, 3), lambda: hip.linear_bwd_dcoef(_fake(4, 8), x, K, OUT, IN, OUT, IN, 1, 3),
                 lambda: hip.linear_project_fwd(x, c, 3, bias=_fake(OUT + 8)), lambda: hip.linear_rbias_fwd_(_fake(3, OUT), x, one, IN, OUT, 3),
                 lambda: hip.linear_rbias_bwd_(_fake(4, IN), dy, _fake(4, OUT), one, IN, OUT, 3, want_scale_bias_grad=True),
                 lambda: hip.linear_bwd_projected(_fake(4, 8), _fake(4, 8), c, IN, 3), lambda: hip.linear_bwd_projected_rbias(_fake(4, 8), _fake(4, 8), None, c, one, IN, 3),
                 lambda: hip.linear_bwd_projected_rbias(dy, _fake(4, 8), _fake(4, 8), c, one, IN, 3, want_scale_bias_grad=True)):
        with pytest.raises(RuntimeError, match="must have"):
            call()


def test_a_bias_of_another_length_or_type_is_left_to_the_general_path():
    """Of a pseudorandom bias the extension module sees coefficients only; a dense one F.linear broadcasts or refuses."""
    from randumb_amd import CreateRandumbTensor

    bias = CreateRandumbTensor(torch.zeros(K), 1, (OUT,))
    assert ops._bias_form(bias, OUT) is not None and ops._bias_form(bias, OUT + 1) is None


# ------------------------------------------------------------------------------------------------ tensors that are not where a layer puts them
def _what_linear_gets(monkeypatch, layer):
    got = {}

    def linear(x, coefs, in_f, out_f, sO, sI, seed, scale_bias, bias):
        got.update(coefs=coefs, bias=bias, seed=seed)
        return x.new_zeros(x.shape[0], out_f)

    monkeypatch.setattr(ops, "linear", linear)
    layer(torch.zeros(4, IN))
    return got


def test_a_parametrized_coefficient_is_used(monkeypatch):
    class Doubled(torch.nn.Module):
        def forward(self, c):
            return 2 * c

    layer = SillyLinear(IN, OUT, [K, K], [1, 2], matrix_coef=True)
    with torch.no_grad():
        layer.weight_coef.normal_()
    before = layer.weight_coef.detach().clone()
    torch.nn.utils.parametrize.register_parametrization(layer, "weight_coef", Doubled())
    got = _what_linear_gets(monkeypatch, layer)
    assert torch.equal(got["coefs"], 2 * before) and got["coefs"].requires_grad


def test_a_pruned_coefficient_is_used(monkeypatch):
    from torch.nn.utils import prune

    layer = SillyLinear(IN, OUT, [K, K], [1, 2], matrix_coef=True)
    with torch.no_grad():
        layer.weight_coef.normal_()
    prune.random_unstructured(layer, "weight_coef", amount=0.5)
    got = _what_linear_gets(monkeypatch, layer)
    assert torch.equal(got["coefs"], layer.weight_coef_orig * layer.weight_coef_mask) and (got["coefs"] == 0).any()


def test_a_coefficient_that_is_a_plain_attribute_is_used(monkeypatch):
    """As in the replicas of nn.DataParallel, whose parameters are attributes."""
    layer = SillyLinear(IN, OUT, [K, K], [1, 2], matrix_coef=True)
    coef = layer.weight_coef.detach().clone()
    del layer._parameters["weight_coef"]
    layer.weight_coef = coef
    assert _what_linear_gets(monkeypatch, layer)["coefs"] is coef


@pytest.mark.parametrize("as_parameter", [True, False])
def test_a_replaced_bias_is_used(as_parameter, monkeypatch):
    layer = SillyLinear(IN, OUT, [K, K], [1, 2], matrix_coef=True)
    dense = torch.nn.Parameter(torch.ones(OUT)) if as_parameter else torch.ones(OUT)
    del layer.bias
    layer.bias = dense
    assert _what_linear_gets(monkeypatch, layer)["bias"] is dense
    layer.bias = None
    assert _what_linear_gets(monkeypatch, layer)["bias"] is None
    assert _what_linear_gets(monkeypatch, SillyLinear(IN, OUT, [K, K], [1, 2], matrix_coef=True, bias=False))["bias"] is None


# ------------------------------------------------------------------------------------------------ modes, transforms, tangents
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("sizes", [(4, 256, 192, 16), (300, 256, 192, 64), (130, 133, 99, 50)])
@pytest.mark.parametrize("inside", [True, False])
def test_fake_tensors_take_the_operators(inside, sizes, dtype):
    """A layer's output with no GPU and no memory: in the mode and out of it."""
    tokens, in_f, out_f, k = sizes
    mode = FakeTensorMode()
    with mode:
        x = torch.empty(tokens, in_f, dtype=dtype, device="cuda", requires_grad=True)
        c = torch.empty(out_f, k, dtype=dtype, device="cuda", requires_grad=True)
        b = torch.empty(out_f, dtype=dtype, device="cuda")
    with mode if inside else contextlib.nullcontext():
        y = ops.linear(x, c, in_f, out_f, in_f, 1, 3, None, b)
    assert y.shape == (tokens, out_f) and y.dtype == dtype and y.device.type == "cuda"


@pytest.mark.parametrize("inside", [True, False])
def test_fake_indices_take_the_embedding_operator(inside):
    mode = FakeTensorMode()
    with mode:
        idx, c = torch.zeros(3, 5, dtype=torch.int64, device="cuda"), torch.empty(K, device="cuda", requires_grad=True)
    with mode if inside else contextlib.nullcontext():
        y = ops.embed_rows(idx, c, 24, 1)
    assert y.shape == (3, 5, 24)


def test_calls_that_do_not_go_past_the_dispatcher():
    """The extension module's methods leave tensors that stand for something else to their callers."""
    ext = _lib.extension()
    x, c, h = _fake(4, IN), _fake(OUT, K), _fake(4, 64, dtype=torch.bfloat16)
    assert ext.linear_one_call(x, c, IN, OUT, IN, 1, 3, None, None, None, -1) is None
    assert ext.linear_projected(x, c, IN, OUT, 3, None, None, -1, None) is None
    assert ext.linear_vector(x, _fake(K), IN, OUT, 3, None, None, None, -1) is None
    assert ext.embed_rows(_fake(3, dtype=torch.int64), _fake(K), 24, 1) is None
    assert ext.rms_norm(h, 1e-6) is None and ext.relu_square(h) is None and ext.add_rms_norm(h, h, 1e-6) is None
    assert ext.cross_entropy(h, _fake(4, dtype=torch.int64), -100) is None
    assert ext.causal_attention(_fake(1, 4, 192, dtype=torch.bfloat16), _fake(32), 1, 1e-6) is None


# ------------------------------------------------------------------------------------------------ blocks whose forward has to run
def test_blocks_whose_call_somebody_replaced_are_called(monkeypatch):
    """RT_GPT hands plain blocks each other's normalisation instead of calling them; whatever has to see the call gets it."""
    from randumb_amd.gpt import RT_Block, RT_GPT, RT_GPTConfig

    model = RT_GPT(RT_GPTConfig(int_dim_gen=iter([8] * 8), seed_gen=iter(range(8)), vocab_size=64, n_layer=2, n_head=2, n_embd=64))
    block = model.h[0]
    assert block._plain()

    class Other(RT_Block):
        pass

    def forward(self, x):
        return x

    with monkeypatch.context() as m:
        m.setattr(RT_Block, "forward", forward)
        assert not block._plain()
    with monkeypatch.context() as m:
        m.setattr(RT_Block, "__call__", forward, raising=False)
        assert not block._plain()
    block.forward = lambda x: x
    assert not block._plain()
    del block.forward
    with monkeypatch.context() as m:
        m.setattr(block, "__class__", Other)
        assert not block._plain()
    for register in ("register_forward_hook", "register_forward_pre_hook", "register_full_backward_hook", "register_full_backward_pre_hook"):
        hook = getattr(block, register)(lambda *a: None)
        assert not block._plain()
        hook.remove()
    assert block._plain()
    block.compile()
    assert not block._plain() and model.h[1]._plain()
