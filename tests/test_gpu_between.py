"""The kernels between the linears of the Hugging Face Llama modules against the modules' own torch ops in float64, and the
calls that have to stay with the original forwards."""
import copy
import functools
import pickle

import pytest
import torch


def _config(**kw):
    from transformers import LlamaConfig
    return LlamaConfig(**{**dict(hidden_size=64, intermediate_size=96, num_hidden_layers=2, num_attention_heads=4,
                                 num_key_value_heads=2, vocab_size=128, max_position_embeddings=64), **kw})


@pytest.mark.gpu
@pytest.mark.parametrize("B,T,heads,hd", [(1, 1, 1, 16), (2, 3, 5, 48), (3, 33, 4, 64), (1, 130, 32, 128)])
@pytest.mark.parametrize("tables", ["one", "each"])
def test_rope_heads(B, T, heads, hd, tables):
    from any_precision_amd import _capi
    gen = torch.Generator().manual_seed(T + hd)
    x = torch.randn((B, T, heads * hd), generator=gen).half()
    cos, sin = (torch.rand((B if tables == "each" else 1, T, hd), generator=gen).half() for _ in range(2))
    got = _capi.torch_module().rope(x.cuda(), cos.cuda(), sin.cuda())
    x = x.double().view(B, T, heads, hd)
    low, high = x.chunk(2, dim=-1)
    a, b = x * cos.double().unsqueeze(2), torch.cat((-high, low), dim=-1) * sin.double().unsqueeze(2)
    # one rounding to fp16 and two in fp32 of each product
    bound = (a.abs() + b.abs()) * (2.0 ** -11 + 2.0 ** -22) + 2.0 ** -24
    assert got.shape == x.shape and bool(((got.cpu().double() - (a + b)).abs() <= bound).all())


@pytest.mark.gpu
def test_what_is_not_plain_execution_is_left_to_torch():
    from any_precision_amd import _capi
    native = _capi.torch_module()
    x, w = torch.randn((3, 64), device="cuda").half(), torch.ones((64,), device="cuda").half()
    assert native.rmsnorm(x, w, 1e-5).shape == x.shape and native.silu_mul(x, x).shape == x.shape
    wide = torch.randn((3, 128), device="cuda").half()
    for bad in (x.float(), x.cpu(), wide[:, ::2], wide.view(-1)[1:193].view(3, 64), x[:0], x.clone().requires_grad_(),
                torch.nn.Parameter(x.clone())):
        assert native.rmsnorm(bad, w, 1e-5) is None and native.silu_mul(bad, bad) is None
    assert native.rmsnorm(x, torch.nn.Parameter(w.clone()), 1e-5) is None     # gradients wanted
    with torch.no_grad():
        assert native.rmsnorm(x, torch.nn.Parameter(w.clone()), 1e-5) is not None
    assert native.rmsnorm(x, w[:32], 1e-5) is None
    from torch.utils._python_dispatch import TorchDispatchMode

    class Counting(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Counting():
        assert native.rmsnorm(x, w, 1e-5) is None
    assert torch.vmap(lambda t: torch.zeros(1, device="cuda") if native.silu_mul(t, t) is None else torch.ones(1, device="cuda"))(x).sum() == 0
    with torch.autograd.forward_ad.dual_level():
        assert native.silu_mul(torch.autograd.forward_ad.make_dual(x, x), x) is None


@pytest.mark.gpu
@pytest.mark.parametrize("kv_heads", [4, 2])
def test_model_forward_with_and_without(kv_heads, monkeypatch):
    """The logits of a model with the kernels and with the original forwards, both against the dense weights in float64; and
    that the kernels served the calls."""
    from transformers.models.llama import modeling_llama
    from any_precision_amd import AnyPrecisionForCausalLM, _capi, between
    config = _config(num_key_value_heads=kv_heads)
    ap = AnyPrecisionForCausalLM.from_config(config, seed=3)
    exact = modeling_llama.LlamaForCausalLM(config).double().eval()
    exact.load_state_dict({k: v.double() for k, v in ap.dense_state_dict(5).items()})
    ids = torch.randint(0, 128, (3, 17), device="cuda")
    mask = torch.ones_like(ids)
    mask[0, :4] = 0
    native, served = _capi.torch_module(), []

    class Counting:
        def __getattr__(self, name):
            def call(*args):
                out = getattr(native, name)(*args)
                if name != "plain" and out is not None:
                    served.append(name)
                return out
            return call

    monkeypatch.setattr(between, "_native", Counting)
    with torch.inference_mode():
        want = exact(ids.cpu(), use_cache=False).logits
        outs = [ap(ids, precision=5, use_cache=False).logits]
        assert sorted(served) == ["rmsnorm"] * 5 + ["rope"] * 4 + ["silu_mul"] * 2          # two layers
        padded = ap(ids, attention_mask=mask, precision=5, use_cache=False).logits
        served.clear()
        outs.append(ap(ids, precision=5, use_cache=True).logits)
        assert sorted(served) == ["rmsnorm"] * 5 + ["silu_mul"] * 2                         # a cache: the module's own attention
        replaced = [m for m in ap.model.modules() if type(m).__module__ == between.__name__]
        assert len(replaced) == 9                                                           # five norms, two MLPs, two attentions
        for m in replaced:
            m.__class__ = type(m).__base__
        served.clear()
        outs.append(ap(ids, precision=5, use_cache=False).logits)
        assert not served
        assert torch.allclose(padded[:, 4:].float(), ap(ids, attention_mask=mask, precision=5, use_cache=False).logits[:, 4:].float(),
                              atol=2e-2, rtol=2e-2)
    # two layers of fp16 activations: a few roundings of 2^-11 each
    for out in outs:
        assert float((out.cpu().double() - want).norm() / want.norm()) < 2.8e-3 * 2 ** 0.5


def test_modules_stay_what_they_are():
    """Names, state-dict keys, copies and pickles on the CPU; the original forward serves CPU tensors."""
    from transformers.models.llama import modeling_llama
    from any_precision_amd import between
    config = _config()
    config._attn_implementation = "sdpa"
    plain = modeling_llama.LlamaForCausalLM(config).eval()
    model = copy.deepcopy(plain)
    between.attach(model)
    assert list(model.state_dict()) == list(plain.state_dict())
    layer = model.model.layers[0]
    assert isinstance(layer.self_attn, modeling_llama.LlamaAttention) and type(layer.self_attn).__name__ == "LlamaAttention"
    assert type(layer.mlp) is not modeling_llama.LlamaMLP
    ids = torch.arange(10).view(2, 5)
    with torch.no_grad():
        want = plain(ids, use_cache=False).logits
        for m in (model, copy.deepcopy(model), pickle.loads(pickle.dumps(model))):
            assert torch.allclose(m(ids, use_cache=False).logits, want, atol=1e-5)
            assert type(m.model.norm) is between.LlamaRMSNorm
    model(ids, use_cache=False).logits.sum().backward()
    plain(ids, use_cache=False).logits.sum().backward()
    for (n, a), (_, b) in zip(model.named_parameters(), plain.named_parameters()):
        assert torch.allclose(a.grad, b.grad, atol=1e-4), n


def _attention(attached):
    from transformers.models.llama import modeling_llama
    from any_precision_amd import between
    config = _config()
    config._attn_implementation = "sdpa"
    torch.manual_seed(5)
    model = modeling_llama.LlamaForCausalLM(config).eval()
    if attached:
        between.attach(model)
    return model.model.layers[0].self_attn


def test_a_trace_of_the_attention_is_the_modules_own():
    """Sizes are tensors under a trace; the replaced forward hands a traced call over."""
    gen = torch.Generator().manual_seed(0)
    x, cos, sin = torch.randn((2, 7, 64), generator=gen), *(torch.rand((2, 7, 16), generator=gen) for _ in range(2))

    class Alone(torch.nn.Module):
        def __init__(self, attention):
            super().__init__()
            self.attention = attention

        def forward(self, x, cos, sin):
            return self.attention(x, (cos, sin))[0]

    with torch.no_grad():
        plain, module = Alone(_attention(False)), Alone(_attention(True))
        want = plain(x, cos, sin)
        traced = torch.jit.trace(module, (x, cos, sin))
        assert torch.equal(traced(x, cos, sin), want) and torch.equal(module(x, cos, sin), want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float64])
def test_attention_on_other_types_and_devices_is_the_modules_own(dtype, monkeypatch):
    """One decision before the projections: the call as a whole goes to the original forward."""
    from transformers.models.llama import modeling_llama
    module = _attention(True).to(dtype)
    calls = []
    stock = modeling_llama.LlamaAttention.forward
    monkeypatch.setattr(modeling_llama.LlamaAttention, "forward", lambda self, *a, **kw: calls.append(1) or stock(self, *a, **kw))
    cos = torch.rand((1, 7, 16)).to(dtype)
    with torch.no_grad():
        module(torch.randn((1, 7, 64)).to(dtype), (cos, cos))
    assert calls == [1]


class _Serving:
    """Stands for the native module on the CPU: serves every call, with torch ops."""
    served = 0

    def plain(self, *tensors):
        return True

    def silu_mul(self, gate, up):
        self.served += 1
        return torch.nn.functional.silu(gate) * up

    def rmsnorm(self, x, weight, eps):
        self.served += 1
        return torch.nn.functional.rms_norm(x, weight.shape, weight, eps)

    def rope(self, x, cos, sin):
        self.served += 1
        x = x.view(*x.shape[:2], -1, cos.shape[-1])
        low, high = x.chunk(2, dim=-1)
        return x * cos.unsqueeze(2) + torch.cat((-high, low), dim=-1) * sin.unsqueeze(2)


@pytest.fixture
def serving(monkeypatch):
    from any_precision_amd import between
    stand_in = _Serving()
    monkeypatch.setattr(between, "_native", lambda: stand_in)
    return stand_in


def _mlp():
    from transformers.models.llama import modeling_llama
    from any_precision_amd import between
    model = modeling_llama.LlamaForCausalLM(_config()).eval()
    between.attach(model)
    return model.model.layers[0].mlp


@pytest.mark.parametrize("change", ["nothing", "torch's class", "a class of that name", "instance forward", "class forward", "hook",
                                    "global hook"])
def test_the_activation_function_is_called_where_it_is_not_plain(serving, monkeypatch, change):
    mlp = _mlp()
    calls = []
    handle = None

    def other(t):
        calls.append(1)
        return t * 3

    if change == "torch's class":
        mlp.act_fn = torch.nn.SiLU()
    elif change == "a class of that name":
        mlp.act_fn = type("SiLU", (torch.nn.Module,), {"forward": lambda self, t: other(t)})()
    elif change == "instance forward":
        mlp.act_fn.forward = other
    elif change == "class forward":
        monkeypatch.setattr(type(mlp.act_fn), "forward", lambda self, t: other(t))
    elif change == "hook":
        handle = mlp.act_fn.register_forward_hook(lambda m, args, out: other(args[0]))
    elif change == "global hook":
        handle = torch.nn.modules.module.register_module_forward_hook(
            lambda m, args, out: other(args[0]) if m is mlp.act_fn else None)
    x = torch.randn((2, 64), generator=torch.Generator().manual_seed(0))
    try:
        with torch.no_grad():
            act = torch.nn.functional.silu if change in ("nothing", "torch's class") else other
            want = mlp.down_proj(act(mlp.gate_proj(x)) * mlp.up_proj(x))
            calls.clear()
            got = mlp(x)
    finally:
        if handle is not None:
            handle.remove()
    assert torch.allclose(got, want, atol=1e-6)
    plain = change in ("nothing", "torch's class")
    assert serving.served == plain and calls == [1] * (not plain)


@pytest.mark.parametrize("change", ["nothing", "LlamaRMSNorm", "LlamaMLP", "LlamaAttention", "rotary", "attention function"])
@pytest.mark.parametrize("when", ["before", "after"])
def test_what_a_program_has_replaced_is_called(serving, monkeypatch, change, when):
    """Forwards replaced on the Hugging Face classes, their rotary embedding and a registered attention function."""
    from transformers.models.llama import modeling_llama
    from any_precision_amd import between
    config = _config()
    config._attn_implementation = "sdpa"
    calls = []

    def counted(function):
        @functools.wraps(function)
        def call(*args, **kwargs):
            calls.append(1)
            return function(*args, **kwargs)
        return call

    def replace():
        if change.startswith("Llama"):
            cls = getattr(modeling_llama, change)
            monkeypatch.setattr(cls, "forward", counted(cls.forward))
        elif change == "rotary":
            monkeypatch.setattr(modeling_llama, "apply_rotary_pos_emb", counted(modeling_llama.apply_rotary_pos_emb))
        elif change == "attention function":
            functions = modeling_llama.ALL_ATTENTION_FUNCTIONS
            monkeypatch.setitem(functions._global_mapping, "sdpa", counted(functions["sdpa"]))

    between._class.cache_clear()        # the classes are made anew
    try:
        if when == "before":
            replace()
        model = modeling_llama.LlamaForCausalLM(config).eval()
        between.attach(model)
        if when == "after":
            replace()
        with torch.no_grad():
            model(torch.arange(10).view(2, 5), use_cache=False)
    finally:
        between._class.cache_clear()
    assert len(calls) == {"nothing": 0, "LlamaRMSNorm": 5}.get(change, 2)
    # of two layers: five norms, two MLPs, four rotary embeddings
    assert serving.served == 11 - {"LlamaRMSNorm": 5, "LlamaMLP": 2, "LlamaAttention": 4, "rotary": 4}.get(change, 0)


def test_a_rotary_embedding_replaced_by_any_callable_is_called(serving, monkeypatch):
    """Also one that has no hash and no code of its own."""
    from transformers.models.llama import modeling_llama
    stock, calls = modeling_llama.apply_rotary_pos_emb, []

    class Replacement:
        __hash__ = None

        def __call__(self, *args, **kwargs):
            calls.append(1)
            return stock(*args, **kwargs)

    module = _attention(True)
    x, cos = torch.randn((1, 7, 64)), torch.rand((1, 7, 16))
    with torch.no_grad():
        module(x, (cos, cos))
        assert serving.served == 2 and calls == []
        monkeypatch.setattr(modeling_llama, "apply_rotary_pos_emb", Replacement())
        module(x, (cos, cos))
    assert serving.served == 2 and calls == [1]


@pytest.mark.gpu
def test_tensors_whose_memory_is_not_their_value_are_left_to_torch():
    """A lazily negated view and a zero tensor without memory."""
    from any_precision_amd import _capi
    native = _capi.torch_module()
    x, w = torch.randn((3, 64), device="cuda").half(), torch.ones((64,), device="cuda").half()
    tables = torch.ones((1, 3, 64), device="cuda").half()
    zero = torch._efficientzerotensor((3, 64), dtype=torch.float16, device="cuda")
    for odd in (torch._neg_view(x), zero):
        assert native.rmsnorm(odd, w, 1e-5) is None and native.silu_mul(odd, x) is None and native.silu_mul(x, odd) is None
        assert native.rope(odd[None], tables, tables) is None and native.plain(odd) is False
    assert native.plain(x) is True
