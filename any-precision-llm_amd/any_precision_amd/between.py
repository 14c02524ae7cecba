"""The steps between the linears of a Hugging Face Llama model (any_precision/modules/AnyPrecisionForCausalLM.py:88-97 runs the
modules as they are) through the library's kernels: RMSNorm, SiLU * up and the rotary embedding, one launch each where the
modules take seven, two and eleven passes over memory.

``attach(model)`` gives the norm, MLP and attention modules of a Llama-architecture model subclasses of their classes;
parameters, state-dict keys, sub-modules and hooks stay what they are.  Every such forward hands over to the original one
for whatever it does not serve: gradients, other devices and types, traces, compilation, modes, a key/value cache, an
attention mask, other attention implementations.
"""
from __future__ import annotations

import functools
import os
import sys

import torch
import torch.nn as nn
from torch.nn.modules.module import _has_any_global_hook

from .linear import _capi       # None where the library is not built

# keyword arguments of an attention call that do not change what it computes without a cache and a mask
_IDLE = {"position_ids", "cache_position", "use_cache", "output_attentions", "output_hidden_states", "return_dict"}


def _native():
    return None if _capi is None or torch.compiler.is_compiling() else _capi.torch_module()


def _norm_forward(module, original, hidden_states):
    native = _native()
    out = None if native is None else native.rmsnorm(hidden_states, module.weight, float(module.variance_epsilon))
    return original(hidden_states) if out is None else out


@functools.lru_cache(None)
def _home(package):
    return os.path.dirname(sys.modules[package].__file__) + os.sep


def _unchanged(function, package):
    """Whether ``function`` and everything it wraps is code of ``package``, and not a replacement someone has put in its place."""
    home = _home(package)
    while function is not None:
        code = getattr(function, "__code__", None)
        if code is None or not code.co_filename.startswith(home):
            return False
        function = getattr(function, "__wrapped__", None)
    return True


@functools.lru_cache(None)
def _silu_forwards():
    """The classes of the activation function that silu_mul computes, with their forwards."""
    from transformers import activations
    found = ((nn.SiLU, "torch"), (getattr(activations, "SiLUActivation", None), "transformers"))
    return {c: c.forward for c, package in found if c is not None and _unchanged(c.forward, package)}


def _plain_silu(act):
    """Whether calling ``act`` is SiLU and nothing else: no replaced forward, no hooks of its own or of all modules."""
    d = act.__dict__
    return (type(act).forward is _silu_forwards().get(type(act)) and "forward" not in d and d.get("_compiled_call_impl") is None
            and not (act._forward_hooks or act._forward_pre_hooks or act._backward_hooks or act._backward_pre_hooks)
            and not _has_any_global_hook())


def _mlp_forward(module, original, x):
    native = _native()
    act = module.act_fn
    if native is None or not _plain_silu(act) or not native.plain(x):
        return original(x)
    gate, up = module.gate_proj(x), module.up_proj(x)
    hidden = native.silu_mul(gate, up)
    return module.down_proj(act(gate) * up if hidden is None else hidden)


def _attention_forward(module, original, hidden_states, position_embeddings=None, attention_mask=None, past_key_values=None,
                       **kwargs):
    native = _native()
    llama = sys.modules["transformers.models.llama.modeling_llama"]       # its rotary embedding and its attention functions
    if (native is None or position_embeddings is None or attention_mask is not None or past_key_values is not None
            or not _unchanged(llama.apply_rotary_pos_emb, "transformers")
            or module.training or torch.is_grad_enabled() or hidden_states.dim() != 3
            or module.config._attn_implementation != "sdpa" or not getattr(module, "is_causal", True)
            or kwargs.get("output_attentions") or any(k not in _IDLE and v is not None for k, v in kwargs.items())
            or not native.plain(hidden_states, *position_embeddings)):
        return original(hidden_states, position_embeddings=position_embeddings, attention_mask=attention_mask,
                        past_key_values=past_key_values, **kwargs)
    cos, sin = position_embeddings
    B, T = hidden_states.shape[:2]
    q, k, v = (p(hidden_states) for p in (module.q_proj, module.k_proj, module.v_proj))
    rotated = native.rope(q, cos, sin), native.rope(k, cos, sin)
    q, k, v = (t.view(B, T, -1, module.head_dim).transpose(1, 2) for t in (q, k, v))
    if None in rotated:     # projections that are not this library's
        q, k = llama.apply_rotary_pos_emb(q, k, cos, sin)
    else:
        q, k = (t.transpose(1, 2) for t in rotated)
    # the registered function of that name: torch's attention, or what the program has put in its place
    ctx, weights = llama.ALL_ATTENTION_FUNCTIONS["sdpa"](module, q, k, v, None, dropout=0.0, scaling=module.scaling, **kwargs)
    return module.o_proj(ctx.reshape(B, T, -1)), weights


_FORWARDS = {"LlamaRMSNorm": _norm_forward, "LlamaMLP": _mlp_forward, "LlamaAttention": _attention_forward}


@functools.lru_cache(None)
def _class(name):
    """The class ``name`` of the Hugging Face Llama model with its forward replaced."""
    from transformers.models.llama import modeling_llama
    base, step = getattr(modeling_llama, name), _FORWARDS[name]
    stock = base.forward if _unchanged(base.forward, "transformers") else None

    @functools.wraps(base.forward)
    def forward(self, *args, **kwargs):
        if base.forward is not stock:       # replaced, before or after the class was made
            return base.forward(self, *args, **kwargs)
        return step(self, functools.partial(stock, self), *args, **kwargs)

    return type(name, (base,), {"forward": forward, "__module__": __name__})


def __getattr__(name):      # pickled modules name their class as one of this module
    if name in _FORWARDS:
        return _class(name)
    raise AttributeError(f"module {__name__!r} has no attribute {name!r}")


def attach(model):
    """Gives the modules of a Llama-architecture ``model`` the forwards above."""
    if getattr(model.config, "model_type", None) != "llama":
        return
    for module in model.modules():
        name = type(module).__name__
        if name in _FORWARDS and type(module) is _class(name).__base__:
            module.__class__ = _class(name)
