"""AnyPrecisionLinear on the GPU: state-dict format, precision switching, both batch branches."""
import os

import numpy as np
import pytest
import torch

from _util import assert_close_gemv, make
from any_precision_amd import packing, synth

pytestmark = pytest.mark.gpu


def _module(L, bias=True, precisions=None):
    from any_precision_amd import AnyPrecisionLinear
    bits = list(range(L.seed_bits, L.parent_bits + 1))
    m = AnyPrecisionLinear(L.K, L.N, bits, bias=bias, precisions=precisions, device="cuda", dtype=torch.float16)
    sd = {k: torch.from_numpy(v) for k, v in packing.pack_layer(L.codes, L.luts).items()}
    if bias:
        sd["bias"] = torch.from_numpy(np.linspace(-1, 1, L.N).astype(np.float16))
    m.load_state_dict(sd)
    return m, sd


def test_state_dict_keys_shapes_dtypes():
    L = make(64, 1056, seed=0)
    m, _ = _module(L)
    sd = m.state_dict()
    assert sorted(sd) == sorted(["qweight", "bias"] + [f"lut{b}" for b in range(3, 9)])
    assert sd["qweight"].shape == (8, 64, 33) and sd["qweight"].dtype == torch.int32
    for b in range(3, 9):
        assert sd[f"lut{b}"].shape == (64, 1 << b) and sd[f"lut{b}"].dtype == torch.float16
    assert m.precision == 8 and m.precisions == list(range(3, 9))


def test_forward_every_branch_and_bias(oracle):
    L = make(128, 4096, seed=1)
    m, sd = _module(L)
    bias = sd["bias"].numpy().astype(np.float64)
    for b in (3, 5, 8):
        for M in (1, 8, 9, 32, 33, 64, 65, 128, 130): # GEMV | fused GEMM (to 128 rows here: 128 x 4096) | dequant + matmul
            x = synth.make_x(M, L.K, seed=M)
            y = m(torch.from_numpy(x).cuda(), precision=b)
            _, want = oracle.matmul_kbit(x, L.qweight, L.luts[b], b, return_f64=True)
            assert y.shape == (M, L.N)
            assert_close_gemv(y, want + bias, f"b={b} M={M}")


def test_strided_activations_are_accepted_on_every_branch(oracle):
    """A transposed or sliced activation view (as Hugging Face modules hand over now and then) gives the
    result of its dense copy on the GEMV, the fused-GEMM and the dequant + matmul branch alike."""
    L = make(96, 2048, seed=4)
    m, sd = _module(L, bias=False)
    for M in (1, 4, 8, 20, 70):
        x = synth.make_x(M, 2 * L.K, seed=M)
        xg = torch.from_numpy(x).cuda()[:, ::2]                 # every other column: stride 2
        assert not xg.is_contiguous()
        _, want = oracle.matmul_kbit(np.ascontiguousarray(x[:, ::2]), L.qweight, L.luts[4], 4, return_f64=True)
        assert_close_gemv(m(xg, precision=4), want, f"strided M={M}")
        xt = torch.from_numpy(np.ascontiguousarray(x[:, ::2].T)).cuda().T    # transposed view of a [K, M] tensor
        assert not xt.is_contiguous() or M == 1
        assert_close_gemv(m(xt, precision=4), want, f"transposed M={M}")


def test_set_precision_and_prune(oracle):
    L = make(32, 1024, seed=2)
    m, _ = _module(L, bias=False, precisions=[3, 4, 6])
    assert m.precision == 6
    with pytest.raises(RuntimeError):
        m.set_precision(8)
    m.prune_precisions()
    assert m.qweight.shape[0] == 6
    assert not hasattr(m, "lut8") and not hasattr(m, "lut5") and hasattr(m, "lut4")
    x = synth.make_x(2, L.K)
    for b in (3, 4, 6):
        m.set_precision(b)
        _, want = oracle.matmul_kbit(x, L.qweight, L.luts[b], b, return_f64=True)
        assert_close_gemv(m(torch.from_numpy(x).cuda()), want, f"b={b}")


def test_constructor_errors():
    from any_precision_amd import AnyPrecisionLinear
    with pytest.raises(RuntimeError):
        AnyPrecisionLinear(64, 8, [3, 4], dtype=torch.float32)
    with pytest.raises(RuntimeError):
        AnyPrecisionLinear(64, 8, [3, 4], precisions=(3, 4))


def test_forward_group_equals_module_by_module(oracle):
    """forward_group (one launch where the dot-product kernel serves the set, a launch per member otherwise, module
    by module beyond 8 rows) against the modules called one by one: the oracle's values at the path's bar, with
    and without biases, joined or as a list."""
    from any_precision_amd.linear import forward_group, forward_swiglu
    layers = [make(n, 4096, seed=70 + n) for n in (256, 64, 64)]
    for bias in (False, True):
        mods = [_module(L, bias=bias)[0] for L in layers]
        for b in (3, 8):
            for rows in (1, 3, 6, 8, 9):
                print(f"forward_group bias={bias} b={b} rows={rows}", flush=True)
                x = synth.make_x(rows, 4096, seed=rows)
                xg = torch.from_numpy(x).cuda()
                outs = forward_group(mods, xg, b)
                joined = forward_group(mods, xg, b, concat=True)
                assert joined.shape == (rows, 384) and torch.equal(joined, torch.cat(outs, dim=-1))
                for L, m, got in zip(layers, mods, outs):
                    _, want = oracle.matmul_kbit(x, L.qweight, L.luts[b], b, return_f64=True)
                    if bias:
                        want = want + m.bias.double().cpu().numpy()
                    assert_close_gemv(got, want, f"forward_group bias={bias} b={b} rows={rows} N={L.N}")
    # SiLU(gate) * up through the one-launch form (up to 4 rows) and through its fallback
    gate, up = _module(layers[1], bias=False)[0], _module(layers[2], bias=False)[0]
    for rows in (2, 6):
        xg = torch.from_numpy(synth.make_x(rows, 4096, seed=9)).cuda()
        got = forward_swiglu(gate, up, xg, 4)
        want = torch.nn.functional.silu(gate(xg, precision=4).float()) * up(xg, precision=4).float()
        assert (got.float() - want).abs().max().item() <= 1e-2 * want.abs().max().item()


def test_forward_takes_the_tiled_gemm_up_to_256_rows_at_3_and_4_bits(oracle):
    """A linear of 4096 rows of a multiple of 128 elements: up to 6 bits go through the fused GEMM up to 256 activation
    rows (3 bits up to 512), 6 bits beyond 256 rows and anything beyond 512 through dequant + matmul; all against the
    oracle."""
    from any_precision_amd.linear import fused_gemm_pays
    L = make(4096, 256, seed=5)
    m, _ = _module(L, bias=False)
    assert fused_gemm_pays(200, 4096, 3, 256) and fused_gemm_pays(256, 4096, 4, 256)
    assert fused_gemm_pays(200, 4096, 5, 256) and fused_gemm_pays(200, 4096, 6, 256) and not fused_gemm_pays(257, 4096, 6, 256)
    assert fused_gemm_pays(257, 4096, 3, 256) and not fused_gemm_pays(513, 4096, 3, 256)
    for b, M in ((3, 200), (3, 256), (4, 256), (5, 200), (6, 200), (6, 257), (8, 256), (3, 257), (3, 513)):
        print(f"linear tiled b={b} M={M}", flush=True)
        x = synth.make_x(M, L.K, seed=M)
        y = m(torch.from_numpy(x).cuda(), precision=b)
        _, want = oracle.matmul_kbit(x, L.qweight, L.luts[b], b, return_f64=True)
        assert_close_gemv(y, want, f"b={b} M={M}")


def test_forward_group_beyond_32_rows_is_one_tiled_launch(oracle):
    """Sets of linears on 9..256 rows go through gemm_kbit_group (one launch of the tiled kernel) where fused_set_pays
    says so, with biases added afterwards; against the oracle, joined or as a list."""
    from any_precision_amd.linear import forward_group, fused_set_pays
    assert fused_set_pays(128, [4096, 4096, 4096], 3, 4096) and fused_set_pays(256, [11008, 11008], 5, 4096)
    assert fused_set_pays(128, [11008, 11008], 8, 4096) and not fused_set_pays(129, [11008, 11008], 8, 4096)
    assert fused_set_pays(256, [4096, 4096, 4096], 8, 4096)
    assert fused_set_pays(128, [4096, 1024, 1024], 8, 4096) and fused_set_pays(9, [4096, 4096], 3, 4096)
    assert not fused_set_pays(32, [11008, 11008], 3, 4096) and not fused_set_pays(8, [4096, 4096], 3, 4096)
    assert fused_set_pays(16, [8192, 1024, 1024], 8, 8192) and not fused_set_pays(16, [8192, 8200], 8, 8192)
    assert fused_set_pays(257, [4096, 4096], 3, 4096) and not fused_set_pays(257, [4096, 4096], 4, 4096)
    assert not fused_set_pays(513, [4096, 4096], 3, 4096) and not fused_set_pays(300, [11008, 11008], 3, 4096)
    assert not fused_set_pays(64, [4096, 4096], 3, 4000)
    layers = [make(n, 256, seed=80 + n) for n in (4096, 512, 520)]
    for bias in (False, True):
        mods = [_module(L, bias=bias)[0] for L in layers]
        for b, rows in ((3, 40), (8, 64), (5, 200), (8, 200), (3, 300)):
            print(f"forward_group tiled bias={bias} b={b} rows={rows}", flush=True)
            x = synth.make_x(rows, 256, seed=rows)
            xg = torch.from_numpy(x).cuda()
            outs = forward_group(mods, xg, b)
            joined = forward_group(mods, xg, b, concat=True)
            assert joined.shape == (rows, 5128) and torch.equal(joined, torch.cat(outs, dim=-1))
            for L, m, got in zip(layers, mods, outs):
                _, want = oracle.matmul_kbit(x, L.qweight, L.luts[b], b, return_f64=True)
                if bias:
                    want = want + m.bias.double().cpu().numpy()
                assert_close_gemv(got, want, f"forward_group tiled bias={bias} b={b} rows={rows} N={L.N}")
    # 9..32 rows: sets whose members all have fewer than 8192 rows of at least 1024 elements (tiles of 16 or 32 rows)
    layers = [make(n, 1024, seed=90 + n) for n in (4096, 200)]
    mods = [_module(L, bias=False)[0] for L in layers]
    for b, rows in ((3, 12), (6, 20), (8, 32)):
        print(f"forward_group narrow tiles b={b} rows={rows}", flush=True)
        x = synth.make_x(rows, 1024, seed=rows)
        outs = forward_group(mods, torch.from_numpy(x).cuda(), b)
        for L, got in zip(layers, outs):
            _, want = oracle.matmul_kbit(x, L.qweight, L.luts[b], b, return_f64=True)
            assert_close_gemv(got, want, f"forward_group narrow tiles b={b} rows={rows} N={L.N}")


@pytest.mark.parametrize("M", [1, 8, 16, 200, 600])
@pytest.mark.parametrize("kind", ["assigned", "over a buffer", "loaded", "parametrised", "buffer", "none again"])
def test_a_bias_of_any_kind_is_added(kind, M):
    """A bias may be a buffer, a parameter (assigned, or loaded with assign=True) or the result of a parametrisation: linears
    and sets of them give the product plus what ``module.bias`` is.  The rows cover every branch of the dispatch."""
    from any_precision_amd.linear import forward_group
    L = make(64, 1024, seed=6)
    plain, _ = _module(L, bias=False)
    m, sd = _module(L, bias=kind not in ("assigned", "none again"))
    value = torch.linspace(-3, 3, L.N).half()
    if kind == "loaded":
        m.load_state_dict({**{k: v.cuda() for k, v in sd.items()}, "bias": torch.nn.Parameter(value.cuda())}, assign=True)
    elif kind == "parametrised":
        class Doubled(torch.nn.Module):
            def forward(self, t):
                return 2 * t
        m.bias.copy_(value / 2)
        torch.nn.utils.parametrize.register_parametrization(m, "bias", Doubled())
    elif kind == "buffer":
        m.bias.copy_(value)
    else:
        m.bias = torch.nn.Parameter(value.cuda())
        if kind == "none again":
            m.bias, value = None, torch.zeros_like(value)
    x = torch.from_numpy(synth.make_x(M, L.K, seed=M)).cuda()
    product = plain(x, precision=4)
    want = product + value.cuda()
    # a set may take another kernel than its member alone: fp32 sums in another order, one unit of fp16 before the bias is
    # added and one after
    bound = 2.0 ** -9 * (product.float().abs() + value.cuda().float().abs()) + 2.0 ** -20
    for got in (m(x, precision=4), forward_group((m, m), x, 4)[1], forward_group((plain, m), x, 4, concat=True)[:, L.N:]):
        assert bool(((got.float() - want.float()).abs() <= bound).all())


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("M", [4, 600])
def test_torch_operations_of_a_linear_are_seen_by_subclasses_and_modes(M, bias):
    """Where the forward takes torch's product (many rows) or adds a bias, a tensor subclass and a torch-function mode see them."""
    from torch.overrides import TorchFunctionMode
    L = make(64, 1024, seed=8)
    m, _ = _module(L, bias=bias)
    x = torch.from_numpy(synth.make_x(M, L.K, seed=M)).cuda()
    want = m(x, precision=4)

    class Marked(torch.Tensor):
        pass

    got = m(x.as_subclass(Marked), precision=4)
    assert type(got) is (Marked if M == 600 else torch.Tensor) and torch.equal(got.as_subclass(torch.Tensor), want)
    seen = []

    class Watching(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(getattr(func, "__name__", ""))
            return func(*args, **(kwargs or {}))

    with Watching():
        got = m(x, precision=4)
    assert torch.equal(got, want) and ("matmul" in seen) == (M == 600) and ("__iadd__" in seen or "add_" in seen) == bias
    m.bias = m.bias.as_subclass(Marked) if bias else None
    assert torch.equal(m(x, precision=4).as_subclass(torch.Tensor), want)


class _Raised(Exception):
    pass


@pytest.mark.parametrize("bias", [False, True])
def test_exceptions_below_a_linear_come_out_as_themselves(bias):
    """A saved-tensor hook's and a dispatch mode's exception, and exhausted memory, keep their types; a non-reentrant checkpoint
    (which ends its second forward by raising in a hook) gives the gradient."""
    from torch.utils._python_dispatch import TorchDispatchMode
    from torch.utils.checkpoint import checkpoint
    from any_precision_amd.linear import AnyPrecisionLinear, forward_group
    L = make(64, 1024, seed=6)
    m, _ = _module(L, bias=bias)
    x = torch.from_numpy(synth.make_x(600, L.K, seed=1)).cuda()          # enough rows for torch's product

    def raising(*_):
        raise _Raised

    with pytest.raises(_Raised), torch.autograd.graph.saved_tensors_hooks(raising, lambda t: t):
        m(x.clone().requires_grad_(), precision=4)

    class Raising(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            raise _Raised

    with pytest.raises(_Raised), Raising():
        m(x, precision=4)
    grads = []
    for kept in (True, False):
        leaf = x.clone().requires_grad_()
        step = lambda t: m(torch.sin(t), precision=4)
        (step(leaf) if kept else checkpoint(step, leaf, use_reentrant=False)).float().square().sum().backward()
        grads.append(leaf.grad)
    assert torch.equal(*grads)
    wide = [AnyPrecisionLinear(1024, 65536, [3], bias=bias, device="cuda", dtype=torch.float16) for _ in range(2)]
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + 2 ** 23) / torch.cuda.mem_get_info()[1])
    held = []
    try:
        with pytest.raises(torch.OutOfMemoryError):
            while True:                 # what is free inside the allocator's segments, in blocks of the smallest result
                held.append(torch.empty((200, 65536), dtype=torch.float16, device="cuda"))
        for call in (lambda: wide[0](x), lambda: forward_group(wide, x), lambda: wide[0](x[:200])):
            with pytest.raises(torch.OutOfMemoryError):
                call()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)


@pytest.mark.parametrize("rows", [1, 4, 40])
@pytest.mark.parametrize("concat", [1, "yes", np.True_, 0, None, np.False_])
def test_concat_is_taken_for_what_it_is_as_a_truth_value(rows, concat):
    from any_precision_amd.linear import forward_group
    L = make(64, 1024, seed=6)
    m, _ = _module(L, bias=False)
    x = torch.from_numpy(synth.make_x(rows, L.K, seed=rows)).cuda()
    want = forward_group((m, m), x, 4, concat=bool(concat))
    got = forward_group((m, m), x, 4, concat=concat)
    assert type(got) is type(want) and torch.equal(torch.cat(tuple(got)), torch.cat(tuple(want)))


@pytest.mark.parametrize("rows,K", [(1, 1024), (4, 1024), (40, 1056), (600, 1024)])
def test_a_mode_sees_the_results_of_a_set_joined(rows, K):
    """Where the results of forward_group are joined by torch, a torch-function mode sees it."""
    from torch.overrides import TorchFunctionMode
    from any_precision_amd.linear import forward_group
    L = make(64, K, seed=6)
    m, _ = _module(L, bias=False)
    x = torch.from_numpy(synth.make_x(rows, K, seed=rows)).cuda()
    want = forward_group((m, m), x, 4, concat=True)
    seen = []

    class Watching(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(getattr(func, "__name__", ""))
            return func(*args, **(kwargs or {}))

    with Watching():
        got = forward_group((m, m), x, 4, concat=True)
    assert torch.equal(got, want) and ("cat" in seen) == (rows > 1)


@pytest.mark.parametrize("N,K", ((1999, 2720), (7, 32), (64, 4096), (1024, 4096), (4096, 11008), (33, 40000)))
def test_a_bias_in_the_launch_is_the_bias_added_afterwards(N, K):
    """Every kernel that takes the bias along, and those that leave it: bit for bit the sum of the bias-free result and the bias."""
    from any_precision_amd import AnyPrecisionLinear, _capi
    lin = AnyPrecisionLinear(K, N, [3, 5, 8], bias=True, device="cuda", dtype=torch.float16)
    g = torch.Generator(device="cuda").manual_seed(N)
    lin.qweight.copy_(torch.randint(-2**31, 2**31, lin.qweight.shape, dtype=torch.int32, device="cuda", generator=g))
    for b in (3, 5, 8):
        lin._buffers[f"lut{b}"].copy_(torch.randn((N, 1 << b), device="cuda", generator=g) * 0.02)
    bias = (torch.randn(N, device="cuda", generator=g) * 4).half()
    bias[0], bias[N - 1] = float("inf"), 60000.0
    lin.bias.copy_(bias)
    for M in (1, 2, 3, 5, 8, 9, 16, 31, 40, 100, 200):
        x = torch.randn((M, K), device="cuda", generator=g).half()
        for b in (3, 5, 8):
            print(f"bias N={N} K={K} M={M} b={b}", flush=True)
            got = lin(x, precision=b)
            lin.bias = None
            want = lin(x, precision=b)
            del lin.bias
            lin.register_buffer("bias", bias.clone())
            assert torch.equal(got, want + bias), (N, K, M, b)
    assert _capi.lib.ap_linear_bias(None, None, None, None, None, 1, 8, 32, 3, None, None) == _capi.AP_ENULL


# (N, K, rows, bits, knobs, added): the dot-product, K-split and block-tile kernels take the bias along; the row-streaming, fine, 4x4x4,
# row-walking and tiled kernels and launches in chunks leave it to the caller
@pytest.mark.parametrize("N,K,M,b,knobs,added", (
    (1999, 2720, 3, 6, {}, 1), (1024, 4096, 1, 4, {}, 1), (512, 2048, 8, 5, {"matmul_mfma4": 0, "matmul_mfma_from": 9}, 1),
    (1024, 4096, 16, 4, {"gemm_block": 0, "gemm_tiled": 0, "gemm_walk": 0}, 1), (1024, 4096, 8, 4, {"matmul_mfma4": 0, "matmul_mfma_from": 4}, 1),
    (4096, 4096, 128, 5, {"gemm_block": 2}, 1), (1999, 2720, 300, 6, {"gemm_block": 2}, 1),
    (14336, 4096, 8, 8, {"matmul_mfma4": 2}, 0), (4096, 4096, 2, 8, {"gemv_stream": 2}, 0), (1024, 4096, 4, 4, {"gemv_fine": 2}, 0),
    (14336, 4096, 16, 8, {"gemm_block": 0, "gemm_tiled": 0, "gemm_walk": 2}, 0),
    (4096, 4096, 128, 5, {"gemm_block": 0, "gemm_tiled": 2}, 0), (1024, 2720, 200, 5, {"gemm_block": 0}, 0)))
def test_which_kernels_take_the_bias_along(N, K, M, b, knobs, added):
    import ctypes
    import any_precision_ext as ext
    from any_precision_amd import _capi
    g = torch.Generator(device="cuda").manual_seed(N + M)
    q = torch.randint(-2**31, 2**31, (b, N, K // 32), dtype=torch.int32, device="cuda", generator=g)
    t = (torch.randn((N, 1 << b), device="cuda", generator=g) * 0.02).half()
    x, bias = torch.randn((M, K), device="cuda", generator=g).half(), (torch.randn(N, device="cuda", generator=g) * 4).half()
    out, flag = torch.empty((M, N), dtype=torch.float16, device="cuda"), ctypes.c_int(-1)
    with _capi.tuning(**knobs):
        rc = _capi.lib.ap_linear_bias(x.data_ptr(), q.data_ptr(), t.data_ptr(), bias.data_ptr(), out.data_ptr(), M, N, K, b,
                                      torch.cuda.current_stream().cuda_stream, ctypes.byref(flag))
        want = (ext.matmul_kbit if M <= 8 else ext.gemm_kbit)(x, q, t, b)
    assert rc == 0 and flag.value == added
    assert torch.equal(out, want + bias if added else want)


SMALL = [(3719, 416, 66, 4), (611, 992, 120, 6), (756, 512, 373, 3), (300, 704, 82, 4)]      # N, K, rows, bits


def _small(N, K, M, b):
    from any_precision_amd.linear import AnyPrecisionLinear
    m = AnyPrecisionLinear(K, N, [b], bias=False, device="cuda", dtype=torch.float16)
    g = torch.Generator(device="cuda").manual_seed(N)
    m.qweight.copy_(torch.randint(-2**31, 2**31, m.qweight.shape, dtype=torch.int32, device="cuda", generator=g))
    table = m._buffers[f"lut{b}"]
    table.copy_(torch.randn(table.shape, device="cuda", generator=g) * 0.02)
    return m, table, torch.randn((M, K), device="cuda", generator=g).half()


# the last three: beyond the line, the pair's calls in both
@pytest.mark.parametrize("N,K,M,b", SMALL + [(717, 256, 248, 7), (2562, 448, 298, 8), (1024, 4096, 320, 8)])
def test_small_linears_take_one_form_in_a_graph_and_outside(N, K, M, b):
    """The fused kernel's bits within the line of ap_gemm_kbit_quick, the pair's beyond, with gradients and for a subclass; a captured call is the
    one that warmed it up, whichever replays."""
    import any_precision_ext as ext
    from any_precision_amd import _capi
    quick = (N, K, M, b) in SMALL
    assert _capi.lib.ap_gemm_kbit_taken(M, N, K, b) == 0 and _capi.lib.ap_gemm_kbit_quick(M, N, K, b) == quick
    m, table, x = _small(N, K, M, b)
    pair = torch.matmul(x, ext.dequant_kbit(m.qweight, table, b).T)
    want = ext.gemm_kbit(x, m.qweight, table, b) if quick else pair
    assert torch.equal(m(x, precision=b), want)
    grad = m(x.clone().requires_grad_(), precision=b)
    assert grad.requires_grad and torch.equal(grad.detach(), pair)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = m(x, precision=b)
    for _ in range(3):
        y.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)


def test_a_module_s_own_call_is_all_the_warm_up_that_its_capture_needs():
    """In a fresh process: nothing but the module has run before it is captured, on either side of the line."""
    import subprocess
    import sys
    code = f"""
import sys
sys.path[:0] = {sys.path!r}
import torch
from test_gpu_linear import SMALL, _small
for case in (SMALL[0], (2562, 448, 298, 8)):
    m, _, x = _small(*case)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        want = m(x, precision=case[3])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = m(x, precision=case[3])
    for _ in range(3):
        y.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want), case
print("captured")
"""
    res = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100, cwd=os.path.dirname(os.path.abspath(__file__)))
    assert res.returncode == 0 and "captured" in res.stdout, res.stdout + res.stderr


def test_where_the_fused_form_is_quick():
    """No GPU is asked: never beyond its range, everything that ap_gemm_kbit_taken takes, and errors as there."""
    from any_precision_amd import _capi
    for N in (64, 255, 256, 1024, 4096, 14336):
        for K in (32, 256, 1024, 4096, 14336):
            for M in (1, 33, 128, 129, 512, 2048, 16384):
                for b in (3, 5, 8):
                    taken, quick = _capi.lib.ap_gemm_kbit_taken(M, N, K, b), _capi.lib.ap_gemm_kbit_quick(M, N, K, b)
                    assert quick == 1 if taken == 1 else quick in (0, 1) and (quick == 0 or (N >= 256 and M * K * N < 2**34))
    assert _capi.lib.ap_gemm_kbit_quick(0, 256, 256, 4) < 0 and _capi.lib.ap_gemm_kbit_quick(64, 256, 250, 4) < 0
    with _capi.tuning(gemm_block=0):
        assert all(_capi.lib.ap_gemm_kbit_quick(M, N, K, b) == _capi.lib.ap_gemm_kbit_taken(M, N, K, b) for N, K, M, b in SMALL)
