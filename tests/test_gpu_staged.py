"""The staged K-split fused GEMM (up to 32 activation rows): against the oracle at the edges of its range, and which calls reach it."""
import ctypes

import pytest
import torch

from _util import assert_bit_exact, assert_close_gemv, layer_to_gpu, make

gpu = pytest.mark.gpu


@pytest.fixture(scope="module")
def ext():
    import any_precision_ext
    return any_precision_ext


def _x(M, K, seed):
    from any_precision_amd import synth
    x = synth.make_x(M, K, seed=seed)
    return x, torch.from_numpy(x).cuda()


def _staged(Ns, M, K, b):
    from any_precision_amd import _capi
    return _capi.lib.ap_linear_staged(len(Ns), (ctypes.c_int * len(Ns))(*Ns), M, K, b)


# K: a quarter of a step of 512 elements, parts of one behind a whole chunk of 1024 (1152, 2944), fewer steps than waves, as many, a different
# number per wave with the last one short (4224, 11008).  N: one row, one block of 16, no multiple of it.  Rows: the edges of every form.
@gpu
@pytest.mark.parametrize("N,K", ((1, 128), (33, 512), (16, 640), (47, 1152), (64, 2048), (30, 2944), (96, 4096), (21, 4224), (16, 11008)))
def test_agrees_with_the_oracle(ext, oracle, N, K):
    from any_precision_amd import _capi
    L = make(N, K, seed=N + K)
    q, luts = layer_to_gpu(L)
    for b in range(3, 9):
        for M in (1, 4, 5, 8, 9, 16, 17, 32):
            x, xg = _x(M, K, seed=M)
            _, want = oracle.matmul_kbit(x, L.qweight, L.luts[b], b, return_f64=True)
            print(f"staged N={N} K={K} b={b} M={M}", flush=True)
            with _capi.tuning(gemm_staged=2):
                got = ext.gemm_kbit(xg, q, luts[b], b)
            assert_close_gemv(got, want, f"N={N} K={K} b={b} M={M}")


@gpu
def test_one_hot_rows_give_the_weights_exactly(ext, oracle):
    from any_precision_amd import _capi
    N, K = 35, 2048 + 640
    L = make(N, K, seed=5)
    q, luts = layer_to_gpu(L)
    ks = list(range(0, K, 97)) + [255, 511, 512, 1023, 1024, 2047, 2048, 2175, 2176, K - 129, K - 128, K - 1]
    x = torch.zeros((len(ks), K), dtype=torch.float16, device="cuda")
    x[torch.arange(len(ks)), torch.tensor(ks)] = 1.0
    for b in range(3, 9):
        w = oracle.dequant_kbit(L.qweight, L.luts[b], b)
        for rows in (4, 8, 16, 32):
            with _capi.tuning(gemm_staged=2):
                got = torch.cat([ext.gemm_kbit(part.contiguous(), q, luts[b], b) for part in x.split(rows)])
            assert_bit_exact(got.t().contiguous(), w[:, ks], f"one-hot b={b} rows={rows}")


@gpu
@pytest.mark.parametrize("N,K", ((4096, 11008), (14336, 4096), (11008, 4224)))
def test_rings_refilled_on_a_full_chip(ext, N, K):
    """Two or three workgroups a CU that go around their rings, planes from memory: against the product of the dequantised weight, and one-hot
    rows exactly over all weight rows.  A result is fp16 of an fp32 sum: 2**-11 of its value, and 2**-13 of the norm of its K terms for the sums of
    both sides (K roundings of 2**-24 as a random walk are 2**-17 of it at most, 2**-15 the largest of half a million)."""
    from any_precision_amd import _capi
    gen = torch.Generator(device="cuda").manual_seed(N + K)
    q = torch.randint(-2**31, 2**31, (8, N, K // 32), dtype=torch.int32, device="cuda", generator=gen)
    for b in (3, 4, 5, 8):
        table = (torch.randn((N, 1 << b), device="cuda", generator=gen) * 0.02).half()
        w = ext.dequant_kbit(q, table, b)
        for M in (4, 8, 16, 32):
            print(f"staged full chip N={N} K={K} b={b} M={M}", flush=True)
            x = torch.randn((M, K), device="cuda", generator=gen).half()
            ks = torch.randint(0, K, (M,), device="cuda", generator=gen)
            hot = torch.zeros((M, K), dtype=torch.float16, device="cuda")
            hot[torch.arange(M, device="cuda"), ks] = 1.0
            want = x.float() @ w.float().t()
            with _capi.tuning(gemm_staged=2):
                first, exact = ext.gemm_kbit(x, q, table, b), ext.gemm_kbit(hot, q, table, b)
                again = ext.gemm_kbit(x, q, table, b)
            assert ((first.float() - want).abs() <= want.abs() * 2**-11 + 2**-13 * 0.02 * K ** 0.5).all(), (b, M)
            assert torch.equal(first, again) and torch.equal(exact, w[:, ks].t()), (b, M)


@gpu
@pytest.mark.parametrize("K", (1024, 1152))
def test_what_is_not_a_number_stays_in_its_row(ext, K):
    """NaN and infinities in one activation row, infinite table entries that no weight of the row uses."""
    from any_precision_amd import _capi
    N = 40
    for b in (3, 4, 5, 8):
        for M in (3, 7, 13, 29):
            q, luts = layer_to_gpu(make(N, K, seed=b))
            x = torch.randn((M, K), device="cuda").half()
            x[1, 3], x[M - 1, K - 1] = float("nan"), float("inf")
            table = luts[b].clone()
            q[:, 7] = 0         # row 7 uses one code only (all planes 0): the others are infinite
            table[7, 1:] = float("inf")
            w = ext.dequant_kbit(q, table, b)
            with _capi.tuning(gemm_staged=2):
                got = ext.gemm_kbit(x, q, table, b)
            clean = [m for m in range(M) if m not in (1, M - 1)]
            assert torch.isfinite(got[clean]).all(), (K, b, M)
            want = x[clean].float() @ w.float().t()
            assert (got[clean].float() - want).norm() <= 1e-3 * want.norm()      # fp16 results of fp32 sums
            assert torch.isnan(got[1]).all() and not torch.isfinite(got[M - 1]).any()


@gpu
def test_sets_strided_results_bias_and_graphs(ext):
    """Linears that share x in one launch, dense and side by side, bit for bit what each alone gives; a bias in the launch; replays."""
    from any_precision_amd import _capi
    Ns, K = (200, 64, 72, 129), 1280
    for b in (3, 4, 6, 8):
        pairs = [layer_to_gpu(make(N, K, seed=N)) for N in Ns]
        qs, ts = [q for q, _ in pairs], [luts[b] for _, luts in pairs]
        for M in (2, 6, 12, 31):
            x = torch.randn((M, K), device="cuda").half()
            with _capi.tuning(gemm_staged=2):
                singles = [ext.gemm_kbit(x, q, t, b) for q, t in zip(qs, ts)]
                outs = ext.gemm_kbit_group(x, qs, ts, b)
                joint = ext.gemm_kbit_group(x, qs, ts, b, concat=True)
                bias, out, added = torch.randn((Ns[3],), device="cuda").half(), torch.empty((M, Ns[3]), dtype=torch.half, device="cuda"), ctypes.c_int()
                _capi.check(_capi.lib.ap_linear(x.data_ptr(), qs[3].data_ptr(), ts[3].data_ptr(), bias.data_ptr(), out.data_ptr(), M, Ns[3], K,
                                                b, torch.cuda.current_stream().cuda_stream, ctypes.byref(added)), "ap_linear")
                torch.cuda.synchronize()
                g = torch.cuda.CUDAGraph()
                with torch.cuda.graph(g):
                    replayed = ext.gemm_kbit_group(x, qs, ts, b, concat=True)
            assert added.value == 1 and torch.equal(out, singles[3] + bias), (b, M)
            assert all(torch.equal(s, o) for s, o in zip(singles, outs)), (b, M)
            assert torch.equal(joint, torch.cat(singles, dim=-1)), (b, M)
            for _ in range(3):
                replayed.zero_()
                torch.cuda.synchronize()
                g.replay()
                torch.cuda.synchronize()
                assert torch.equal(replayed, joint), (b, M)


@gpu
def test_modules_of_three_to_thirty_two_rows_are_served_by_it():
    """AnyPrecisionLinear and forward_group where the rule takes the kernel: the bits of a forced call."""
    import any_precision_ext as ext
    from any_precision_amd import AnyPrecisionLinear, _capi
    from any_precision_amd.linear import forward_group
    gen = torch.Generator(device="cuda").manual_seed(3)

    def linear(K, N, bias):
        m = AnyPrecisionLinear(K, N, [4, 8], bias=bias, device="cuda", dtype=torch.float16)
        m.qweight.copy_(torch.randint(-2**31, 2**31, m.qweight.shape, dtype=torch.int32, device="cuda", generator=gen))
        for b in (4, 8):
            m._buffers[f"lut{b}"].copy_(torch.randn((N, 1 << b), device="cuda", generator=gen) * 0.02)
        if bias:
            m.bias.copy_(torch.randn((N,), device="cuda", generator=gen))
        return m

    one, three = linear(2048, 2560, True), [linear(2048, N, False) for N in (2048, 512, 512)]
    for rows, b in ((6, 4), (8, 8), (16, 4), (32, 8)):
        assert _staged([2560], rows, 2048, b) == 1 and _staged([2048, 512, 512], rows, 2048, b) == 1
        x = torch.randn((2, rows // 2, 2048), device="cuda", generator=gen).half()
        with torch.inference_mode():
            got, joint, split = one(x, precision=b), forward_group(three, x, b, concat=True), forward_group(three, x, b)
            with _capi.tuning(gemm_staged=2):
                want = ext.gemm_kbit(x.view(rows, -1), one.qweight, one._buffers[f"lut{b}"], b) + one.bias
                wants = [ext.gemm_kbit(x.view(rows, -1), m.qweight, m._buffers[f"lut{b}"], b) for m in three]
        assert torch.equal(got.view(rows, -1), want), (rows, b)
        assert torch.equal(joint.view(rows, -1), torch.cat(wants, dim=-1)), (rows, b)
        assert all(torch.equal(s.view(rows, -1), w) for s, w in zip(split, wants)), (rows, b)


@gpu
@pytest.mark.parametrize("rows", (2, 4, 8, 16))
def test_modes_see_a_small_set_joined(rows):
    """At 2..8 rows torch joins a set's results wherever a mode could see it, also where the staged kernel serves the set; the same results."""
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode
    from any_precision_amd import AnyPrecisionLinear
    from any_precision_amd.linear import forward_group
    K, Ns = 4096, (4096, 4096, 4096)
    assert _staged(Ns, rows, K, 3) == (rows > 2)
    gen = torch.Generator(device="cuda").manual_seed(rows)
    members = []
    for N in Ns:
        m = AnyPrecisionLinear(K, N, [3], bias=False, device="cuda", dtype=torch.float16)
        m.qweight.copy_(torch.randint(-2**31, 2**31, m.qweight.shape, dtype=torch.int32, device="cuda", generator=gen))
        m._buffers["lut3"].copy_(torch.randn((N, 8), device="cuda", generator=gen) * 0.02)
        members.append(m)
    x = torch.randn((rows, K), device="cuda", generator=gen).half()
    want, seen = forward_group(members, x, 3, concat=True), []

    class Functions(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(getattr(func, "__name__", ""))
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func._schema.name.split("::")[-1])
            return func(*args, **(kwargs or {}))

    for mode in (Functions, Dispatch):
        seen.clear()
        with mode():
            got = forward_group(members, x, 3, concat=True)
        assert torch.equal(got, want) and ("cat" in seen) == (rows <= 8), (mode, seen)


_KNOBS = ("gemv_target_waves", "gemv_rows", "gemv_wpl", "dequant_blocks_per_cu", "matmul_mfma_from", "gemm_split", "matmul_mfma4", "gemv4_groups", "gemm_rb2",
          "gemv_stream", "gemv_stream_waves", "gemv_fine", "gemm_walk", "gemm_walk_wgs", "gemm_tiled", "gemm_tile", "gemm_tile_split", "gemm_lookahead",
          "gemm_block", "gemm_block_tile", "gemm_staged")


def test_which_calls_the_rule_takes():
    """Only calls that the kernel serves, none that another knob forces or forbids, and one row and two never; errors as ap_gemm_kbit has them."""
    from any_precision_amd import _capi
    for K in (32, 96, 128, 512, 544, 1024, 4064, 4096, 11008):
        for Ns in ([1], [16], [4096], [14336], [4096, 1024, 1024], [11008, 11008]):
            for b in range(3, 9):
                for M in (1, 2, 3, 4, 5, 8, 9, 16, 17, 32, 33, 128):
                    taken = _staged(Ns, M, K, b)
                    assert taken == 0 or (taken == 1 and K % 128 == 0 and 3 <= M <= 32), (K, Ns, b, M)
                    with _capi.tuning(gemm_staged=0):
                        assert _staged(Ns, M, K, b) == 0
                    with _capi.tuning(gemm_staged=2):
                        assert _staged(Ns, M, K, b) == (1 if K % 128 == 0 and M <= 32 else 0)
    assert _staged([4096], 16, 4096, 4) == 1 and _staged([4096], 8, 14336, 8) == 1 and _staged([4096] * 3, 16, 4096, 4) == 1
    for knobs in ({"gemm_tiled": 2}, {"gemm_block": 0}, {"gemm_rb2": 2}, {"matmul_mfma_from": 9}, {"gemv_rows": 2}):
        with _capi.tuning(**knobs):
            assert _staged([4096], 16, 4096, 4) == 0, knobs
    # every knob that chooses a form, and two at once; those that size a grid leave the choice alone
    value = ctypes.c_int()
    for name in _KNOBS:
        assert _capi.lib.ap_get_tuning(name.encode(), ctypes.byref(value)) == 0
        with _capi.tuning(**{name: value.value + 1}):
            assert _staged([4096], 16, 4096, 4) == (name in ("dequant_blocks_per_cu", "gemv_stream_waves", "gemm_walk_wgs", "gemm_staged")), name
            with _capi.tuning(gemm_split=2):
                assert _staged([4096], 16, 4096, 4) == (name == "gemm_staged")
        assert _staged([4096], 16, 4096, 4) == 1
    assert _staged([4096], 16, 4096, 9) < 0 and _staged([4096], 0, 4096, 4) < 0 and _staged([64] * 5, 16, 4096, 4) < 0
    assert _staged([1 << 25], 16, 1 << 14, 3) == 0           # planes of 4 GiB and more: beyond 32-bit offsets


def test_the_rule_at_a_few_rows_is_one_of_rounds():
    """Many bits on long rows at 3 and 4 rows: where the CUs are used evenly, one block of 16 rows each or two; and what the kernel is slower at."""
    for M, b in ((3, 5), (3, 6), (4, 7), (4, 8)):
        for K in (8320, 11008, 14336):
            for rows, taken in ((2048, 0), (2944, 0), (3072, 1), (4096, 1), (4112, 0), (5120, 0), (6144, 1), (8192, 1), (8208, 1), (14336, 1)):
                assert _staged([rows], M, K, b) == taken, (rows, M, K, b)
    assert [_staged([16384], 4, 5120, b) for b in (4, 5, 6)] == [1, 1, 0]
    assert [_staged([12288], 12, K, 5) for K in (1152, 1536, 1664)] == [0, 0, 1]
    assert [_staged([4096] * 3, 3, K, 3) for K in (1024, 2048, 4096)] == [0, 0, 1]
    assert [_staged([1024] * 3, 6, K, 8) for K in (1280, 2560, 4096)] == [0, 0, 1] and [_staged([1024] * 3, M, 2048, 7) for M in (6, 7, 8)] == [0, 1, 1]
