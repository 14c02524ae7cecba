"""The block-tile fused GEMM (ap_gemm_kbit from 9 activation rows on): every tile against the oracle at the edges of its range."""
import pytest
import torch

from _util import assert_bit_exact, assert_close_gemv, layer_to_gpu, make

pytestmark = pytest.mark.gpu
TILES = (841, 342, 324, 442, 424, 242, 224, 218, 124)
NOT_BUILT = {(8, 424), (8, 218)}      # their tables do not fit the LDS


@pytest.fixture(scope="module")
def ext():
    import any_precision_ext
    return any_precision_ext


def _x(M, K, seed):
    from any_precision_amd import synth
    x = synth.make_x(M, K, seed=seed)
    return x, torch.from_numpy(x).cuda()


def _tiles(b):
    return [t for t in TILES if (b, t) not in NOT_BUILT]


# K: one half-step of 256 elements; a part of one behind it (288, 992, 2720); fewer half-steps than groups; a different number per
# group (1280, 11008).  N: no multiple of any tile, of 4, of 8.
@pytest.mark.parametrize("N,K", ((131, 256), (64, 288), (77, 992), (128, 1280), (200, 2720), (96, 4096), (33, 11008)))
def test_every_tile_agrees_with_the_oracle(ext, oracle, N, K):
    from any_precision_amd import _capi
    L = make(N, K, seed=N + K)
    q, luts = layer_to_gpu(L)
    for b in range(3, 9):
        for M in (1, 32, 65, 257):
            x, xg = _x(M, K, seed=M)
            _, want = oracle.matmul_kbit(x, L.qweight, L.luts[b], b, return_f64=True)
            for tile in _tiles(b):
                print(f"block tile N={N} K={K} b={b} M={M} tile={tile}", flush=True)
                with _capi.tuning(gemm_block=2, gemm_block_tile=tile):
                    got = ext.gemm_kbit(xg, q, luts[b], b)
                assert_close_gemv(got, want, f"N={N} K={K} b={b} M={M} tile={tile}")


def test_one_hot_rows_give_the_weights_exactly(ext, oracle):
    from any_precision_amd import _capi
    N, K = 70, 2080 + 512
    L = make(N, K, seed=5)
    q, luts = layer_to_gpu(L)
    ks = list(range(0, K, 37)) + [255, 256, 1023, 1024, 2047, 2048, K - 1, K - 32, K - 33]
    x = torch.zeros((len(ks), K), dtype=torch.float16, device="cuda")
    x[torch.arange(len(ks)), torch.tensor(ks)] = 1.0
    for b in range(3, 9):
        w = oracle.dequant_kbit(L.qweight, L.luts[b], b)
        for tile in _tiles(b):
            with _capi.tuning(gemm_block=2, gemm_block_tile=tile):
                got = ext.gemm_kbit(x, q, luts[b], b)
            assert_bit_exact(got.t().contiguous(), w[:, ks], f"one-hot b={b} tile={tile}")


@pytest.mark.parametrize("K", (1024, 1056))
def test_what_is_not_a_number_stays_in_its_row(ext, K):
    """NaN and infinities in one activation row, an infinite table entry that no weight of the row uses."""
    from any_precision_amd import _capi
    N, M = 40, 70
    for b in (3, 4, 5, 8):
        q, luts = layer_to_gpu(make(N, K, seed=b))
        x = torch.randn((M, K), device="cuda").half()
        x[5, 3], x[M - 1, K - 1] = float("nan"), float("inf")
        table = luts[b].clone()
        # row 7 uses one code only (all planes 0): the others are infinite
        q[:, 7] = 0
        table[7, 1:] = float("inf")
        w = ext.dequant_kbit(q, table, b)
        for tile in _tiles(b):
            with _capi.tuning(gemm_block=2, gemm_block_tile=tile):
                got = ext.gemm_kbit(x, q, table, b)
            clean = [m for m in range(M) if m not in (5, M - 1)]
            assert torch.isfinite(got[clean]).all(), (K, b, tile)
            want = x[clean].float() @ w.float().t()
            assert (got[clean].float() - want).norm() <= 1e-3 * want.norm()      # fp16 results of fp32 sums
            assert torch.isnan(got[5]).all() and not torch.isfinite(got[M - 1]).any()


def test_sets_and_strided_results(ext):
    """Linears that share x in one launch, dense and side by side, bit for bit what each alone gives; replayed from a graph."""
    from any_precision_amd import _capi
    Ns, K, M = (200, 64, 72, 129), 1280, 100
    for b in (3, 4, 6, 8):
        gpu = [layer_to_gpu(make(N, K, seed=N)) for N in Ns]
        qs, ts = [q for q, _ in gpu], [luts[b] for _, luts in gpu]
        x = torch.randn((M, K), device="cuda").half()
        for tile in _tiles(b):
            with _capi.tuning(gemm_block=2, gemm_block_tile=tile):
                singles = [ext.gemm_kbit(x, q, t, b) for q, t in zip(qs, ts)]
                outs = ext.gemm_kbit_group(x, qs, ts, b)
                joint = ext.gemm_kbit_group(x, qs, ts, b, concat=True)
                torch.cuda.synchronize()
                g = torch.cuda.CUDAGraph()
                with torch.cuda.graph(g):
                    replayed = ext.gemm_kbit_group(x, qs, ts, b, concat=True)
            assert all(torch.equal(s, o) for s, o in zip(singles, outs)), (b, tile)
            assert torch.equal(joint, torch.cat(singles, dim=-1)), (b, tile)
            for _ in range(3):
                replayed.zero_()
                torch.cuda.synchronize()
                g.replay()
                torch.cuda.synchronize()
                assert torch.equal(replayed, joint), (b, tile)


def test_linear_takes_it_for_plain_forwards_and_stays_differentiable(ext):
    """At 600 rows and 5 bits a 1024-row linear goes through the block-tile kernel; where gradients, tangents or batching follow the
    call it goes through torch's product as before."""
    from any_precision_amd import AnyPrecisionLinear, _capi
    N, K, M, b = 1024, 512, 600, 5
    assert not _capi.gemm_pays(M, N, K, b) and _capi.lib.ap_gemm_kbit_taken(M, N, K, b) == 1
    lin = AnyPrecisionLinear(K, N, list(range(3, 9)), bias=False, device="cuda", dtype=torch.float16)
    q, luts = layer_to_gpu(make(N, K, seed=1))
    lin.qweight.copy_(q)
    for i, t in luts.items():
        lin._buffers[f"lut{i}"].copy_(t)
    x = torch.randn((M, K), device="cuda").half()
    w = ext.dequant_kbit(q, luts[b], b)
    y = lin(x, precision=b)
    assert torch.equal(y, ext.gemm_kbit(x, q, luts[b], b))
    leaf = x.clone().requires_grad_()
    out = lin(leaf, precision=b)
    out.backward(torch.ones_like(out))
    want = w.float().sum(0)
    assert (leaf.grad.float() - want).norm() <= 1e-2 * want.norm() * M ** 0.5
    with torch.no_grad():
        assert torch.equal(lin(leaf, precision=b), y)
    tangent = torch.func.jvp(lambda a: lin(a, precision=b), (x,), (x,))[1]
    assert (tangent.float() - y.float()).norm() <= 1e-2 * y.float().norm()
    batched = torch.func.vmap(lambda a: lin(a, precision=b))(x.view(1, M, K))
    assert (batched.float().view(M, N) - y.float()).norm() <= 1e-2 * y.float().norm()


def test_autocast_decides_the_type_of_the_product(ext):
    """A linear and a set where only the plain route is the kernel: under autocast the results are those of torch's product, of its type."""
    import ctypes
    from any_precision_amd import AnyPrecisionLinear, _capi
    from any_precision_amd.linear import forward_group
    K, M, b, Ns = 512, 512, 5, (2048, 2080)
    mods = []
    for N in Ns:
        mods.append(AnyPrecisionLinear(K, N, list(range(3, 9)), bias=False, device="cuda", dtype=torch.float16))
        q, luts = layer_to_gpu(make(N, K, seed=N))
        mods[-1].qweight.copy_(q)
        mods[-1]._buffers[f"lut{b}"].copy_(luts[b])
        assert not _capi.gemm_pays(M, N, K, b) and _capi.lib.ap_gemm_kbit_taken(M, N, K, b) == 1
    assert not _capi.gemm_group_pays(M, list(Ns), K, b)
    assert _capi.lib.ap_gemm_kbit_group_taken(len(Ns), (ctypes.c_int * len(Ns))(*Ns), M, K, b) == 1
    x = torch.randn((M, K), device="cuda").half()
    dense = [ext.dequant_kbit(m.qweight, m._buffers[f"lut{b}"], b) for m in mods]
    plain = [ext.gemm_kbit(x, m.qweight, m._buffers[f"lut{b}"], b) for m in mods]
    with torch.autocast("cuda", dtype=torch.bfloat16):
        want = [torch.matmul(x, w.t()) for w in dense]
        got, joint = [m(x, precision=b) for m in mods], forward_group(mods, x, b, concat=True)
        sets = forward_group(mods, x, b)
        with torch.autocast("cuda", enabled=False):
            inner = [m(x, precision=b) for m in mods]
    assert all(y.dtype == torch.bfloat16 and torch.equal(y, z) for y, z in zip(got, want))
    assert all(y.dtype == torch.bfloat16 and torch.equal(y, z) for y, z in zip(sets, want))
    assert joint.dtype == torch.bfloat16 and torch.equal(joint, torch.cat(want, dim=-1))
    with torch.autocast("cuda", dtype=torch.float16):
        half = [m(x, precision=b) for m in mods]
    assert all(torch.equal(y, p) and torch.equal(z, p) for y, z, p in zip(half, inner, plain))


def test_the_rule_keeps_to_its_range():
    """No GPU is asked: where ap_gemm_kbit_taken says yes beyond ap_gemm_kbit_pays."""
    from any_precision_amd import _capi
    taken = _capi.lib.ap_gemm_kbit_taken
    assert taken(512, 14336, 4096, 5) == 1 and taken(1024, 14336, 4096, 5) == 0 and taken(1024, 4096, 14336, 5) == 1
    assert taken(2048, 4096, 4096, 3) == 1 and taken(2049, 4096, 4096, 3) == 0 and taken(512, 512, 4096, 5) == 0
    assert taken(256, 4096, 224, 5) == _capi.lib.ap_gemm_kbit_pays(256, 4096, 224, 5)     # shorter than a half-step
    # inside the range, where the pair is faster (us pair / block tile: 31 / 33, 60 / 73, 47 / 56, 152 / 198)
    for M, N, K, b in ((507, 2652, 2368, 8), (584, 6473, 4224, 5), (281, 10304, 2368, 8), (898, 8784, 7168, 6)):
        assert taken(M, N, K, b) == 0, (M, N, K, b)
    assert taken(512, 4096, 4100, 5) == _capi.AP_ESHAPE and taken(0, 4096, 4096, 5) == _capi.AP_EBATCH
    with _capi.tuning(gemm_block=0):
        assert taken(512, 14336, 4096, 5) == 0


def test_tiles_are_counted_on_the_xcd_that_has_most(ext):
    """2560 rows are 20 blocks of 128: three on four of the XCDs, two on the others.  At 1527 rows 12 x 20 tiles of 128 x 128 are two rounds
    of the former; 6 x 20 of 256 x 128 are one.  The two add up K in different orders, so the results tell which ran."""
    from any_precision_amd import _capi
    N, K, M, b = 2560, 2560, 1527, 6
    g = torch.Generator(device="cuda").manual_seed(1)
    q = torch.randint(-2**31, 2**31, (b, N, K // 32), dtype=torch.int32, device="cuda", generator=g)
    t = (torch.randn((N, 1 << b), device="cuda", generator=g) * 0.02).half()
    x = torch.randn((M, K), device="cuda", generator=g).half()
    got = {}
    for tile in (0, 442, 841):
        with _capi.tuning(gemm_block=2, gemm_block_tile=tile):
            got[tile] = ext.gemm_kbit(x, q, t, b)
    assert torch.equal(got[0], got[841]) and not torch.equal(got[0], got[442])


# (N, K, rows, bits): one shape of each line that keeps a call with the kernels before this one, and one just across it.  Short rows: the
# tiled kernel, and the K-split kernel on rows of no multiple of 128 elements; 2560 x 2560: tiles that do not go evenly over the XCDs.
@pytest.mark.parametrize("N,K,M,b,block", (
    (5696, 384, 107, 4, False), (3520, 256, 208, 6, False), (3520, 1280, 208, 6, True), (2560, 2560, 1395, 3, False), (2560, 2560, 512, 3, True),
    (1181, 544, 98, 5, False), (1184, 3232, 98, 5, True), (1999, 2720, 128, 6, True), (1999, 2720, 80, 6, False), (4096, 480, 64, 3, False), (4096, 4128, 64, 3, True), (6000, 1120, 40, 4, False),
    (6000, 1760, 40, 4, True), (6000, 2720, 40, 6, False), (12000, 992, 40, 6, False), (12000, 1056, 40, 6, True), (3000, 480, 200, 5, False),
    (3000, 544, 200, 5, True), (6912, 384, 46, 6, False), (6912, 256, 46, 6, True), (2000, 288, 300, 5, True)))
def test_who_serves_a_call(ext, N, K, M, b, block):
    """Bit for bit the kernel that the rule names: the order of the additions tells the others' results from its own."""
    from any_precision_amd import _capi
    g = torch.Generator(device="cuda").manual_seed(N + K + M)
    q = torch.randint(-2**31, 2**31, (b, N, K // 32), dtype=torch.int32, device="cuda", generator=g)
    t = (torch.randn((N, 1 << b), device="cuda", generator=g) * 0.02).half()
    x = torch.randn((M, K), device="cuda", generator=g).half()
    got = ext.gemm_kbit(x, q, t, b)
    with _capi.tuning(gemm_block=0):
        others = ext.gemm_kbit(x, q, t, b)
    with _capi.tuning(gemm_block=2):
        own = ext.gemm_kbit(x, q, t, b)
    assert not torch.equal(own, others)
    assert torch.equal(got, own if block else others)


# (members, K, rows, bits): gate and up in one launch from 9 rows on, and where the rule leaves them one by one
@pytest.mark.parametrize("Ns,K,M,b,taken", (
    ((10016, 10000), 4096, 9, 3, 1), ((10016, 10000), 4096, 16, 8, 1), ((10016, 10000), 4096, 13, 5, 1), ((10016, 10000), 4096, 12, 5, 0),
    ((10016, 10000), 4096, 16, 4, 0), ((10016, 10000), 5120, 11, 4, 1), ((10016, 10000), 4096, 32, 4, 1), ((10016, 9983), 4096, 32, 3, 1), ((9000, 1200), 4096, 17, 5, 0),
    ((9000, 1240), 4096, 17, 5, 1),
    ((14000, 6016), 4096, 16, 3, 0), ((10016, 10000), 4128, 9, 3, 0), ((10016, 10000), 4128, 17, 3, 1)))
def test_wide_sets_of_few_rows(ext, Ns, K, M, b, taken):
    """Against the fp32 product of the exact weights: one rounding to fp16 and K additions in fp32 on either side."""
    import ctypes
    from any_precision_amd import _capi
    assert _capi.lib.ap_gemm_kbit_group_taken(len(Ns), (ctypes.c_int * len(Ns))(*Ns), M, K, b) == taken
    g = torch.Generator(device="cuda").manual_seed(K + M + b)
    qs = [torch.randint(-2**31, 2**31, (b, n, K // 32), dtype=torch.int32, device="cuda", generator=g) for n in Ns]
    ts = [(torch.randn((n, 1 << b), device="cuda", generator=g) * 0.02).half() for n in Ns]
    x = torch.randn((M, K), device="cuda", generator=g).half()
    got = ext.gemm_kbit_group(x, qs, ts, b)
    if taken:
        with _capi.tuning(gemm_block=2):
            same = ext.gemm_kbit_group(x, qs, ts, b)
    else:       # what a module asks and what the set's call does are one rule
        same = [ext.gemm_kbit(x, q, t, b) for q, t in zip(qs, ts)]
    for q, t, y, z in zip(qs, ts, got, same):
        w = ext.dequant_kbit(q, t, b).float()
        bound = 2.0 ** -24 * 2 * K * (x.float().abs() @ w.abs().t()) + 2.0 ** -11 * (x.float() @ w.t()).abs() + 2.0 ** -24
        assert ((y.float() - x.float() @ w.t()).abs() <= bound).all(), (Ns, K, M, b)
        assert torch.equal(y, z), (Ns, K, M, b)


def test_long_wide_linears_of_few_rows(ext):
    """9..16 activation rows on 10240 rows of 8192 elements, and 17 on 10240 of 4096: the block-tile kernel."""
    from any_precision_amd import _capi
    for N, K, M in ((10240, 8192, 9), (10240, 8192, 16), (10240, 4096, 17)):
        for b in range(3, 9):
            q = torch.randint(-2**31, 2**31, (b, N, K // 32), dtype=torch.int32, device="cuda")
            t = (torch.randn((N, 1 << b), device="cuda") * 0.02).half()
            x = torch.randn((M, K), device="cuda").half()
            y = ext.gemm_kbit(x, q, t, b)
            with _capi.tuning(gemm_block=2):
                assert torch.equal(ext.gemm_kbit(x, q, t, b), y), (N, K, M, b)
            want = x.float() @ ext.dequant_kbit(q, t, b).float().t()
            assert (y.float() - want).norm() <= 1e-3 * want.norm(), (N, K, M, b)
