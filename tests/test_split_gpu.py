"""GPU tests of gemm_split_kernel: large products on the bf16 matrix cores, every operand
value split into three bf16 parts (gemm_split.hip), taken by the dispatcher's own choice.

The shapes reach its two tiles (256x128, 128x128), ragged M and N, k-tiles of 16
with every kind of tail, and k ranges. Small-integer operands make the exact answer known in
any summation order. On random operands the error against fp64 is compared with that of the
fp32 kernels on the same call (direct loads forced: no split), which it must not exceed, and
the bits must differ, which shows that the split kernel ran."""
import ctypes

import numpy as np
import pytest
import torch

from my_pytchon_opencl_lib_amd import _native

pytestmark = pytest.mark.gpu

LAYOUTS = [(0, 0), (0, 1), (1, 0), (1, 1)]


def say(*a):
    print(*a, flush=True)


def run(ta, tb, M, N, K, a, lda, sA, b, ldb, sB, bias, c, ldc, sC, batch=1, acc=False):
    _native.call("migemm_gemm_strided_batched_ex",
                 ctypes.c_void_p(torch.cuda.current_stream().cuda_stream), ta, tb, M, N, K,
                 ctypes.c_void_p(a.data_ptr()), lda, sA, ctypes.c_void_p(b.data_ptr()), ldb, sB,
                 None if bias is None else ctypes.c_void_p(bias.data_ptr()),
                 ctypes.c_void_p(c.data_ptr()), ldc, sC, batch, int(acc))


def case(M, K, N, ta, tb, batch=1, pad=0, off=0, ints=True, seed=0):
    """Operands as (device buffer view, ld, stride) and their fp64 op(A), op(B): rows padded
    by `pad` NaN, the first element `off` floats into the buffer."""
    g = torch.Generator(device="cuda:0").manual_seed(seed)

    def one(rows, cols):
        ld = cols + pad
        buf = torch.full((off + batch * rows * ld,), float("nan"), device="cuda:0")
        x = (torch.randint(-4, 5, (batch, rows, cols), generator=g, device="cuda:0").float()
             if ints else torch.randn(batch, rows, cols, generator=g, device="cuda:0"))
        buf[off:].view(batch, rows, ld)[:, :, :cols] = x
        return buf[off:], ld, rows * ld, x.double()

    a, lda, sA, a64 = one(*((K, M) if ta else (M, K)))
    b, ldb, sB, b64 = one(*((N, K) if tb else (K, N)))
    a64 = a64.transpose(1, 2).contiguous() if ta else a64
    b64 = b64.transpose(1, 2).contiguous() if tb else b64
    return (a, lda, sA), (b, ldb, sB), a64, b64


# (M, K, N, tile, k ranges): both tiles, whole and in ranges; K % 16 = 1, 0, 15, 9, 15, 11
SHAPES = [(2100, 1009, 1900, "128x128", 1), (4097, 144, 3073, "128x128", 1),
          (5000, 511, 2049, "128x128", 1), (3552, 1865, 2240, "256x128", 1),
          (2144, 2495, 1024, "256x128", 3), (1030, 2571, 1290, "128x128", 2)]


def wide_ints(shape, bits, nonzero, g):
    """Integers of `bits` bits, `nonzero` of them in each row and the others 0."""
    keep = torch.rand(shape, generator=g, device="cuda:0").argsort(-1) < nonzero
    return torch.randint(1 - (1 << bits), 1 << bits, shape, generator=g,
                         device="cuda:0").float() * keep


@pytest.mark.parametrize("M,K,N,tile,ranges", SHAPES)
@pytest.mark.parametrize("ta,tb", LAYOUTS)
def test_split_exact(M, K, N, tile, ranges, ta, tb):
    """Odd sizes, rows off 16-byte boundaries, NaN between the rows; bias and C += result.
    One operand's integers have mid and low parts too: of 18 bits, 16 to a sum, the other
    one's of up to 3 (|sum| <= 16 2^18 4 = 2^24)."""
    g = torch.Generator(device="cuda:0").manual_seed(M)
    for pad, off, bias, acc, wide in [(0, 0, False, False, "a"), (3, 1, True, True, "b"),
                                      (0, 0, False, False, "")]:
        say("split exact", M, K, N, ta, tb, pad, off, bias, acc, wide)
        (a, lda, sA), (b, ldb, sB), a64, b64 = case(M, K, N, ta, tb, pad=pad, off=off, seed=K)
        if wide == "a":
            a64 = wide_ints((M, K), 18, 16, g).double()[None]
            a.view(-1, lda)[:, :lda - pad] = a64[0].t() if ta else a64[0]
        elif wide == "b":
            b64 = wide_ints((N, K), 18, 16, g).double().t()[None].contiguous()
            b.view(-1, ldb)[:, :ldb - pad] = b64[0].t() if tb else b64[0]
        # (with bias and C too, the sums stay below 2^24: checked)
        bv = torch.arange(N, device="cuda:0").remainder(41).sub(20).float() if bias else None
        c = torch.full((M, N + pad), 7.0 if acc else float("nan"), device="cuda:0")
        run(ta, tb, M, N, K, a, lda, sA, b, ldb, sB, bv, c, N + pad, 0, acc=acc)
        plan = _native.last_plan()
        assert plan.startswith(f"tiled-split tile={tile} splits={ranges} "), plan
        expect = (a64 @ b64)[0]
        if bias:
            expect = expect + bv.double()
        if acc:
            expect = expect + 7.0
        assert float(expect.abs().max()) < 2 ** 24
        assert torch.equal(c[:, :N], expect.float())
        if pad:
            assert bool((c[:, N:] == 7.0).all() if acc else c[:, N:].isnan().all())


# (M, K, N, batch): one range; k ranges as the fp32 plan has them (6400 x 4096 x 512 in 3,
# 500 x 12000 x 6565 in 6); more ranges than it has (512 x 6400 x 4096); a batch
RANDOM = [(2100, 1009, 1900, 1), (4096, 512, 3000, 1), (4096, 2048, 4096, 1),
          (6400, 4096, 512, 1), (500, 12000, 6565, 1), (512, 6400, 4096, 1),
          (900, 1000, 1400, 8)]


@pytest.mark.parametrize("M,K,N,batch", RANDOM)
@pytest.mark.parametrize("ta,tb", LAYOUTS)
def test_split_error_no_larger_than_fp32(M, K, N, batch, ta, tb):
    """N(0,1) operands. The error of a sum of K rounded terms is a random quantity; over the
    >= 2.7 million outputs compared here its norm varies by less than 1 %, so 1.02 times the
    fp32 kernel's is the bound for "no larger"."""
    (a, lda, sA), (b, ldb, sB), a64, b64 = case(M, K, N, ta, tb, batch=batch, ints=False, seed=N)
    c64 = a64 @ b64
    err, outs = [], []
    for direct, kernel in ((0, "tiled-split "), (2, "tiled-direct ")):
        c = torch.full((batch, M, N), float("nan"), device="cuda:0")
        with _native.tuned(direct=direct):
            run(ta, tb, M, N, K, a, lda, sA, b, ldb, sB, None, c, N, M * N, batch)
        assert _native.last_plan().startswith(kernel), _native.last_plan()
        err.append(float((c - c64).norm() / c64.norm()))
        outs.append(c)
    say("split error", M, K, N, batch, ta, tb, err)
    assert err[0] <= 1.02 * err[1]


# Operands of real use that are not dense: (name, A of N(0,1) values -> A)
SPARSE = [("relu", lambda a, g: a.clamp(min=0)),
          ("quarter", lambda a, g: a * (torch.rand(a.shape, generator=g, device=a.device) < 0.25)),
          ("sixteen in K", lambda a, g: a * (torch.rand(a.shape, generator=g, device=a.device)
                                             < 16.0 / 1009)),
          ("positive", lambda a, g: a.abs())]


@pytest.mark.parametrize("name,change", SPARSE, ids=[s[0] for s in SPARSE])
@pytest.mark.parametrize("M,K,N", [(2100, 1009, 1900), (2500, 4095, 2500), (500, 12000, 6565)])
def test_split_error_of_sparse_and_one_sided_operands(M, K, N, name, change):
    """As above for operands with zeros, around which each rounding of a sum tells, and for
    values of one sign, whose sums show a rounding that is not to nearest."""
    (a, lda, _), (b, ldb, _), _, b64 = case(M, K, N, 0, 0, ints=False, seed=K)
    g = torch.Generator(device="cuda:0").manual_seed(31)
    a = change(a, g).contiguous()
    if name == "positive":
        b = b.abs()
    c64 = a.view(M, K).double() @ b.view(K, N).double()
    err = []
    for direct, kernel in ((0, "tiled-split "), (2, "tiled-direct ")):
        c = torch.full((M, N), float("nan"), device="cuda:0")
        with _native.tuned(direct=direct):
            run(0, 0, M, N, K, a, lda, 0, b, ldb, 0, None, c, N, 0)
        assert _native.last_plan().startswith(kernel), _native.last_plan()
        err.append(float((c - c64).norm() / c64.norm()))
    say("split error", name, M, K, N, err)
    assert err[0] <= err[1]


@pytest.mark.parametrize("ta,tb", LAYOUTS)
def test_split_sums_of_one_product(ta, tb):
    """One value per row of op(A): each output is one product, whose error has no sum to hide
    in. The bound: the products of parts that are left out, (1 + 2^-10) 2^-24 of it; the fp32
    rounding of the result, 2^-24; five roundings or truncations of a sum below 2^-6 of it,
    under 2^-27 together. Values near 1 are the worst. Integer products of up to 24 bits are
    exact."""
    M, K, N = 2100, 1009, 1900
    (a, lda, _), (b, ldb, _), _, _ = case(M, K, N, ta, tb, ints=False, seed=41)
    g = torch.Generator(device="cuda:0").manual_seed(42)
    at = torch.randint(K, (M,), generator=g, device="cuda:0")
    m = torch.arange(M, device="cuda:0")

    def product(av, bv):  # values of the M entries and of op(B)
        a.zero_()
        a.view(*((K, M) if ta else (M, K)))[(at, m) if ta else (m, at)] = av
        b.copy_((bv.t() if tb else bv).reshape(-1))
        c = torch.full((M, N), float("nan"), device="cuda:0")
        run(ta, tb, M, N, K, a, lda, 0, b, ldb, 0, None, c, N, 0)
        assert _native.last_plan().startswith("tiled-split "), _native.last_plan()
        return c.double(), av.double()[:, None] * bv.double()[at]

    uniform = lambda *s: torch.rand(*s, generator=g, device="cuda:0")  # noqa: E731
    worst = []
    for av, bv in [(1 + 0.05 * uniform(M), 1 + 0.05 * uniform(K, N)),
                   (uniform(M) - 0.5, uniform(K, N) - 0.5)]:
        c, expect = product(av, bv)
        worst.append(float(((c - expect).abs() / expect.abs().clamp(min=1e-30)).max()) * 2 ** 24)
    say("split one product", ta, tb, worst)
    assert max(worst) <= 2.13
    for bits in (12, 17):  # 12 x 12 and 17 x 7 bits
        c, expect = product(
            torch.randint(1 << bits, (M,), generator=g, device="cuda:0").float(),
            torch.randint(1 << (24 - bits), (K, N), generator=g, device="cuda:0").float())
        assert torch.equal(c, expect)


@pytest.mark.parametrize("ta,tb", LAYOUTS)
def test_split_nonfinite_and_tiny_operands(ta, tb):
    """Infinities and NaN reach the outputs that fp32 arithmetic says, tiny values keep their
    precision, a value above bf16's rounding overflow stays finite, and every other output is
    the exact product."""
    M, K, N = 2100, 1009, 1900
    (a, lda, _), (b, ldb, _), a64, b64 = case(M, K, N, ta, tb, seed=5)

    def put(x, t, i, k, value):  # element (i, k) of op(A), or (k, i) of op(B)
        x.view(*((K, -1) if t else (-1, K)))[(k, i) if t else (i, k)] = value

    put(a, ta, 7, 1000, float("inf"))
    put(a, ta, 300, 3, float("nan"))
    put(b, not tb, 1899, 500, float("-inf"))
    a64[0, 7, 1000], a64[0, 300, 3], b64[0, 500, 1899] = np.inf, np.nan, -np.inf
    put(a, ta, 1900, 16, 3.4e38)
    b.view(*((N, K) if tb else (K, N)))[(slice(None), 16) if tb else 16] = 0.25
    a64[0, 1900, 16], b64[0, 16, :] = float(np.float32(3.4e38)), 0.25
    c = torch.empty(M, N, device="cuda:0")
    say("split nonfinite", ta, tb)
    run(ta, tb, M, N, K, a, lda, 0, b, ldb, 0, None, c, N, 0)
    # (CPU: IEEE products one by one)
    expect = torch.from_numpy(a64[0].cpu().numpy() @ b64[0].cpu().numpy()).float()
    rows = torch.ones(M, dtype=torch.bool)
    rows[1900] = False
    got = c.cpu()
    assert torch.equal(torch.nan_to_num(got[rows], nan=123.5), torch.nan_to_num(expect[rows], nan=123.5))
    big = got[1900, :1899].double() / expect[1900, :1899].double()
    assert bool(((big - 1).abs() < 1e-6).all())
    # sums past 2^82, which overflow scaled, stay finite too (here |sum| <= 16 K 2^110 < 2^124)
    (a, lda, _), (b, ldb, _), a64, b64 = case(M, K, N, ta, tb, seed=7)
    run(ta, tb, M, N, K, a * 2.0 ** 55, lda, 0, b * 2.0 ** 55, ldb, 0, None, c, N, 0)
    assert torch.equal(c, (a64 @ b64)[0].float() * 2.0 ** 110)
    # tiny: A of 2^-126 .. 2^-122, subnormals among them, B scaled up by 2^60
    (a, lda, _), (b, ldb, _), a64, b64 = case(M, K, N, ta, tb, ints=False, seed=6)
    a *= 2.0 ** -124
    b *= 2.0 ** 60
    a64 = (a.view(K, M).t() if ta else a.view(M, K)).double().contiguous()
    b64 = (b.view(N, K).t() if tb else b.view(K, N)).double().contiguous()
    run(ta, tb, M, N, K, a, lda, 0, b, ldb, 0, None, c, N, 0)
    c64 = a64 @ b64
    assert float((c.double() - c64).norm() / c64.norm()) < 1e-6  # fp32 chain: 5.7e-7


@pytest.mark.parametrize("ta,tb", LAYOUTS)
def test_split_small_operands_bit_for_bit(ta, tb):
    """A power of two times an operand is that power times the result, bit for bit, down to
    fp32's least normal and subnormal values (every bf16 part of a scaled value is a normal
    number): no precision is lost on the way and no tile is computed in another way, whose
    bits would differ."""
    M, K, N = 2100, 1009, 1900
    (a, lda, _), (b, ldb, _), _, _ = case(M, K, N, ta, tb, ints=False, seed=21)
    a.copy_((1 + a.abs() % 15) * a.sign())  # magnitudes of [1, 16): normal down to 2^-126
    b.copy_((1 + b.abs() % 15) * b.sign())

    def product(x, y):
        c = torch.full((M, N), float("nan"), device="cuda:0")
        run(ta, tb, M, N, K, x, lda, 0, y, ldb, 0, None, c, N, 0)
        assert _native.last_plan().startswith("tiled-split "), _native.last_plan()
        return c

    plain = product(a, b)
    for e in (60, 103, 110, 126):
        say("split small operands", ta, tb, e)
        small = 2.0 ** -(e // 2) * 2.0 ** -(e - e // 2)
        assert torch.equal(product(a * small, b * 2.0 ** 40) * 2.0 ** (e - 40), plain)
        assert torch.equal(product(a * 2.0 ** 40, b * small) * 2.0 ** (e - 40), plain)
    # n 2^-149 for integers |n| < 2^23 are the floats whose bits are n
    g = torch.Generator(device="cuda:0").manual_seed(22)
    n = torch.randint(1, 1 << 23, a.shape, generator=g, device="cuda:0", dtype=torch.int32)
    sign = torch.where(a < 0, -1.0, 1.0)
    tiny = torch.copysign(n.view(torch.float32), sign)
    c = product(tiny, b * 2.0 ** 100)
    assert torch.equal(c * 2.0 ** 49, product(n.float() * sign, b))


def test_split_graph_capture_without_a_workspace():
    """512 x 6400 x 4096 TN runs in more k ranges than the fp32 plan, which has one: captured
    on a stream that holds no workspace it still runs, in one range, and replays agree."""
    M, K, N = 512, 6400, 4096
    (a, lda, _), (b, ldb, _), a64, b64 = case(M, K, N, 1, 0, seed=9)
    expect = (a64 @ b64)[0].float()
    c = torch.full((M, N), float("nan"), device="cuda:0")
    run(1, 0, M, N, K, a, lda, 0, b, ldb, 0, None, c, N, 0)
    assert torch.equal(c, expect)
    cap = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=cap):
        run(1, 0, M, N, K, a, lda, 0, b, ldb, 0, None, c, N, 0)
    for _ in range(3):
        c.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(c, expect)


def test_split_graph_capture_in_a_workspace_for_fewer_ranges():
    """6400 x 4096 x 512 NT: 3 k ranges on the fp32 MFMA, more in the split kernel. A capture
    on a stream that reserved room for the 3 runs those in it; replays agree with fp64."""
    M, K, N = 6400, 4096, 512
    (a, lda, _), (b, ldb, _), a64, b64 = case(M, K, N, 0, 1, seed=11)
    expect = (a64 @ b64)[0].float()
    c = torch.full((M, N), float("nan"), device="cuda:0")
    cap = torch.cuda.Stream()
    held = ctypes.c_size_t(0)
    s = ctypes.c_void_p(cap.cuda_stream)
    _native.call("migemm_workspace_reserve", s, 3 * M * N * 4)
    _native.call("migemm_workspace_size", s, ctypes.byref(held))
    assert 3 * M * N * 4 <= held.value < 5 * M * N * 4
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=cap):
        run(0, 1, M, N, K, a, lda, 0, b, ldb, 0, None, c, N, 0)
    plan = _native.last_plan()
    assert plan.startswith("tiled-direct ") and "splits=3 " in plan, plan
    say("replay in 3 ranges")
    for _ in range(3):
        c.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(c, expect)
    _native.call("migemm_workspace_release", s)
