"""Each kernel alone against its plain reference, at sizes other than the engine's: widths and
vocabularies that are no power of two, head sizes in steps of 16, key/value groups, windows."""

import math

import numpy as np
import pytest
import torch

import helpers
import plain_gpt as P
from mini_gpt_inference_amd.ops import kernels
from mini_gpt_inference_amd.ops.residual import PendingSums

pytestmark = pytest.mark.gpu
DEV = "cuda"
TDT = {"float32": torch.float32, "bfloat16": torch.bfloat16}


def rnd(gen, *shape, dtype="float32", scale=1.0):
    t = torch.randn(*shape, generator=gen, dtype=torch.float32) * scale
    return t.to(TDT[dtype])


def i32(values):
    return torch.tensor(list(values), dtype=torch.int32, device=DEV)


# ----------------------------------------------------------------------------- embedding, norm
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("with_pos", [True, False])
def test_embed(dtype, with_pos):
    g = torch.Generator().manual_seed(0)
    tok, pos = rnd(g, 37, 80, dtype=dtype), rnd(g, 19, 80, dtype=dtype)
    ids, positions = [5, 36, 0, 5, 12, 7, 30], [0, 18, 3, 4, 4, 9, 1]
    x = torch.full((7, 80), float("nan"), device=DEV)
    kernels.embed(i32(ids), i32(positions), tok.to(DEV), pos.to(DEV) if with_pos else None, x, 7)
    want = tok.double()[ids] + (pos.double()[positions] if with_pos else 0)
    helpers.assert_close(x, want, "float32", "embed")     # the sum itself is float32 in both cases


@pytest.mark.parametrize("out_dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("width,bias,eps", [(80, True, 1e-5), (1000, False, 1e-2), (48, True, 1e-6), (75, True, 1e-5),
                                            (1030, False, 1e-5), (1600, True, 1e-5), (512, True, 1e-5), (2052, True, 1e-5),
                                            (256, True, 1e-5), (768, False, 1e-5), (1024, True, 1e-5), (1280, True, 1e-5),
                                            (2048, False, 1e-5)])
def test_layer_norm(out_dtype, width, bias, eps):
    g = torch.Generator().manual_seed(1)
    x = rnd(g, 9, width, scale=3.0) + 2.0
    x[3] = 5.0 + 1e-3 * torch.randn(width, generator=g)     # an almost constant row: eps decides
    w, b = 1 + 0.1 * rnd(g, width), rnd(g, width) if bias else None
    out = torch.empty(9, width, dtype=TDT[out_dtype], device=DEV)
    kernels.layer_norm(x.to(DEV), w.to(DEV), b.to(DEV) if bias else None, out, 9, eps)
    want = P.plain_layer_norm(x.double(), w.double(), b.double() if bias else None, eps)
    helpers.assert_close(out, want, out_dtype, "layer_norm")
    rows = [8, 0, 3]
    out2 = torch.empty(3, width, dtype=TDT[out_dtype], device=DEV)
    kernels.layer_norm(x.to(DEV), w.to(DEV), b.to(DEV) if bias else None, out2, 3, eps, rows=i32(rows))
    helpers.assert_close(out2, want[rows], out_dtype, "layer_norm gather")


@pytest.mark.parametrize("out_dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("width", [516, 772, 1028, 1540, 2044, 4096, 4100])
def test_layer_norm_of_rows_in_several_waves(out_dtype, width):
    """A 16-byte piece a lane: in 3, 4, 6 or 8 waves where the rows are few, else in one; in 16 waves; longer rows go to the
    kernel that reads them three times."""
    test_layer_norm(out_dtype, width, True, 1e-5)


@pytest.mark.parametrize("out_dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("width", [512, 516, 768, 1000, 1280, 1284, 1600, 1796, 2044, 2048, 2052, 4096])
def test_layer_norm_keeps_its_sums_whatever_the_number_of_rows(out_dtype, width):
    """Few rows of 513 to 2,048 values have a workgroup of several waves each, more rows a wave each (the line lies at 1,920
    waves): a row's result is the same bits in both."""
    g = torch.Generator().manual_seed(width)
    few = 1920 // (-(-width // 256))
    x, w, b = (rnd(g, few + 1, width, scale=3.0) + 1.0).to(DEV), rnd(g, width).to(DEV), rnd(g, width).to(DEV)
    got = [torch.empty(n, width, dtype=TDT[out_dtype], device=DEV) for n in (few + 1, few, 3)]
    for out in got:
        kernels.layer_norm(x, w, b, out, out.shape[0], 1e-5)
    assert torch.equal(got[0][:few], got[1]) and torch.equal(got[0][:3], got[2])
    helpers.assert_close(got[0][:3], torch.nn.functional.layer_norm(x[:3].double(), (width,), w.double(), b.double(), 1e-5),
                         out_dtype, "layer_norm")


# ----------------------------------------------------------------------------- linear
def _linear_want(a, w, bias, epi, prev):
    y = P.plain_linear(a.double(), w.double(), None if bias is None else bias.double())
    if epi == kernels.EPI_GELU:
        y = P.plain_gelu_tanh(y)
    if epi == kernels.EPI_RESIDUAL:
        y = prev.double() + y
    if epi == kernels.EPI_RELU2:
        y = torch.relu(y) ** 2
    return y


@pytest.mark.parametrize("low,high,error", [(2.0 ** -7, 1.0, 2.0e-7), (1.0, 4.0, 1.0e-7)])
def test_gelu_of_the_bfloat16_products_beside_the_midpoints_of_bfloat16(low, high, error):
    """Inputs whose exact GELU lies within a few 1e-7 of the middle between two bfloat16 values: every one that lies further from it
    than the activation's error in 32 bits is rounded to its own side.  The farthest that is not lies 1.80e-7 and 0.92e-7 of its value
    away (4 and 2 % of them are on the wrong side); as u / (1 + exp(-2 z)) it was 1.12e-7 in [1, 4)."""
    values = (torch.arange(0x3000, 0x4100, dtype=torch.int32) << 16).view(torch.float32).double()
    middle = (values[:-1] + values[1:]) / 2
    below, above = torch.zeros_like(middle), torch.full_like(middle, 16.0)
    for _ in range(80):
        at = (below + above) / 2
        under = P.plain_gelu_tanh(at) < middle
        below, above = torch.where(under, at, below), torch.where(under, above, at)
    there = (below >= low) & (below < high)
    u = (below[there].float().view(torch.int32)[:, None] + torch.arange(-8, 9, dtype=torch.int32)).view(torch.float32).flatten()
    middle = middle[there].repeat_interleave(17)
    exact = P.plain_gelu_tanh(u.double())
    out = torch.empty(1, u.numel(), dtype=torch.bfloat16, device=DEV)
    a, w = torch.zeros(1, 64, dtype=torch.bfloat16, device=DEV), torch.zeros(u.numel(), 64, dtype=torch.bfloat16, device=DEV)
    assert kernels.linear_mfma(a, w, u.to(DEV), out, 1, kernels.EPI_GELU)
    wrong = (out[0].double().cpu() > middle) != (exact > middle)
    assert ((exact - middle).abs() / middle)[wrong].max() <= error


@pytest.mark.parametrize("epi", [kernels.EPI_NONE, kernels.EPI_GELU, kernels.EPI_RESIDUAL])
@pytest.mark.parametrize("a_dt,w_dt,o_dt", [("float32", "float32", "float32"), ("bfloat16", "bfloat16", "bfloat16"),
                                            ("bfloat16", "bfloat16", "float32"), ("bfloat16", "float32", "bfloat16")])
def test_linear_generic(a_dt, w_dt, o_dt, epi):
    if epi == kernels.EPI_RESIDUAL and o_dt != "float32":
        pytest.skip("the residual stream is float32")
    g = torch.Generator().manual_seed(2)
    n, k, o = 70, 48, 203
    a, w, bias = rnd(g, n, k, dtype=a_dt), rnd(g, o, k, dtype=w_dt, scale=0.3), rnd(g, o)
    prev = rnd(g, n, o, dtype=o_dt)
    out = prev.clone().to(DEV)
    kernels.linear_generic(a.to(DEV), w.to(DEV), bias.to(DEV), out, n, epi)
    tol = "float32" if (a_dt, w_dt, o_dt) == ("float32",) * 3 else "bfloat16"
    helpers.assert_close(out, _linear_want(a, w, bias, epi, prev), tol, "linear_generic")


@pytest.mark.parametrize("n_few", [1, 7, 16, 17, 32])
@pytest.mark.parametrize("a_dt,w_dt,o_dt,epi", [("float32", "float32", "float32", kernels.EPI_NONE),
                                                ("float32", "float32", "float32", kernels.EPI_RESIDUAL),
                                                ("float32", "float32", "float32", kernels.EPI_GELU),
                                                ("bfloat16", "float32", "bfloat16", kernels.EPI_GELU),
                                                ("bfloat16", "bfloat16", "float32", kernels.EPI_NONE)])
def test_linear_generic_few_rows_and_many_agree_bit_for_bit(a_dt, w_dt, o_dt, epi, n_few):
    """Few rows go to a kernel with a workgroup per 16 x 16 outputs, more to tiles: every element's sum
    runs in the same order along k in both, so a row's result is the same
    bits whichever kernel its step's size chooses (a decode step against a prompt's step).  (What is float32
    throughout goes to the same kernel in both here: test_float32_product_keeps_its_sums_whatever_the_tiles.)"""
    g = torch.Generator().manual_seed(23)
    n, k, o = 50, 208, 137      # an inner size that is no multiple of the few-rows kernel's stage of 64
    a, w, bias = rnd(g, n, k, dtype=a_dt), rnd(g, o, k, dtype=w_dt), rnd(g, o)
    prev = rnd(g, n, o, dtype=o_dt)
    many = prev.clone().to(DEV)
    kernels.linear_generic(a.to(DEV), w.to(DEV), bias.to(DEV), many, n, epi)
    few = prev.clone().to(DEV)
    kernels.linear_generic(a.to(DEV), w.to(DEV), bias.to(DEV), few, n_few, epi)
    assert torch.equal(few[:n_few], many[:n_few])
    assert torch.equal(few[n_few:], prev[n_few:].to(DEV)), "rows beyond n_rows were written"
    helpers.assert_close(few[:n_few], _linear_want(a, w, bias, epi, prev)[:n_few],
                         "float32" if "bfloat16" not in (a_dt, w_dt, o_dt) else "bfloat16", "few rows")


@pytest.mark.parametrize("k", [1, 3, 36, 40, 75, 130])
@pytest.mark.parametrize("n", [5, 70])
@pytest.mark.parametrize("a_dt,w_dt,o_dt", [("float32", "float32", "float32"), ("bfloat16", "bfloat16", "bfloat16")])
def test_linear_generic_takes_any_inner_size(a_dt, w_dt, o_dt, n, k):
    """Inner sizes that are no multiple of the kernels' stages (16 and 64), few rows and many: the
    stage's tail is zeros, the row's result the same chain of multiply-adds."""
    g = torch.Generator().manual_seed(k)
    o = 37
    a, w, bias = rnd(g, n + 1, k, dtype=a_dt), rnd(g, o, k, dtype=w_dt), rnd(g, o)
    a[n] = float("nan")         # the row behind the last one is never read into a sum
    out = torch.full((n + 1, o), 7.0, dtype=TDT[o_dt], device=DEV)
    kernels.linear_generic(a.to(DEV), w.to(DEV), bias.to(DEV), out, n, kernels.EPI_GELU)
    helpers.assert_close(out[:n], _linear_want(a[:n], w, bias, kernels.EPI_GELU, None), o_dt if o_dt == "bfloat16" else "float32",
                         f"inner size {k}")
    assert (out[n] == 7.0).all()


@pytest.mark.parametrize("k", [1, 15, 17, 64, 65, 128, 192, 193, 256, 258, 300, 512, 4100, 4352])
def test_float32_product_keeps_its_sums_whatever_the_tiles(k):
    """A product that is float32 throughout goes to one of several kernels by its size: a workgroup per 16 x 16 outputs, whose waves
    have groups of 32 k or blocks of 256, tiles of 64 x 64 and of 128 x 128, and for inner sizes of whole groups these without
    checks and tiles of 32 x 32.  An element's bits are the same in all, also where rows of the operands are not 16-byte aligned;
    the error against 64 bits is that of float32 sums (a chain of eight groups of 32 k in a block of 256, then the blocks: below
    1e-6 of the result's norm)."""
    g = torch.Generator().manual_seed(k)
    o, n = 3501, 1030                                  # 9 x 28 tiles of 128 x 128, all but the last row and column whole
    a, w, bias = rnd(g, n, k + 3).to(DEV), rnd(g, o, k).to(DEV), rnd(g, o).to(DEV)
    whole = torch.empty(n, o, device=DEV)
    assert kernels.linear_exact_kernel(n, o, k, aligned=False) == "tile128"
    kernels.linear_generic(a[:, :k], w, bias, whole, n)          # a row stride that is not the inner size
    want = a[:, :k].double() @ w.double().T + bias.double()
    assert ((whole.double() - want).norm() / want.norm()).item() < 1e-6
    used = set()
    for rows, cols in ((1, o), (16, o), (17, 37), (70, 200), (130, o), (300, 515), (n, 130), (n, 1500), (1025, 3456), (n, 3500)):
        used.add(kernels.linear_exact_kernel(rows, cols, k, aligned=k % 4 == 0))
        part = torch.full((rows + 1, cols), 7.0, device=DEV)
        kernels.linear_generic(a[:rows, :k].contiguous(), w[:cols].contiguous(), bias[:cols].contiguous(), part, rows)
        assert torch.equal(part[:rows], whole[:rows, :cols]), f"{rows} rows, {cols} columns"
        assert (part[rows] == 7.0).all()
    assert used == ({"rows", "tile64", "tile128"} if k % 32 else {"rows", "lds32", "lds64", "lds128"})


@pytest.mark.parametrize("n,k,o,kernel", [(5, 64, 257, "rows"), (20, 700, 640, "rows"), (40, 1100, 2300, "rows"), (300, 384, 768, "lds32"),
                                          (600, 320, 515, "lds32"), (129, 32, 1500, "lds32"), (1030, 96, 1500, "lds64"),
                                          (1030, 192, 1500, "lds64"), (1030, 160, 3501, "lds128"), (500, 301, 900, "tile64"),
                                          (1030, 65, 3498, "tile128"), (9, 1030, 64, "parts"), (40, 600, 132, "parts")])
def test_float32_product_of_infinities_and_in_float32_precision(n, k, o, kernel):
    """Float32 operands taken apart into three bfloat16 each: infinities, NaN and values that bfloat16 rounds to infinity come out as
    float32 multiply-adds give them, in the rows and columns that they are in and nowhere else; all other elements are within
    2e-7 of the norm of the product in 64 bits (a sum over k / 32 groups with six roundings each, of 2^-25 in the mean, is off
    by 2^-25 sqrt(6 + k / 32) at most where no partial sum is larger than the result: 1.9e-7 at 1,100), which the sum of
    single products is not from a k of 128 on."""
    g = torch.Generator().manual_seed(n + k)
    a, w = rnd(g, n, k), rnd(g, o, k, scale=0.05)
    a[0, 0], a[0, 5], a[1, k - 1], a[2, 31] = float("inf"), 0.5, float("-inf"), float("nan")
    w[3, 2], w[4, k - 1], w[5, 1] = float("inf"), float("nan"), 3.4e38
    a[n - 1, 1], a[:n - 1, 1] = 1e-3, 0.0
    want = (a.double() @ w.double().T).float()
    got = torch.full((n, o), 7.0, device=DEV)
    if kernel == "parts":
        sums = torch.empty(kernels.linear_exact_blocks(k), n, o, device=DEV)
        kernels.linear_exact_parts(a.to(DEV), w.to(DEV), sums, n)
        got = sums.sum(dim=0)
    else:
        assert kernels.linear_exact_kernel(n, o, k, aligned=k % 4 == 0) == kernel
        kernels.linear_generic(a.to(DEV), w.to(DEV), None, got, n)
    got, finite = got.cpu(), want.isfinite()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got[want.isinf()], want[want.isinf()])
    assert finite[3:, 6:].all() and torch.isclose(got[n - 1, 5], want[n - 1, 5], rtol=1e-6)
    part, exact = got[3:, 6:].double(), a[3:].double() @ w[6:].double().T
    assert ((part - exact).norm() / exact.norm()).item() < 2e-7


@pytest.mark.parametrize("a_size,w_size", [(1e-33, 1), (1e-35, 1), (1, 1e-37), (1e-40, 1e6), (1e-35, 1e25), (1e-18, 1e-18), (1e30, 1e-30),
                                           (1e30, 1e3)])
@pytest.mark.parametrize("n,k,o", [(5, 64, 257), (40, 1100, 2300), (300, 384, 768), (1030, 192, 1500), (1030, 160, 3501), (500, 301, 900)])
def test_float32_product_of_the_smallest_and_largest_operands(n, k, o, a_size, w_size):
    """Operands down to denormal ones, in each kernel: as close to 64 bits as others are, where the product is a float32 number that
    is not denormal (1e-35 times its own last bit is denormal: 2^-149 / 1e-35 is 1e-10); 1e-40 itself has 2^16 steps, which the product in
    64 bits is of too.  The bound is that of float32 sums, which the largest ones are computed by."""
    g = torch.Generator().manual_seed(n)
    a, w = (rnd(g, n, k).double() * a_size).float(), (rnd(g, o, k).double() * w_size).float()
    got = torch.empty(n, o, device=DEV)
    kernels.linear_generic(a.to(DEV), w.to(DEV), None, got, n)
    want = a.double() @ w.double().T
    unit = want.abs().max()
    assert (((got.cpu().double() - want) / unit).norm() / (want / unit).norm()).item() < 5e-7
    if o % 4 == 0:
        sums = torch.empty(kernels.linear_exact_blocks(k), n, o, device=DEV)
        kernels.linear_exact_parts(a.to(DEV), w.to(DEV), sums, n)
        assert (((sums.cpu().double().sum(dim=0) - want) / unit).norm() / (want / unit).norm()).item() < 5e-7


@pytest.mark.parametrize("n,o", [(5, 64), (17, 260), (300, 515), (1030, 1500), (1030, 3500)])
def test_float32_product_of_an_inner_size_of_one(n, o):
    """One product is rounded once, in each kernel that takes inner sizes which are no whole groups."""
    g = torch.Generator().manual_seed(n)
    a, w = rnd(g, n, 1).to(DEV), rnd(g, o, 1).to(DEV)
    got = torch.empty(n, o, device=DEV)
    kernels.linear_generic(a, w, None, got, n)
    assert torch.equal(got, a * w.T)
    if o % 4 == 0:
        sums = torch.empty(1, n, o, device=DEV)
        kernels.linear_exact_parts(a, w, sums, n)
        assert torch.equal(sums[0], a * w.T)


@pytest.mark.parametrize("k", [769, 1001, 1025, 1028, 1149, 1152, 1280, 2300, 4100, 4609])
def test_float32_product_of_few_rows_under_long_inner_sizes(k):
    """A wave has two groups of 32 k at a time, three from an inner size of 1,025 on, or a block of 256 from 1,153 on, of which the last
    may end anywhere, in one round or two (beyond 16 blocks): the bits of the sums over blocks, added up in order."""
    g = torch.Generator().manual_seed(k)
    for rows, cols in ((1, 300), (16, 52), (17, 132), (40, 900)):
        a, w = rnd(g, rows, k).to(DEV), rnd(g, cols, k).to(DEV)
        assert kernels.linear_exact_kernel(rows, cols, k, aligned=k % 4 == 0) == "rows"
        got = torch.full((rows + 1, cols), 7.0, device=DEV)
        kernels.linear_generic(a, w, None, got, rows)
        sums = torch.empty(kernels.linear_exact_blocks(k), rows, cols, device=DEV)
        kernels.linear_exact_parts(a, w, sums, rows)
        total = torch.zeros(rows, cols, device=DEV)
        for block in sums:
            total += block
        assert torch.equal(got[:rows], total) and (got[rows] == 7.0).all(), f"{rows} rows, {cols} columns"


@pytest.mark.parametrize("k", [37, 320, 1100, 2048])
@pytest.mark.parametrize("large,beside", [(3.4e38, 1.0), (1e33, 1e-33)])
def test_float32_product_done_again_has_the_same_bits_whatever_the_tiles(k, large, beside):
    """Elements of rows with a value whose parts are not finite, computed once more in float32, in each kernel, beside rows that are
    not; also where that value's product is no larger than the others', so that the bits of the other blocks show."""
    g = torch.Generator().manual_seed(k)
    o, n = 1500, 1030
    a, w = rnd(g, n, k).to(DEV), rnd(g, o, k, scale=0.05).to(DEV)
    a[::3, k // 2] = large
    w[:, k // 2] *= beside
    whole = torch.empty(n, o, device=DEV)
    kernels.linear_generic(a, w, None, whole, n)
    want = a.double() @ w.double().T
    assert whole.isfinite().all() and ((whole.double() - want).norm(dim=1) / want.norm(dim=1)).max().item() < 1e-6
    for rows, cols in ((1, o), (17, 37), (70, 200), (130, o), (300, 515), (n, 130)):
        part = torch.empty(rows, cols, device=DEV)
        kernels.linear_generic(a[:rows], w[:cols].contiguous(), None, part, rows)
        assert torch.equal(part, whole[:rows, :cols]), f"{rows} rows, {cols} columns"
        if cols % 4 == 0:
            sums = torch.empty(kernels.linear_exact_blocks(k), rows, cols, device=DEV)
            kernels.linear_exact_parts(a[:rows], w[:cols].contiguous(), sums, rows)
            total = torch.zeros(rows, cols, device=DEV)
            for block in sums:
                total += block
            assert torch.equal(total, whole[:rows, :cols]), f"{rows} rows, {cols} columns, sums over blocks"


@pytest.mark.parametrize("n,k,o,parts", [(1201, 2048, 512, False), (1201, 512, 2048, False), (4, 3072, 768, False), (64, 768, 2304, False),
                                         (500, 1001, 900, False), (16, 3072, 768, True)])
def test_float32_product_of_nan_rows_takes_no_multiple_of_its_time(n, k, o, parts):
    """All elements are computed once more: on the matrix cores' float32 rate, 16 / 6 of the bfloat16 parts' work, with operands
    straight from memory (measured 2 to 5 times in all; a serial sum an element took 30 to 300 times)."""
    def us(a):
        call = (lambda: kernels.linear_exact_parts(a, w, out, n)) if parts else (lambda: kernels.linear_generic(a, w, None, out, n))
        times = []
        for _ in range(8):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(20):
                call()
            end.record()
            end.synchronize()
            times.append(start.elapsed_time(end) * 50)
        return sorted(times)[2]

    g = torch.Generator().manual_seed(n)
    a, w = rnd(g, n, k).to(DEV), rnd(g, o, k).to(DEV)
    out = torch.empty((kernels.linear_exact_blocks(k), n, o) if parts else (n, o), device=DEV)
    plain, nan = us(a), us(torch.full_like(a, float("nan")))
    assert out.isnan().all()
    assert nan < 10 * plain, f"{nan:.0f} us with rows of NaN, {plain:.0f} without"


@pytest.mark.parametrize("epi", [kernels.EPI_NONE, kernels.EPI_GELU, kernels.EPI_RESIDUAL])
@pytest.mark.parametrize("n,k,o,kernel", [(300, 768, 768, "lds32"), (97, 768, 2303, "lds32"), (129, 32, 1500, "lds32"),
                                          (600, 512, 515, "lds32"), (1201, 2048, 512, "lds64"), (255, 96, 1024, "lds32"),
                                          (1030, 64, 1500, "lds64"), (400, 512, 2048, "lds64"), (1030, 160, 3501, "lds128"),
                                          (1500, 96, 2000, "tile64"), (3400, 160, 3072, "lds128")])
def test_float32_product_straight_into_lds(n, k, o, kernel, epi):
    """Aligned rows of whole groups, of which nothing is checked, in tiles of 32 x 32, 64 x 64 and 128 x 128, with one step and with
    more, and 64 x 64 tiles that keep steps of one group: the bits of the same product over rows that are not aligned for that."""
    g = torch.Generator().manual_seed(n + k)
    assert kernels.linear_exact_kernel(n, o, k) == kernel and not kernels.linear_exact_kernel(n, o, k, aligned=False).startswith("lds")
    a, w, bias, old = rnd(g, n, k + 1).to(DEV)[:, :k], rnd(g, o, k).to(DEV), rnd(g, o).to(DEV), rnd(g, n + 1, o).to(DEV)
    want, got = old.clone(), old.clone()
    kernels.linear_generic(a, w, bias, want, n, epi)
    kernels.linear_generic(a.contiguous(), w, bias, got, n, epi)
    assert torch.equal(got, want) and torch.equal(got[n], old[n])


@pytest.mark.parametrize("n,k,o,kernel,unaligned", [
    (16, 3072, 768, "rows", "rows"), (188, 768, 768, "rows", "rows"), (190, 768, 768, "lds32", "rows"),
    (300, 768, 1600, "lds32", "tile64"), (300, 768, 2304, "lds64", "tile64"), (300, 800, 2304, "lds32", "tile64"),
    (40, 768, 8400, "lds32", "rows"), (400, 768, 2304, "lds64", "tile64"), (2000, 512, 2048, "lds128", "tile128"),
    (2000, 96, 1000, "lds64", "tile64"), (2300, 96, 1000, "tile64", "tile64"),            # 512 and 576 tiles
    (700, 384, 3000, "tile64", "tile64"), (1500, 384, 3000, "lds64", "tile64"),           # a third round hardly begun, or more
    (2000, 192, 3000, "lds64", "tile64"), (4400, 192, 3000, "tile64", "tile64"), (4400, 256, 3000, "lds64", "tile64"),
    (3400, 768, 3072, "lds128", "tile128"), (4096, 768, 3072, "lds128", "tile128"), (5000, 768, 3072, "lds128", "tile128"),
    (4096, 1152, 3072, "lds128", "tile128"), (4096, 96, 3072, "lds128", "tile128")])
def test_float32_product_kernel_by_size(n, k, o, kernel, unaligned):
    """Both sides of the lines between the kernels."""
    assert kernels.linear_exact_kernel(n, o, k) == kernel and kernels.linear_exact_kernel(n, o, k, aligned=False) == unaligned


@pytest.mark.parametrize("epi", [kernels.EPI_GELU, kernels.EPI_RESIDUAL, kernels.EPI_RELU2])
@pytest.mark.parametrize("k,o", [(64, 3500), (300, 3501), (37, 3499)])
def test_float32_product_epilogues_whatever_the_tiles(k, o, epi):
    """The epilogues of the three kernels, with 16-byte stores (3,500 columns) and without: the same bits in all, and those
    of the plain product behind the plain function (a sum, a square) or within float32 rounding of it (GELU)."""
    g, n = torch.Generator().manual_seed(o + epi), 1030
    a, w, bias, old = rnd(g, n, k).to(DEV), rnd(g, o, k, scale=k ** -0.5).to(DEV), rnd(g, o).to(DEV), rnd(g, n, o).to(DEV)
    plain = torch.empty(n, o, device=DEV)
    kernels.linear_generic(a, w, bias, plain, n)
    used, got = set(), {}
    for rows, cols in ((n, o), (20, o), (300, 1540), (300, 1537), (n, 1500)):
        used.add(kernels.linear_exact_kernel(rows, cols, k, aligned=k % 4 == 0))
        out = old[:rows + 1, :cols].clone(memory_format=torch.contiguous_format)
        kernels.linear_generic(a[:rows].contiguous(), w[:cols].contiguous(), bias[:cols].contiguous(), out, rows, epi)
        got[rows, cols] = out[:rows]
        assert torch.equal(got[rows, cols], got[n, o][:rows, :cols]) and (rows == n or torch.equal(out[rows], old[rows, :cols]))
    assert used == ({"rows", "tile64", "tile128"} if k % 32 else {"rows", "lds32", "lds64", "lds128"})
    if epi == kernels.EPI_RESIDUAL:
        assert torch.equal(got[n, o], old + plain)
    elif epi == kernels.EPI_RELU2:
        assert torch.equal(got[n, o], torch.relu(plain) ** 2)
    else:
        helpers.assert_close(got[n, o], torch.nn.functional.gelu(plain.double(), approximate="tanh"), "float32", "GELU")


@pytest.mark.parametrize("n,k,h,hk,d,kernel", [
    (1, 64, 4, 4, 16, "rows"), (16, 300, 3, 1, 10, "rows"), (40, 36, 3, 3, 12, "rows"), (300, 512, 8, 8, 64, "lds32"),
    (300, 36, 8, 8, 64, "tile64"), (1030, 256, 24, 20, 128, "lds64"), (70, 33, 1, 1, 33, "rows"), (1030, 256, 100, 37, 20, "lds128"),
    (1030, 65, 60, 23, 33, "tile128"), (1025, 300, 10, 9, 124, "tile128")])
def test_float32_product_stores_keys_and_values(n, k, h, hk, d, kernel):
    """The projection that also stores its key and value columns into their pages: the same bits as the plain product
    followed by the kernel that copies them, in each of the product's kernels and also where no four columns of a head
    lie together; a padded row (slot -1) is stored nowhere."""
    g = torch.Generator().manual_seed(n)
    q_width, kv_width, page = h * d, hk * d, 5
    o = q_width + 2 * kv_width
    assert kernels.linear_exact_kernel(n, o, k, aligned=k % 4 == 0) == kernel
    a, w, bias = rnd(g, n, k).to(DEV), rnd(g, o, k).to(DEV), rnd(g, o).to(DEV)
    pages = -(-n // page) + 1
    slots = torch.randperm(pages * page, generator=g)[:n].to(torch.int32)
    slots[n // 2] = -1 if n > 1 else slots[n // 2]
    slots = slots.to(DEV)
    got, want = torch.full((n, o), 7.0, device=DEV), torch.full((n, o), 7.0, device=DEV)
    pools = [torch.full((pages, hk, page, d), float("nan"), device=DEV) for _ in range(4)]
    assert kernels.linear_exact_qkv(a, w, bias, got, n, (pools[0], pools[1], slots, q_width, kv_width))
    kernels.linear_generic(a, w, bias, want, n)
    kernels.kv_write(want, q_width, q_width + kv_width, pools[2], pools[3], slots, n)
    assert torch.equal(got, want)
    assert torch.equal(pools[0].nan_to_num(9.0), pools[2].nan_to_num(9.0))
    assert torch.equal(pools[1].nan_to_num(9.0), pools[3].nan_to_num(9.0))


@pytest.mark.parametrize("n,k,h,d", [(1, 4, 1, 4), (3, 64, 4, 16), (16, 128, 2, 64), (17, 132, 3, 20), (16, 256, 4, 64), (5, 260, 5, 32),
                                     (16, 512, 8, 64), (33, 512, 2, 64), (2, 516, 2, 36), (16, 768, 12, 64), (1, 640, 10, 64)])
@pytest.mark.parametrize("gather,with_bias", [(False, True), (True, False)])
def test_float32_product_that_norms_its_rows_has_the_bits_of_both_kernels(n, k, h, d, gather, with_bias):
    """The product with the LayerNorm inside, plain, with an activation and with keys and values into their pages, against the
    LayerNorm kernel and the product behind it: the same bits, in rows with an infinity and a NaN too."""
    gen = torch.Generator().manual_seed(n * 1000 + k)
    x = rnd(gen, n + 5, k, scale=2.0)
    x[0, 1], x[n // 2, k - 1] = float("inf"), float("nan")
    x[n - 1] = 3.0 + 1e-3 * rnd(gen, k)                     # far from zero, nearly equal
    x = x.to(DEV)
    rows = torch.randperm(n + 5, generator=gen)[:n].to(torch.int32).to(DEV) if gather else None
    gain, shift = rnd(gen, k).to(DEV), rnd(gen, k).to(DEV) if with_bias else None
    o = 3 * h * d
    w, bias = rnd(gen, o, k, scale=k ** -0.5).to(DEV), rnd(gen, o).to(DEV) if with_bias else None
    assert kernels.linear_exact_norms(n, o, k)
    normed = torch.empty(n, k, device=DEV)
    kernels.layer_norm(x, gain, shift, normed, n, 1e-5, rows)
    for epi in (kernels.EPI_NONE, kernels.EPI_GELU, kernels.EPI_RELU2):
        want, got = torch.empty(n, o, device=DEV), torch.full((n + 1, o), 7.0, device=DEV)
        kernels.linear_generic(normed, w, bias, want, n, epi)
        assert kernels.linear_exact_normed(x, gain, shift, 1e-5, w, bias, got, n, epi, rows)
        assert torch.equal(got[:n].nan_to_num(nan=1e30), want.nan_to_num(nan=1e30)) and (got[n] == 7.0).all()
    slots = torch.randperm(48, generator=gen)[:n].to(torch.int32)
    slots[n - 1] = -1
    results = []
    for inside in (False, True):
        pools = torch.full((2, 3, h, 16, d), 7.0, device=DEV)
        out = torch.full((n, o), 7.0, device=DEV)
        scatter = (pools[0], pools[1], slots.to(DEV), h * d, h * d)
        if inside:
            assert kernels.linear_exact_normed(x, gain, shift, 1e-5, w, bias, out, n, rows=rows, scatter=scatter)
        else:
            assert kernels.linear_exact_qkv(normed, w, bias, out, n, scatter)
        results.append((out.nan_to_num(nan=1e30), pools.nan_to_num(nan=1e30)))
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])


@pytest.mark.parametrize("n,o,k,norms", [(16, 4096, 512, True), (16, 4097, 512, False), (32, 2048, 512, True), (33, 2048, 512, False),
                                         (3, 300, 768, True), (3, 300, 772, False), (3, 300, 66, False),
                                         (16, 4096, 516, True), (17, 1536, 640, True), (17, 1537, 640, False), (32, 2048, 516, False),
                                         (64, 768, 768, True), (64, 784, 768, False)])
def test_which_float32_products_norm_their_rows(n, o, k, norms):
    assert kernels.linear_exact_norms(n, o, k) == norms
    if not norms:
        x, gain, w = torch.zeros(n, k, device=DEV), torch.ones(k, device=DEV), torch.zeros(o, k, device=DEV)
        assert not kernels.linear_exact_normed(x, gain, None, 1e-5, w, None, torch.zeros(n, o, device=DEV), n)


@pytest.mark.parametrize("n,k,o", [(1, 64, 16), (8, 768, 8192), (9, 1030 // 8 * 8, 8200), (12, 2048, 8193), (16, 40, 33), (3, 4096, 100), (16, 320, 48),
                                   (16, 8, 40), (16, 56, 20), (5, 2120, 50), (16, 2744, 33), (7, 312, 40), (16, 328, 20), (3, 440, 33), (2, 504, 17)])
@pytest.mark.parametrize("o_dt", ["float32", "bfloat16"])
def test_linear_rows_once(n, k, o, o_dt):
    """A pass over the matrix for up to 16 rows: one stage and two, inner sizes that are no whole steps, ragged columns."""
    g = torch.Generator().manual_seed(n * k + o)
    a, w = rnd(g, n, k, dtype="bfloat16"), rnd(g, o, k, dtype="bfloat16", scale=k ** -0.5)
    out = torch.full((n + 1, o), 7.0, dtype=torch.float32 if o_dt == "float32" else torch.bfloat16, device=DEV)
    assert kernels.linear_rows_once(a.to(DEV), w.to(DEV), out, n)
    helpers.assert_close(out[:n], a.double() @ w.double().T, o_dt, f"{n} {k} {o}")
    assert (out[n] == 7.0).all()


@pytest.mark.parametrize("n,k,o,once", [
    (4, 2048, 14336, False), (5, 2048, 14336, True), (12, 2048, 14336, True), (13, 2048, 14336, False), (8, 2048, 14320, False), (8, 1024, 50257, False),
    (9, 1024, 16384, False), (8, 1600, 16384, False), (12, 4096, 8192, True), (13, 4096, 8192, False), (4, 4096, 8208, True), (5, 4096, 8208, False),
    (12, 4096, 11264, True), (8, 6144, 8192, True), (9, 6144, 8192, False), (3, 6144, 9216, True), (4, 6144, 9216, False), (6, 10240, 8192, True),
    (7, 10240, 8192, False)])
def test_which_very_wide_outputs_go_once_over_the_matrix(monkeypatch, n, k, o, once):
    """Through the entry that chooses, on both sides of the lines: few rows go to the kernel that reads the matrix once, and nothing
    else does."""
    from types import SimpleNamespace

    from mini_gpt_inference_amd.ops import linear as L
    from mini_gpt_inference_amd.parts.base import Workspace

    calls, plain = [], kernels.linear_rows_once
    monkeypatch.setattr(kernels, "linear_rows_once", lambda *args: calls.append(plain(*args)) or calls[-1])
    g = torch.Generator().manual_seed(n + k)
    a = rnd(g, n, k, dtype="bfloat16").to(DEV)
    w = (torch.randn(o, k, device=DEV, generator=torch.Generator(DEV).manual_seed(n)) * k ** -0.5).to(torch.bfloat16)
    ctx = SimpleNamespace(exact=False, dtype=torch.bfloat16, n_rows=n, pending=None, copy_budget=None, workspace=Workspace(torch.device(DEV)))
    out = torch.empty(n, o, device=DEV)
    L.linear(ctx, a, w, None, out, n)
    assert calls == ([True] if once else [])
    helpers.assert_close(out, a.double() @ w.double().T, "float32", f"{n} {k} {o}")


@pytest.mark.parametrize("n,k,o", [(6, 2048, 16384), (3, 4096, 8192), (13, 2048, 16384), (4, 512, 8192)])
@pytest.mark.parametrize("o_dt", ["float32", "bfloat16"])
def test_very_wide_output_into_a_wider_buffer(n, k, o, o_dt):
    """Few rows in one pass over the matrix, and the kernels around that: what lies beside the output's columns is left alone."""
    from types import SimpleNamespace

    from mini_gpt_inference_amd.ops import linear as L
    from mini_gpt_inference_amd.parts.base import Workspace

    g = torch.Generator().manual_seed(n)
    a, w = rnd(g, n, k, dtype="bfloat16").to(DEV), rnd(g, o, k, dtype="bfloat16", scale=k ** -0.5).to(DEV)
    ctx = SimpleNamespace(exact=False, dtype=torch.bfloat16, n_rows=n, pending=None, copy_budget=None, workspace=Workspace(torch.device(DEV)))
    out = torch.full((n + 1, o + 24), 7.0, dtype=TDT[o_dt], device=DEV)
    L.linear(ctx, a, w, None, out, n)
    helpers.assert_close(out[:n, :o], (a.double() @ w.double().T).cpu(), o_dt if o_dt == "bfloat16" else "float32", f"{n} {k} {o}")
    assert (out[n] == 7.0).all() and (out[:, o:] == 7.0).all()


@pytest.mark.parametrize("n,k,o", [(1, 1, 4), (1, 1537, 512), (3, 256, 60), (4, 3072, 768), (16, 257, 64), (17, 1026, 68),
                                   (17, 3072, 768), (33, 5000, 260), (70, 2048, 2048), (128, 768, 1028), (130, 4097, 1600)])
def test_float32_product_left_as_sums_over_its_blocks(n, k, o):
    """The sums over the blocks of k, added up by the LayerNorm that reads the rows next (all rows, some of them, or with no
    LayerNorm at all): the same bits as the product that adds to the residual and the LayerNorm of that."""
    g = torch.Generator().manual_seed(n + k)
    a, w, x = rnd(g, n, k + k % 4).to(DEV)[:, :k], rnd(g, o, k).to(DEV), rnd(g, n, o).to(DEV)
    bias, gain, beta = rnd(g, o).to(DEV), rnd(g, o).to(DEV), rnd(g, o).to(DEV)
    rows = i32([(7 * i) % n for i in range(min(n, 5))])
    for b, shift in ((bias, beta), (None, None)):
        want_x, want, want_rows = x.clone(), torch.empty_like(x), torch.empty(len(rows), o, device=DEV)
        kernels.linear_generic(a, w, b, want_x, n, kernels.EPI_RESIDUAL)
        kernels.layer_norm(want_x, gain, shift, want, n, 1e-5)
        kernels.layer_norm(want_x, gain, shift, want_rows, len(rows), 1e-5, rows)
        sums = torch.full((kernels.linear_exact_blocks(k), n, o), float("nan"), device=DEV)
        kernels.linear_exact_parts(a, w, sums, n)
        got_x, got, got_rows, settled = x.clone(), torch.empty_like(x), torch.empty_like(want_rows), torch.empty_like(x)
        pending = PendingSums(got_x, sums, len(sums), exact=True, bias=b)
        assert kernels.residual_layer_norm(pending, gain, shift, 1e-5, rows, got_rows, len(rows))
        assert kernels.residual_settle(pending, settled, n)
        assert kernels.residual_layer_norm(pending, gain, shift, 1e-5, None, got, n, settled=got_x)
        assert torch.equal(got_x, want_x) and torch.equal(settled, want_x)
        assert torch.equal(got, want) and torch.equal(got_rows, want_rows)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_linear_generic_refuses_epilogues_that_it_does_not_have(dtype):
    """The code that sends key and value columns to their pages among them: the plain product has no pages to send them to."""
    a, w = torch.zeros(4, 40, dtype=getattr(torch, dtype), device=DEV), torch.zeros(8, 40, dtype=getattr(torch, dtype), device=DEV)
    out = torch.full((4, 8), 7.0, dtype=a.dtype, device=DEV)
    for epilogue in (kernels.SK_EPI_QKV, 4, 6, -1):
        with pytest.raises(kernels.KernelError):
            kernels.linear_generic(a, w, None, out, 4, epilogue)
    assert (out == 7.0).all()


def test_linear_generic_refuses_tensors_off_the_gpu():
    a, w = torch.zeros(4, 40, device=DEV), torch.zeros(8, 40, device=DEV)
    with pytest.raises(kernels.KernelError, match="GPU"):
        kernels.linear_generic(a.cpu(), w, None, torch.zeros(4, 8, device=DEV), 4)


# general=False lets the kernel for a decode step's rows (at most 16, inner size a multiple of 32)
# take what it can; general=True keeps every case on the kernel for up to 64 rows
@pytest.mark.parametrize("general", [False, True])
@pytest.mark.parametrize("n,k,o", [(1, 64, 257), (8, 512, 1536), (17, 96, 503), (33, 80, 48), (64, 2048, 512), (40, 512, 1536), (24, 768, 48), (60, 96, 64), (50, 768, 1003),
                                   (5, 48, 16), (16, 160, 503), (12, 1600, 48), (7, 2048, 512), (3, 32, 20),
                                   (9, 768, 130)])
@pytest.mark.parametrize("epi,o_dt", [(kernels.EPI_NONE, "bfloat16"), (kernels.EPI_NONE, "float32"),
                                      (kernels.EPI_GELU, "bfloat16"), (kernels.EPI_RESIDUAL, "float32")])
def test_linear_skinny(n, k, o, epi, o_dt, general):
    g = torch.Generator().manual_seed(3)
    a, w, bias = rnd(g, n + 2, k, dtype="bfloat16"), rnd(g, o, k, dtype="bfloat16", scale=k ** -0.5), rnd(g, o)
    prev = rnd(g, n + 2, o, dtype=o_dt)
    out = prev.clone().to(DEV)
    assert kernels.linear_skinny(a.to(DEV), w.to(DEV), bias.to(DEV), out, n, epi, general_only=general)
    if not general and k % 32 == 0:
        # the same product from the packed copy of the matrix: the same sums in the same order
        packed = kernels.pack_weight(w.to(DEV))
        out_p = prev.clone().to(DEV)
        assert kernels.linear_skinny(a.to(DEV), w.to(DEV), bias.to(DEV), out_p, n, epi, w_packed=packed)
        assert torch.equal(out_p, out), "the packed matrix gives another result"
        # more than 16 rows: all rows in one workgroup per column tile, or 16 rows to a workgroup
        for mode in (kernels.ROWS_SHARE_W, kernels.ROWS_GROUPS):
            out_m = prev.clone().to(DEV)
            assert kernels.linear_skinny(a.to(DEV), w.to(DEV), bias.to(DEV), out_m, n, epi, w_packed=packed,
                                         rows_mode=mode)
            helpers.assert_close(out_m[:n], _linear_want(a, w, bias, epi, prev)[:n], "bfloat16", f"rows mode {mode}")
            assert torch.equal(out_m[n:], prev[n:].to(DEV)), "rows beyond n_rows were written"
        # 16, 8, 4 or 1 rows to a workgroup: the same sums whatever the groups
        outs = []
        for rpg in (16, 8, 1):
            out_g = prev.clone().to(DEV)
            assert kernels.linear_skinny(a.to(DEV), w.to(DEV), bias.to(DEV), out_g, n, epi, w_packed=packed,
                                         rows_mode=kernels.ROWS_GROUPS, rows_per_group=rpg)
            outs.append(out_g)
        assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2]), "the groups' size changes the result"
        helpers.assert_close(outs[2][:n], _linear_want(a, w, bias, epi, prev)[:n], "bfloat16", "groups of 1 row")
        assert torch.equal(outs[2][n:], prev[n:].to(DEV)), "rows beyond n_rows were written"
    helpers.assert_close(out[:n], _linear_want(a, w, bias, epi, prev)[:n], "bfloat16", f"skinny {n}x{k}x{o}")
    assert torch.equal(out[n:], prev[n:].to(DEV)), "rows beyond n_rows were written"
    out2 = prev.clone().to(DEV)
    assert kernels.linear_skinny(a.to(DEV), w.to(DEV), None, out2, n, epi, general_only=general)
    helpers.assert_close(out2[:n], _linear_want(a, w, None, epi, prev)[:n], "bfloat16", "skinny without bias")


@pytest.mark.parametrize("n,k,o", [(65, 64, 257), (300, 512, 1536), (129, 96, 503), (2048, 80, 48), (128, 2048, 128),
                                   (1000, 48, 130), (600, 1072, 136)])
@pytest.mark.parametrize("epi,o_dt", [(kernels.EPI_NONE, "bfloat16"), (kernels.EPI_NONE, "float32"),
                                      (kernels.EPI_GELU, "bfloat16"), (kernels.EPI_RESIDUAL, "float32")])
def test_linear_mfma(n, k, o, epi, o_dt):
    g = torch.Generator().manual_seed(6)
    a, w, bias = rnd(g, n, k, dtype="bfloat16"), rnd(g, o, k, dtype="bfloat16", scale=k ** -0.5), rnd(g, o)
    prev = rnd(g, n, o, dtype=o_dt)
    out = prev.clone().to(DEV)
    assert kernels.linear_mfma(a.to(DEV), w.to(DEV), bias.to(DEV), out, n, epi)
    helpers.assert_close(out, _linear_want(a, w, bias, epi, prev), "bfloat16", f"mfma {n}x{k}x{o}")
    # rows beyond n_rows are left alone
    out2 = prev.clone().to(DEV)
    assert kernels.linear_mfma(a.to(DEV), w.to(DEV), None, out2, n - 3, epi)
    assert torch.equal(out2[n - 3:], prev[n - 3:].to(DEV))
    helpers.assert_close(out2[:n - 3], _linear_want(a, w, None, epi, prev)[:n - 3], "bfloat16", "mfma partial rows")


@pytest.mark.parametrize("n,k,o", [(300, 80, 257), (513, 512, 520), (256, 2048, 256), (1000, 48, 130), (70, 64, 1030),
                                   (40, 1616, 272)])
@pytest.mark.parametrize("epi,o_dt", [(kernels.EPI_NONE, "bfloat16"), (kernels.EPI_NONE, "float32"),
                                      (kernels.EPI_GELU, "bfloat16"), (kernels.EPI_RESIDUAL, "float32")])
@pytest.mark.parametrize("shape", [0, 1, 2, 3, 4, 5, 6, 7])
def test_linear_mfma_each_tile_shape(n, k, o, epi, o_dt, shape):
    """Each tile shape forced at sizes that cut its tiles everywhere: rows and columns past the end, an
    inner size that ends inside a step, several tiles each way.  Shapes 5 and 6: the 64 x 64 and 32 x 32
    tiles with four steps on their way from memory, in whole rounds of four (inner sizes of 1, 2, 8, 26
    and 32 steps: rounds that end beyond the last step).  Shape 7: the 64 x 64 tile with two wave groups,
    each one half of every step along k (also a last step of which only the first half exists); float32
    outputs only."""
    if shape == 7 and o_dt != "float32":
        a, w = torch.zeros(64, 64, dtype=torch.bfloat16, device=DEV), torch.zeros(64, 64, dtype=torch.bfloat16, device=DEV)
        assert not kernels.linear_mfma(a, w, None, torch.zeros(64, 64, dtype=torch.bfloat16, device=DEV), 64, epi, shape=7)
        return
    g = torch.Generator().manual_seed(16)
    a, w, bias = rnd(g, n, k, dtype="bfloat16"), rnd(g, o, k, dtype="bfloat16", scale=k ** -0.5), rnd(g, o)
    prev = rnd(g, n + 2, o, dtype=o_dt)
    out = prev.clone().to(DEV)
    assert kernels.linear_mfma(a.to(DEV), w.to(DEV), bias.to(DEV), out, n, epi, shape=shape)
    helpers.assert_close(out[:n], _linear_want(a, w, bias, epi, prev[:n]), "bfloat16", f"shape {shape} {n}x{k}x{o}")
    assert torch.equal(out[n:], prev[n:].to(DEV)), "rows beyond n_rows were written"


@pytest.mark.parametrize("n,k,o", [(300, 64, 257), (513, 512, 520), (256, 2048, 256), (1000, 128, 130), (130, 192, 400),
                                   (200, 320, 72), (40, 2112, 272)])
@pytest.mark.parametrize("epi,o_dt", [(kernels.EPI_NONE, "bfloat16"), (kernels.EPI_NONE, "float32"),
                                      (kernels.EPI_GELU, "bfloat16"), (kernels.EPI_RESIDUAL, "float32")])
@pytest.mark.parametrize("shape", [8, 9, 10, 11, 12])
def test_linear_mfma_slices_straight_into_lds(n, k, o, epi, o_dt, shape):
    """The variants whose operand slices go from memory straight into LDS (tiles of 32 x 32 and 64 x 64 with
    four stages, 128 x 64 with three, 128 x 192 with two, 32 x 32 with six), forced at sizes that cut their tiles
    everywhere and at inner sizes of 1, 2, 3, 5, 8, 32 and 33 steps: fewer steps than stages, as many, and more."""
    g = torch.Generator().manual_seed(26)
    a, w, bias = rnd(g, n, k, dtype="bfloat16"), rnd(g, o, k, dtype="bfloat16", scale=k ** -0.5), rnd(g, o)
    prev = rnd(g, n + 2, o, dtype=o_dt)
    out = prev.clone().to(DEV)
    assert kernels.linear_mfma(a.to(DEV), w.to(DEV), bias.to(DEV), out, n, epi, shape=shape)
    helpers.assert_close(out[:n], _linear_want(a, w, bias, epi, prev[:n]), "bfloat16", f"shape {shape} {n}x{k}x{o}")
    assert torch.equal(out[n:], prev[n:].to(DEV)), "rows beyond n_rows were written"


@pytest.mark.parametrize("n,k,o", [(1, 64, 16), (300, 64, 257), (513, 512, 520), (256, 128, 384), (1000, 192, 130), (130, 256, 400),
                                   (257, 320, 193)])
@pytest.mark.parametrize("epi,o_dt", [(kernels.EPI_NONE, "bfloat16"), (kernels.EPI_NONE, "float32"),
                                      (kernels.EPI_GELU, "bfloat16"), (kernels.EPI_RELU2, "bfloat16"),
                                      (kernels.EPI_RESIDUAL, "float32")])
@pytest.mark.parametrize("shape", [13, 14, 15, 16])
def test_linear_mfma_with_its_halves_out_of_step(n, k, o, epi, o_dt, shape):
    """The variants whose two halves read and multiply in turn (256 x 256, 128 x 256, 256 x 192 and 128 x 192), at sizes that cut
    their tiles and at 1, 2, 3, 4, 5 and 8 steps: the sums of an element run over k in the order of the other variants, so the
    results are those of the 32 x 32 tiles bit by bit."""
    g = torch.Generator().manual_seed(n)
    a, w, bias = rnd(g, n, k, dtype="bfloat16"), rnd(g, o, k, dtype="bfloat16", scale=k ** -0.5), rnd(g, o)
    prev = rnd(g, n + 2, o, dtype=o_dt)
    out, small = prev.clone().to(DEV), prev.clone().to(DEV)
    assert kernels.linear_mfma(a.to(DEV), w.to(DEV), bias.to(DEV), out, n, epi, shape=shape)
    assert kernels.linear_mfma(a.to(DEV), w.to(DEV), bias.to(DEV), small, n, epi, shape=8)
    helpers.assert_close(out[:n], _linear_want(a, w, bias, epi, prev[:n]), "bfloat16", f"shape {shape} {n}x{k}x{o}")
    assert torch.equal(out, small)


@pytest.mark.parametrize("n,k,o,shape,shape_f32,shape_added,shape_grouped", [
    (1500, 1600, 4800, 14, 14, 14, 14), (4096, 1600, 6400, 13, 13, 11, 13), (4096, 1600, 4800, 15, 15, 11, 11),
    (4096, 1600, 1600, 14, 14, 14, 14), (2000, 768, 2304, 16, 16, 16, 11), (2000, 3072, 768, 10, 10, 10, 10),
    (511, 1600, 4800, -1, -1, -1, -1), (512, 1600, 4800, 10, 19, 19, 10),       # rows
    (2000, 704, 2304, 11, 11, 11, 11),                                          # 11 steps: the rules for fewer
    (2176, 768, 512, -1, -1, -1, -1), (2240, 768, 512, 10, 10, 10, 10),         # 136 and 144 tiles of 128 x 64
    (1600, 1280, 1280, -1, -1, -1, -1), (1664, 1280, 1280, 10, 19, 19, 10),     # a second round of the 64 x 64 tiles and a third
    (1300, 4096, 1024, 10, 10, 9, 10), (850, 5120, 1280, 10, 10, 10, 10), (5000, 5120, 1280, 14, 14, 14, 14),
    (1600, 2048, 10880, 11, 11, 11, 11), (3300, 5440, 2048, 14, 14, 14, 14), (12288, 3072, 768, 15, 15, 15, 15),
    (4608, 1024, 2048, 15, 15, 11, 11),                                         # groups whose second half may be padding
    (600, 768, 50304, 11, 11, 11, 11), (1024, 768, 50304, 13, 13, 13, 13), (720, 1600, 50304, 13, 13, 13, 13),
    (850, 1600, 50304, 11, 11, 11, 11)])
def test_linear_mfma_choice_among_the_large_variants(n, k, o, shape, shape_f32, shape_added, shape_grouped):
    """What the model of rounds chooses for bfloat16 and float32 outputs, for sums added to float32 rows and for rows in groups, on
    both sides of its lines."""
    assert kernels.linear_mfma_choice(n, o, k, torch.bfloat16) == shape
    assert kernels.linear_mfma_choice(n, o, k, torch.float32) == shape_f32
    assert kernels.linear_mfma_choice(n, o, k, torch.float32, kernels.EPI_RESIDUAL) == shape_added
    assert kernels.linear_mfma_choice(n, o, k, torch.bfloat16, grouped=True) == shape_grouped


@pytest.mark.parametrize("n,k,o", [(1500, 1600, 4800), (1500, 1600, 6400), (4096, 1600, 1600), (6000, 768, 2304), (2000, 768, 2304),
                                   (2000, 3072, 768)])
def test_linear_mfma_of_many_rows_keeps_its_sums_whatever_the_tile(n, k, o):
    """The variant that the model of rounds chooses, forced, gives the same bits; the plain choice is that variant."""
    g = torch.Generator().manual_seed(o)
    a, w, bias = rnd(g, n, k, dtype="bfloat16").to(DEV), rnd(g, o, k, dtype="bfloat16", scale=k ** -0.5).to(DEV), rnd(g, o).to(DEV)
    out, forced = (torch.empty(n, o, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    shape = kernels.linear_mfma_choice(n, o, k, torch.bfloat16)
    assert shape >= 10
    assert kernels.linear_mfma(a, w, bias, out, n, kernels.EPI_NONE)
    assert kernels.linear_mfma(a, w, bias, forced, n, kernels.EPI_NONE, shape=shape)
    assert torch.equal(out, forced)
    want = a.float() @ w.float().T + bias
    assert ((out.float() - want).norm() / want.norm()).item() < 4e-3      # rounding to bfloat16: 2 ** -9 of each value at most


@pytest.mark.parametrize("n,k,o", [(1, 64, 16), (300, 64, 257), (513, 512, 520), (256, 128, 384), (1000, 192, 130), (257, 320, 193)])
@pytest.mark.parametrize("epi", [kernels.EPI_NONE, kernels.EPI_RESIDUAL])
@pytest.mark.parametrize("shape", [19, 23, 25])
def test_linear_mfma_with_two_chains_of_sums(n, k, o, epi, shape):
    """The variants whose float32 sums are two chains, at sizes that cut their tiles and at 1, 2, 3, 5 and 8 steps: the bits of
    the two wave groups that share a 64 x 64 tile, each a chain over its half of every step."""
    g = torch.Generator().manual_seed(n)
    a, w, bias = rnd(g, n, k, dtype="bfloat16"), rnd(g, o, k, dtype="bfloat16", scale=k ** -0.5), rnd(g, o)
    prev = rnd(g, n + 2, o)
    out, groups = prev.clone().to(DEV), prev.clone().to(DEV)
    assert kernels.linear_mfma(a.to(DEV), w.to(DEV), bias.to(DEV), out, n, epi, shape=shape)
    assert kernels.linear_mfma(a.to(DEV), w.to(DEV), bias.to(DEV), groups, n, epi, shape=7)
    helpers.assert_close(out[:n], _linear_want(a, w, bias, epi, prev[:n]), "bfloat16", f"shape {shape} {n}x{k}x{o}")
    assert torch.equal(out, groups)
    assert not kernels.linear_mfma(a.to(DEV), w.to(DEV), bias.to(DEV), out.to(torch.bfloat16), n, kernels.EPI_NONE, shape=shape)


@pytest.mark.parametrize("n,k,o", [(800, 1600, 1600), (2048, 1024, 1024), (4096, 1280, 1280), (3000, 3200, 1600), (6000, 3072, 768)])
@pytest.mark.parametrize("epi", [kernels.EPI_NONE, kernels.EPI_RESIDUAL])
def test_linear_mfma_of_many_rows_keeps_two_chains_of_float32_sums(n, k, o, epi):
    """Float32 outputs of the sizes whose 64 x 64 tiles have two wave groups: whatever tile is chosen, the bits are theirs."""
    g = torch.Generator().manual_seed(o)
    a, w, bias = rnd(g, n, k, dtype="bfloat16").to(DEV), rnd(g, o, k, dtype="bfloat16", scale=k ** -0.5).to(DEV), rnd(g, o).to(DEV)
    out = rnd(g, n, o).to(DEV)
    groups = out.clone()
    assert kernels.linear_mfma(a, w, bias, out, n, epi)
    assert kernels.linear_mfma(a, w, bias, groups, n, epi, shape=7)
    assert torch.equal(out, groups)


@pytest.mark.parametrize("pairs,experts,k,o,epi,dt", [
    (700, 5, 1024, 2048, kernels.EPI_RELU2, "bfloat16"), (900, 9, 2048, 2816, kernels.EPI_NONE, "bfloat16"),
    (1900, 7, 2048, 2816, kernels.EPI_RELU2, "bfloat16"), (900, 9, 768, 2560, kernels.EPI_NONE, "bfloat16"),
    (700, 5, 768, 2600, kernels.EPI_NONE, "float32"), (2000, 17, 768, 1040, kernels.EPI_NONE, "float32"),
    (1500, 14, 4096, 1024, kernels.EPI_NONE, "float32")])
def test_grouped_products_of_many_rows(pairs, experts, k, o, epi, dt):
    """Experts' products through the large variants (inner sizes of 12 steps and more, 140 tiles and more): runs that end inside a
    group of 256 slots, an expert without pairs, groups that nobody uses; every used row has the bits of its expert's own product
    through the 32 x 32 tiles (two chains of sums: through the two wave groups), within the tolerance of the plain one."""
    g = torch.Generator().manual_seed(pairs + o)
    share = torch.rand(experts, generator=g) + 0.2
    share[experts // 2] = 0.0
    table = torch.multinomial(share, pairs, replacement=True, generator=g).to(torch.int32)[:, None].contiguous()
    w = rnd(g, experts, o, k, dtype="bfloat16", scale=k ** -0.5).to(DEV)
    h = rnd(g, pairs, k, dtype="bfloat16").to(DEV)
    slots = kernels.expert_slots(pairs, 1, experts, 256)
    st, sp, te = (torch.zeros(n, dtype=torch.int32, device=DEV) for n in (slots, slots, slots // 256))
    kernels.expert_route(None, None, table.to(DEV), pairs, experts, st, sp, te, 256)
    rows = torch.zeros(slots, k, dtype=torch.bfloat16, device=DEV)
    assert kernels.gather_rows(h, st, rows, slots)
    out = torch.full((slots, o), 7.0, dtype=TDT[dt], device=DEV)
    shape = kernels.linear_mfma_choice(slots, o, k, TDT[dt], epi, grouped=True)
    assert shape >= 10 and int((te < 0).sum()) > 0
    assert kernels.grouped_linear_tiled(rows, w, te, st, out, slots, epi)
    for e in range(experts):
        mine = (table[:, 0] == e).nonzero().flatten().to(DEV)
        if e == experts // 2:
            assert len(mine) == 0
            continue
        used = ((te.repeat_interleave(256) == e) & (st >= 0)).nonzero().flatten()
        assert sorted(st[used].tolist()) == mine.tolist()
        own = torch.empty(len(used), o, dtype=TDT[dt], device=DEV)
        assert kernels.linear_mfma(rows[used], w[e], None, own, len(used), epi, shape=7 if shape >= 17 else 4)
        assert torch.equal(out[used], own), f"expert {e}, shape {shape}"
        plain = rows[used].double() @ w[e].double().T
        want = torch.relu(plain) ** 2 if epi == kernels.EPI_RELU2 else plain
        helpers.assert_close(own, want, "bfloat16", f"expert {e}")


@pytest.mark.parametrize("n,k,o,shape", [(2304, 768, 5632, 13), (1600, 1024, 4096, 14), (2500, 1024, 4096, 15), (1500, 1024, 2816, 16),
                                         (2048, 1024, 2048, 10)])
def test_xielu_behind_a_product_of_many_rows(n, k, o, shape):
    """The activation as the epilogue of the large variants: the bits of the same product through few rows at a time."""
    g = torch.Generator().manual_seed(n)
    assert kernels.linear_mfma_choice(n, o, k, torch.bfloat16) == shape
    a, w = rnd(g, n, k, dtype="bfloat16").to(DEV), rnd(g, o, k, dtype="bfloat16", scale=k ** -0.5).to(DEV)
    bias, coef = rnd(g, o).to(DEV), torch.tensor([0.8, 1.3], device=DEV)
    out, few = (torch.empty(n, o, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    assert kernels.linear_mfma_xielu(a, w, bias, out, n, coef)
    for r in range(0, n, 256):
        rows = min(256, n - r)                 # under 512: none of the large variants
        assert kernels.linear_mfma_xielu(a[r:r + rows], w, bias, few[r:r + rows], rows, coef)
    assert torch.equal(out, few)
    v = a.double() @ w.double().T + bias.double()
    want = torch.where(v > 0, 0.8 * v * v, 1.3 * (torch.expm1(v.clamp(max=0)) - v)) + v / 2
    helpers.assert_close(out, want, "bfloat16", "xielu")


@pytest.mark.parametrize("n,shape,k", [(300, 13, 64), (130, 14, 192), (520, 15, 128), (257, 16, 256)])
def test_linear_mfma_halves_store_keys_and_values(n, shape, k):
    test_linear_mfma_stores_keys_and_values(n, shape, k)


def test_linear_mfma_straight_into_lds_wants_whole_steps():
    """An inner size that is no multiple of 64 is refused by those variants (nothing can be zeroed on its way
    into LDS), and the library's own choice then goes through registers."""
    g = torch.Generator().manual_seed(27)
    n, k, o = 256, 2064, 512
    a, w, bias = rnd(g, n, k, dtype="bfloat16"), rnd(g, o, k, dtype="bfloat16", scale=k ** -0.5), rnd(g, o)
    out = torch.zeros(n, o, device=DEV)
    for shape in (8, 9, 10, 11, 12):
        assert not kernels.linear_mfma(a.to(DEV), w.to(DEV), bias.to(DEV), out, n, kernels.EPI_NONE, shape=shape)
    assert not kernels.linear_mfma(a.to(DEV), w.to(DEV), bias.to(DEV), out, n, kernels.EPI_NONE, shape=13)
    assert kernels.linear_mfma(a.to(DEV), w.to(DEV), bias.to(DEV), out, n, kernels.EPI_NONE)
    helpers.assert_close(out, _linear_want(a, w, bias, kernels.EPI_NONE, None), "bfloat16", "through registers")


@pytest.mark.parametrize("n,k,o,shape", [(256, 2048, 512, 8), (2048, 2048, 512, 9), (2048, 3072, 768, 10), (8192, 512, 1536, 11),
                                         (1024, 3072, 768, 9), (2048, 1600, 4800, 11), (32, 1600, 4800, 12), (64, 1600, 6400, 8)])
def test_linear_mfma_chooses_the_variants_straight_into_lds(n, k, o, shape):
    """A long inner size (32 steps and more) with few tiles, a wide output under many rows, and few rows under
    a large matrix (the rows of a decode step; six stages while the tiles are at most 256): the library takes
    those variants by itself, so its result equals the forced one bit by bit."""
    g = torch.Generator().manual_seed(28)
    a, w, bias = rnd(g, n, k, dtype="bfloat16"), rnd(g, o, k, dtype="bfloat16", scale=k ** -0.5), rnd(g, o)
    prev = rnd(g, n, o)
    out, out_f = prev.clone().to(DEV), prev.clone().to(DEV)
    assert kernels.linear_mfma(a.to(DEV), w.to(DEV), bias.to(DEV), out, n, kernels.EPI_RESIDUAL)
    assert kernels.linear_mfma(a.to(DEV), w.to(DEV), bias.to(DEV), out_f, n, kernels.EPI_RESIDUAL, shape=shape)
    assert torch.equal(out, out_f)
    helpers.assert_close(out, _linear_want(a, w, bias, kernels.EPI_RESIDUAL, prev), "bfloat16", "chosen")


@pytest.mark.parametrize("n,k,o,shape,parts", [(100, 2048, 96, 4, 4), (70, 1040, 132, 3, 2), (300, 6400, 64, 3, 8),
                                                (33, 576, 40, 4, 3), (130, 1600, 260, 2, 4), (64, 1600, 528, 6, 2),
                                                (50, 3200, 96, 5, 4), (48, 6400, 1600, None, 0), (90, 4128, 200, 7, 3),
                                                (100, 2048, 96, 8, 4), (300, 6400, 64, 9, 8), (130, 1600, 260, 10, 4),
                                                (140, 1088, 400, 11, 3), (64, 1600, 528, 12, 2)])
@pytest.mark.parametrize("epi,o_dt", [(kernels.EPI_NONE, "bfloat16"), (kernels.EPI_NONE, "float32"),
                                      (kernels.EPI_GELU, "bfloat16"), (kernels.EPI_RESIDUAL, "float32")])
def test_linear_mfma_split_along_the_inner_size(n, k, o, shape, parts, epi, o_dt):
    """Several workgroups per tile, each with a stretch of the inner size (also one that ends inside a step
    and a number of stretches that leaves the last one short), their sums joined by the second kernel."""
    g = torch.Generator().manual_seed(18)
    a, w, bias = rnd(g, n, k, dtype="bfloat16"), rnd(g, o, k, dtype="bfloat16", scale=k ** -0.5), rnd(g, o)
    prev = rnd(g, n + 2, o, dtype=o_dt)
    out = prev.clone().to(DEV)
    if shape is None:      # what the library chooses by itself: a split, 32 x 32 tiles, four steps in flight
        assert kernels.linear_mfma_partials(n, o, k, epi) > 0
        parts = kernels.linear_mfma_partials(n, o, k, epi) // (n * o)
    scratch = torch.full((parts * n * o + 8,), float("nan"), device=DEV)
    if shape is None:
        parts = None
    assert kernels.linear_mfma(a.to(DEV), w.to(DEV), bias.to(DEV), out, n, epi, shape=shape, k_parts=parts,
                               partials=scratch)
    helpers.assert_close(out[:n], _linear_want(a, w, bias, epi, prev[:n]), "bfloat16", f"split {parts} of {k}")
    assert torch.equal(out[n:], prev[n:].to(DEV)), "rows beyond n_rows were written"
    # twice the same: the sums are joined in a fixed order
    out2 = prev.clone().to(DEV)
    assert kernels.linear_mfma(a.to(DEV), w.to(DEV), bias.to(DEV), out2, n, epi, shape=shape, k_parts=parts,
                               partials=scratch)
    assert torch.equal(out, out2)
    # a buffer that is too small is refused when the split is forced, and not used when it is not
    if shape is not None:
        assert not kernels.linear_mfma(a.to(DEV), w.to(DEV), bias.to(DEV), out2, n, epi, shape=shape, k_parts=parts,
                                       partials=scratch[:16])


def test_linear_mfma_splits_by_itself_when_tiles_are_few_and_the_inner_size_long():
    g = torch.Generator().manual_seed(19)
    n, k, o = 140, 6416, 1600
    need = kernels.linear_mfma_partials(n, o, k, kernels.EPI_RESIDUAL)
    assert need > 0 and need % (n * o) == 0
    assert kernels.linear_mfma_partials(2048, 2048, 512, kernels.EPI_GELU) == 0
    # (an inner size of whole steps under 128 rows and more is not split even with the buffer there: it goes
    # straight into LDS, four steps deep; test_linear_mfma_chooses_the_variants_straight_into_lds)
    a, w, bias = rnd(g, n, k, dtype="bfloat16"), rnd(g, o, k, dtype="bfloat16", scale=k ** -0.5), rnd(g, o)
    prev = rnd(g, n, o)
    out, out1 = prev.clone().to(DEV), prev.clone().to(DEV)
    assert kernels.linear_mfma(a.to(DEV), w.to(DEV), bias.to(DEV), out, n, kernels.EPI_RESIDUAL,
                               partials=torch.empty(need, device=DEV))
    assert kernels.linear_mfma(a.to(DEV), w.to(DEV), bias.to(DEV), out1, n, kernels.EPI_RESIDUAL)   # unsplit
    want = _linear_want(a, w, bias, kernels.EPI_RESIDUAL, prev)
    helpers.assert_close(out, want, "bfloat16", "split by itself")
    helpers.assert_close(out1, want, "bfloat16", "unsplit")
    assert not torch.equal(out, out1)      # another order of summation: it did split


def test_linear_mfma_chooses_the_largest_tiles_for_a_large_problem():
    """160 tiles of 256 x 256: the library takes that shape by itself, so the result equals the forced one bit by bit."""
    g = torch.Generator().manual_seed(17)
    n, k, o = 4096, 320, 2560
    a, w, bias = rnd(g, n, k, dtype="bfloat16"), rnd(g, o, k, dtype="bfloat16", scale=k ** -0.5), rnd(g, o)
    out, out_w = (torch.empty(n, o, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    assert kernels.linear_mfma(a.to(DEV), w.to(DEV), bias.to(DEV), out, n, kernels.EPI_GELU)
    assert kernels.linear_mfma(a.to(DEV), w.to(DEV), bias.to(DEV), out_w, n, kernels.EPI_GELU, shape=0)
    assert torch.equal(out, out_w)
    helpers.assert_close(out, _linear_want(a, w, bias, kernels.EPI_GELU, None), "bfloat16", "large")


@pytest.mark.parametrize("general", [False, True])
@pytest.mark.parametrize("n,k,o,ln_bias,gather", [(8, 512, 1536, True, False), (3, 96, 503, False, True),
                                                  (40, 80, 257, True, True), (64, 2048, 64, False, False), (64, 512, 2048, True, False), (33, 768, 96, True, True),
                                                  (17, 1600, 48, True, False), (16, 1600, 130, True, True),
                                                  (1, 160, 48, False, False), (5, 768, 2050, True, True),
                                                  (2, 1024, 272, True, True), (4, 1600, 144, False, True), (7, 512, 80, True, True),
                                                  (1, 1600, 4800, True, True), (8, 2048, 96, True, True)])
def test_linear_skinny_through_a_folded_layer_norm(n, k, o, ln_bias, gather, general):
    g = torch.Generator().manual_seed(4)
    x = rnd(g, 70, k, scale=2.0) + 0.5
    x[:, 3] += 40.0                      # an outlier channel, as residual streams have
    lw, lb = 1 + 0.1 * rnd(g, k), rnd(g, k) if ln_bias else None
    w, bias = rnd(g, o, k, dtype="bfloat16", scale=k ** -0.5), rnd(g, o)
    rows = torch.randperm(70, generator=g)[:n].tolist() if gather else list(range(n))
    wf, colsum, bias_f = kernels.fold_layer_norm(w.to(DEV), lw.to(DEV), lb.to(DEV) if ln_bias else None, bias.to(DEV))
    # the fold itself: W' = W * gain, S = row sums of W', b' = b + W beta
    helpers.assert_close(wf, w.double() * lw.double(), "bfloat16", "folded matrix")
    helpers.assert_close(colsum, wf.double().sum(1), "float32", "column sums")
    helpers.assert_close(bias_f, bias.double() + (w.double() @ lb.double() if ln_bias else 0), "float32", "folded bias")
    out = torch.empty(n, o, dtype=torch.float32, device=DEV)
    assert kernels.linear_skinny(None, wf, bias_f, out, n, kernels.EPI_NONE, ln_x=x.to(DEV), ln_colsum=colsum,
                                 ln_eps=1e-5, ln_rows=i32(rows) if gather else None, general_only=general)
    if not general and k % 32 == 0:
        out_p = torch.empty_like(out)
        assert kernels.linear_skinny(None, wf, bias_f, out_p, n, kernels.EPI_NONE, ln_x=x.to(DEV), ln_colsum=colsum,
                                     ln_eps=1e-5, ln_rows=i32(rows) if gather else None,
                                     w_packed=kernels.pack_weight(wf))
        assert torch.equal(out_p, out), "the packed matrix gives another result"
    h = P.plain_layer_norm(x.double()[rows], lw.double(), lb.double() if ln_bias else None, 1e-5)
    helpers.assert_close(out, P.plain_linear(h, w.double(), bias.double()), "bfloat16", "LN + skinny")
    if not general and k % 32 == 0:
        for mode in (kernels.ROWS_SHARE_W, kernels.ROWS_GROUPS):
            out_m = torch.full((n + 1, o), float("nan"), dtype=torch.float32, device=DEV)
            assert kernels.linear_skinny(None, wf, bias_f, out_m, n, kernels.EPI_NONE, ln_x=x.to(DEV),
                                         ln_colsum=colsum, ln_eps=1e-5, ln_rows=i32(rows) if gather else None,
                                         rows_mode=mode)
            helpers.assert_close(out_m[:n], P.plain_linear(h, w.double(), bias.double()), "bfloat16",
                                 f"LN + skinny, rows mode {mode}")
            assert torch.isnan(out_m[n:]).all(), "rows beyond n_rows were written"
        for rpg in (16, 8, 4, 2, 1):
            out_g = torch.full((n + 1, o), float("nan"), dtype=torch.float32, device=DEV)
            assert kernels.linear_skinny(None, wf, bias_f, out_g, n, kernels.EPI_NONE, ln_x=x.to(DEV),
                                         ln_colsum=colsum, ln_eps=1e-5, ln_rows=i32(rows) if gather else None,
                                         rows_mode=kernels.ROWS_GROUPS, rows_per_group=rpg)
            # the rows' statistics are summed in an order that follows the rows of a workgroup,
            # so the results agree to rounding, not bit by bit
            helpers.assert_close(out_g[:n], P.plain_linear(h, w.double(), bias.double()), "bfloat16",
                                 f"LN + skinny, {rpg} rows to a workgroup")
            assert torch.isnan(out_g[n:]).all(), "rows beyond n_rows were written"


@pytest.mark.parametrize("general", [False, True])
@pytest.mark.parametrize("outlier", [None, 0, 7])
def test_folded_layer_norm_of_rows_far_from_zero(general, outlier):
    """Rows whose values lie 50 standard deviations from zero (and one channel further out still, also
    the first one): what the product rounds to bfloat16 must be the distance from a value of the
    row, not the value, or the rounding error of the offset drowns the row."""
    g = torch.Generator().manual_seed(40)
    n, k, o = 6, 256, 96
    x = rnd(g, n, k, scale=1.0) + torch.tensor([100.0, -100.0, 50.0, 0.0, 300.0, -75.0])[:, None]
    if outlier is not None:
        x[:, outlier] += 400.0
    lw, lb = 1 + 0.1 * rnd(g, k), rnd(g, k)
    w, bias = rnd(g, o, k, dtype="bfloat16", scale=k ** -0.5), rnd(g, o)
    wf, colsum, bias_f = kernels.fold_layer_norm(w.to(DEV), lw.to(DEV), lb.to(DEV), bias.to(DEV))
    out = torch.empty(n, o, dtype=torch.float32, device=DEV)
    assert kernels.linear_skinny(None, wf, bias_f, out, n, kernels.EPI_NONE, ln_x=x.to(DEV), ln_colsum=colsum,
                                 ln_eps=1e-5, general_only=general)
    h = P.plain_layer_norm(x.double(), lw.double(), lb.double(), 1e-5)
    helpers.assert_close(out, P.plain_linear(h, w.double(), bias.double()), "bfloat16", "LN of rows far from zero")


@pytest.mark.parametrize("general,n,rows_mode,rpg", [(False, 6, 0, 0), (True, 6, 0, 0), (True, 40, 0, 0),
                                                     (False, 40, kernels.ROWS_SHARE_W, 0),
                                                     (False, 40, kernels.ROWS_GROUPS, 0), (False, 64, kernels.ROWS_GROUPS, 0),
                                                     (False, 6, kernels.ROWS_GROUPS, 4), (False, 13, kernels.ROWS_GROUPS, 8),
                                                     (False, 40, kernels.ROWS_GROUPS, 4), (False, 16, 0, 0), (False, 7, kernels.ROWS_GROUPS, 1),
                                                     (False, 9, kernels.ROWS_GROUPS, 2)])
def test_linear_skinny_stores_keys_and_values(general, n, rows_mode, rpg):
    g = torch.Generator().manual_seed(5)
    k, h, hk, d, page, pages = 64, 4, 2, 16, 4, 23
    qw, kvw = h * d, hk * d
    a, w, bias = rnd(g, n, k, dtype="bfloat16"), rnd(g, qw + 2 * kvw, k, dtype="bfloat16", scale=0.2), rnd(g, qw + 2 * kvw)
    kp = torch.full((pages, hk, page, d), float("nan"), dtype=torch.bfloat16, device=DEV)
    vp = kp.clone()
    slots = [4 * 8 + 3, 0, 7, -1, 4 * 2 + 1, 4 * 8 + 0]
    if n > 6:   # distinct slots all over the pool, a padded token now and then
        slots = torch.randperm(pages * page, generator=g)[:n].tolist()
        slots = [-1 if t % 9 == 4 else s for t, s in enumerate(slots)]
    out = torch.empty(n, qw + 2 * kvw, dtype=torch.bfloat16, device=DEV)
    assert kernels.linear_skinny(a.to(DEV), w.to(DEV), bias.to(DEV), out, n, kernels.SK_EPI_QKV,
                                 scatter=(kp, vp, i32(slots), qw, kvw), general_only=general, rows_mode=rows_mode,
                                 rows_per_group=rpg)
    want = P.plain_linear(a.double(), w.double(), bias.double())
    helpers.assert_close(out, want, "bfloat16", "qkv")
    written = torch.zeros(pages * page, dtype=torch.bool)
    for t, slot in enumerate(slots):
        if slot < 0:
            continue
        written[slot] = True
        for head in range(hk):
            helpers.assert_close(kp[slot // page, head, slot % page], want[t, qw + head * d:qw + (head + 1) * d],
                                 "bfloat16", "stored key")
            helpers.assert_close(vp[slot // page, head, slot % page],
                                 want[t, qw + kvw + head * d:qw + kvw + (head + 1) * d], "bfloat16", "stored value")
    untouched = kp.float().cpu().permute(0, 2, 1, 3).reshape(pages * page, -1)[~written]
    assert torch.isnan(untouched).all(), "a slot that no token owns was written"


@pytest.mark.parametrize("n,k,o", [(64, 2048, 512), (40, 1024, 256), (17, 2048, 48), (33, 3072, 768), (24, 3072, 768)])
@pytest.mark.parametrize("epi,o_dt", [(kernels.EPI_NONE, "bfloat16"), (kernels.EPI_NONE, "float32"),
                                      (kernels.EPI_GELU, "bfloat16"), (kernels.EPI_RESIDUAL, "float32")])
def test_linear_skinny_with_the_inner_size_split_over_workgroups(n, k, o, epi, o_dt):
    """With scratch for the parts, a long inner size under more than 16 rows whose rows stay in one
    workgroup per column tile runs as two launches; the result is the unsplit kernel's up to the order
    of four sums.  Left to choose, the launcher splits only what it does not deal out in groups of
    16 rows (a small matrix with an inner size up to 2048)."""
    g = torch.Generator().manual_seed(16)
    need = 4 * n * o
    groups = kernels.linear_skinny_row_groups(n, o, k)
    assert groups == (o * k * 2 <= 6 << 20 if k <= 2048 else n > 32 and o * k * 2 <= 8 << 20)
    assert kernels.linear_skinny_partials(n, o, k, False, epi) == (0 if groups else need)
    # up to 16 rows: split only from an inner size of 3072 on
    assert kernels.linear_skinny_partials(16, o, k, False, epi) == (4 * 16 * o if k >= 3072 else 0)
    assert kernels.linear_skinny_partials(n, o, 512, False, epi) == 0         # a short inner size
    assert kernels.linear_skinny_partials(n, o, k, True, epi) == 0            # not through a folded LayerNorm
    a, w, bias = rnd(g, n + 2, k, dtype="bfloat16"), rnd(g, o, k, dtype="bfloat16", scale=k ** -0.5), rnd(g, o)
    prev = rnd(g, n + 2, o, dtype=o_dt)
    partials = torch.full((need,), float("nan"), device=DEV)
    for b in (bias, None):
        out = prev.clone().to(DEV)
        assert kernels.linear_skinny(a.to(DEV), w.to(DEV), None if b is None else b.to(DEV), out, n, epi,
                                     partials=partials, rows_mode=kernels.ROWS_SHARE_W)
        assert not torch.isnan(partials[:need]).any(), "the parts were not written: no split happened"
        partials.fill_(float("nan"))
        helpers.assert_close(out[:n], _linear_want(a, w, b, epi, prev)[:n], "bfloat16", f"split {n}x{k}x{o}")
        assert torch.equal(out[n:], prev[n:].to(DEV)), "rows beyond n_rows were written"
    # too little scratch: the unsplit kernel, same result
    out2 = prev.clone().to(DEV)
    assert kernels.linear_skinny(a.to(DEV), w.to(DEV), bias.to(DEV), out2, n, epi, partials=partials[:need // 2],
                                 rows_mode=kernels.ROWS_SHARE_W)
    assert torch.isnan(partials).all(), "too little scratch was written to"
    helpers.assert_close(out2[:n], _linear_want(a, w, bias, epi, prev)[:n], "bfloat16", "unsplit")


@pytest.mark.parametrize("n,k,o", [(1, 3072, 768), (8, 6400, 1600), (16, 3072, 48), (3, 4096, 512)])
@pytest.mark.parametrize("epi,o_dt", [(kernels.EPI_NONE, "bfloat16"), (kernels.EPI_GELU, "bfloat16"),
                                      (kernels.EPI_RESIDUAL, "float32")])
def test_linear_skinny_few_rows_with_a_long_inner_size_split_over_workgroups(n, k, o, epi, o_dt):
    """Up to 16 rows under an inner size of 3072 and more and few column tiles: four workgroups per
    tile take a quarter of the inner size each when the caller brings scratch, one takes it all
    without; both against the plain product."""
    g = torch.Generator().manual_seed(61)
    need = kernels.linear_skinny_partials(n, o, k, False, epi)
    assert need == 4 * n * o
    assert kernels.linear_skinny_partials(n, o, 2048, False, epi) == 0       # not worth a second kernel
    assert kernels.linear_skinny_partials(n, 2048, k, False, epi) == 0       # column tiles enough
    a, w, bias = rnd(g, n + 1, k, dtype="bfloat16"), rnd(g, o, k, dtype="bfloat16", scale=k ** -0.5), rnd(g, o)
    prev = rnd(g, n + 1, o, dtype=o_dt)
    want = _linear_want(a, w, bias, epi, prev)
    partials = torch.full((need,), float("nan"), device=DEV)
    packed = kernels.pack_weight(w.to(DEV))
    for wp in (None, packed):
        out = prev.clone().to(DEV)
        assert kernels.linear_skinny(a.to(DEV), w.to(DEV), bias.to(DEV), out, n, epi, partials=partials, w_packed=wp)
        assert not torch.isnan(partials).any(), "the parts were not written: no split happened"
        partials.fill_(float("nan"))
        helpers.assert_close(out[:n], want[:n], "bfloat16", f"few rows split {n}x{k}x{o}")
        assert torch.equal(out[n:], prev[n:].to(DEV)), "rows beyond n_rows were written"
    whole = prev.clone().to(DEV)
    assert kernels.linear_skinny(a.to(DEV), w.to(DEV), bias.to(DEV), whole, n, epi)
    helpers.assert_close(whole[:n], want[:n], "bfloat16", "unsplit")


@pytest.mark.parametrize("n,shape,k", [(70, None, 96), (300, 3, 96), (1100, 2, 96), (300, 1, 96), (520, 0, 96),
                                       (40, None, 832), (60, 6, 96), (33, 5, 1024), (200, 8, 256), (300, 9, 128),
                                       (520, 10, 192), (1100, 11, 64), (60, 12, 832)])
def test_linear_mfma_stores_keys_and_values(n, shape, k):
    """The tiled kernel's fused QKV product: the tile shape chosen by the size and each larger one forced
    (at 40 rows over 13 steps the library takes the variant with four steps in flight by itself);
    groups of heads; padded rows (slot -1) leave the pools alone."""
    g = torch.Generator().manual_seed(15)
    h, hk, d, page = 6, 2, 16, 8
    pages = n // page + 3
    qw, kvw = h * d, hk * d
    a, w, bias = rnd(g, n, k, dtype="bfloat16"), rnd(g, qw + 2 * kvw, k, dtype="bfloat16", scale=0.2), rnd(g, qw + 2 * kvw)
    kp = torch.full((pages, hk, page, d), float("nan"), dtype=torch.bfloat16, device=DEV)
    vp = kp.clone()
    slots = torch.randperm(pages * page, generator=g)[:n].tolist()
    for t in range(0, n, 7):
        slots[t] = -1
    out = torch.empty(n, qw + 2 * kvw, dtype=torch.bfloat16, device=DEV)
    assert kernels.linear_mfma(a.to(DEV), w.to(DEV), bias.to(DEV), out, n, kernels.EPI_NONE,
                               scatter=(kp, vp, i32(slots), qw, kvw), shape=shape)
    want = P.plain_linear(a.double(), w.double(), bias.double())
    helpers.assert_close(out, want, "bfloat16", "qkv")
    kflat = kp.float().cpu().permute(0, 2, 1, 3).reshape(pages * page, kvw)
    vflat = vp.float().cpu().permute(0, 2, 1, 3).reshape(pages * page, kvw)
    live = torch.tensor([s for s in slots if s >= 0])
    rows = torch.tensor([t for t, s in enumerate(slots) if s >= 0])
    helpers.assert_close(kflat[live], want[rows, qw:qw + kvw], "bfloat16", "stored keys")
    helpers.assert_close(vflat[live], want[rows, qw + kvw:], "bfloat16", "stored values")
    untouched = torch.ones(pages * page, dtype=torch.bool)
    untouched[live] = False
    assert torch.isnan(kflat[untouched]).all() and torch.isnan(vflat[untouched]).all()


@pytest.mark.parametrize("n,k,o,parts", [(1, 64, 16, 1), (15, 192, 257, 1), (16, 320, 40, 1), (17, 256, 48, 1), (31, 576, 33, 1),
                                         (32, 1600, 130, 1), (32, 1344, 66, 1), (3, 2048, 100, 2), (16, 2112, 100, 4), (32, 5440, 36, 4),
                                         (20, 832, 64, 3)])
@pytest.mark.parametrize("epi,o_dt", [(kernels.EPI_NONE, "bfloat16"), (kernels.EPI_NONE, "float32"), (kernels.EPI_GELU, "bfloat16"),
                                      (kernels.EPI_RELU2, "bfloat16"), (kernels.EPI_RESIDUAL, "float32")])
@pytest.mark.parametrize("shape", [26, 27])
def test_linear_mfma_of_a_few_rows(n, k, o, parts, epi, o_dt, shape):
    """The kernel whose waves take steps of their own, with 16 and 32 columns a workgroup: steps for one wave alone and for some of
    them only, more and fewer than the stages; ragged rows and columns; stretches of the inner size, the last one shorter."""
    g = torch.Generator().manual_seed(n + k)
    a, w, bias = rnd(g, n, k, dtype="bfloat16"), rnd(g, o, k, dtype="bfloat16", scale=k ** -0.5), rnd(g, o)
    prev = rnd(g, n + 2, o, dtype=o_dt)
    out = prev.clone().to(DEV)
    scratch = torch.full((parts * n * o,), float("nan"), device=DEV)
    assert kernels.linear_mfma(a.to(DEV), w.to(DEV), bias.to(DEV), out, n, epi, shape=shape, k_parts=parts, partials=scratch)
    helpers.assert_close(out[:n], _linear_want(a, w, bias, epi, prev[:n]), "bfloat16", f"shape {shape} {n}x{k}x{o}")
    assert torch.equal(out[n:], prev[n:].to(DEV)), "rows beyond n_rows were written"
    many = torch.zeros(33, k, dtype=torch.bfloat16, device=DEV)
    assert not kernels.linear_mfma(many, w.to(DEV), None, torch.zeros(33, o, dtype=TDT[o_dt], device=DEV), 33, epi, shape=shape)
    short = torch.zeros(o, 48, dtype=torch.bfloat16, device=DEV)
    assert not kernels.linear_mfma(many[:, :48].contiguous(), short, None, out, n, epi, shape=shape)


@pytest.mark.parametrize("n,shape", [(2, 26), (16, 27), (17, 26), (32, 27)])
def test_linear_mfma_of_a_few_rows_stores_keys_and_values(n, shape):
    test_linear_mfma_stores_keys_and_values(n, shape, 320)


@pytest.mark.parametrize("n,k,o,rows,split", [
    (1, 1600, 4800, True, 1), (32, 1600, 4800, True, 1), (33, 1600, 4800, False, None), (4, 768, 2304, True, 1), (8, 704, 2304, True, 1),
    (7, 704, 2304, False, None), (8, 768, 1920, False, None), (8, 1024, 3072, False, None), (8, 1024, 4096, True, 1),
    (3, 1600, 7184, False, None), (4, 1600, 7184, True, 1), (8, 1600, 8208, False, None), (8, 4096, 752, False, None),
    (1, 6400, 1600, True, 2), (32, 6400, 1600, True, 4), (8, 5440, 2048, True, 1), (16, 5440, 2048, True, 2), (32, 5440, 2048, True, 4),
    (16, 8192, 2048, True, 1), (32, 8192, 2048, True, 4), (18, 2688, 1024, True, 1), (19, 2688, 1024, True, 4), (16, 1616, 1616, False, None)])
def test_which_products_of_a_few_rows_have_a_kernel_of_their_own(n, k, o, rows, split):
    """On both sides of the lines; where it is taken, its float32 sums are no further from 64 bits than the decode kernel's and the 32 x 32
    tiles', also where operands that are not aligned leave it to others."""
    from types import SimpleNamespace

    from mini_gpt_inference_amd.ops import linear as L
    from mini_gpt_inference_amd.parts.base import Workspace

    g = torch.Generator().manual_seed(k + n)
    a, w = rnd(g, n, k, dtype="bfloat16").to(DEV), rnd(g, o, k, dtype="bfloat16", scale=k ** -0.5).to(DEV)
    plan = kernels.linear_rows_plan(n, o, k)
    assert (plan is not None) == rows
    if not rows:
        return
    assert plan[1] == split and kernels.linear_rows_plan(n, o, k, True)[1] == 1
    want = a.double() @ w.double().T
    error = lambda t: ((t.double() - want).norm() / want.norm()).item()
    ctx = SimpleNamespace(exact=False, dtype=torch.bfloat16, n_rows=n, pending=None, copy_budget=None, workspace=Workspace(torch.device(DEV)))
    got, decode, tiles, odd = (torch.zeros(n, o, device=DEV) for _ in range(4))
    L.linear_add(ctx, a, w, None, got, n, may_leave_parts=True)
    assert (ctx.pending is not None) == (split > 1)
    if split > 1:
        assert kernels.residual_settle(ctx.pending, got, n)
        ctx.pending, added = None, torch.zeros_like(got)
        L.linear_add(ctx, a, w, None, added, n)
        helpers.assert_close(added, got.double().cpu(), "float32", "added up at once")
    assert kernels.linear_skinny(a, w, None, decode, n, kernels.EPI_RESIDUAL)
    assert kernels.linear_mfma(a, w, None, tiles, n, kernels.EPI_RESIDUAL, shape=4)
    assert error(got) <= 1.01 * min(error(decode), error(tiles)), (error(got), error(decode), error(tiles))
    unaligned = torch.zeros(n * k + 1, dtype=torch.bfloat16, device=DEV)[1:].view(n, k)
    unaligned.copy_(a)
    L.linear_add(ctx, unaligned, w, None, odd, n)
    helpers.assert_close(odd, want, "bfloat16", "operands that are not aligned")


@pytest.mark.parametrize("n,k,o", [(16, 768, 2304), (17, 768, 2304), (5, 1600, 4800), (6, 1600, 4800), (10, 1280, 3840), (11, 1280, 3840)])
def test_layer_norm_in_front_of_a_product_of_a_few_rows(n, k, o):
    """On both sides of the lines between the LayerNorm folded into the decode kernel and one of its own."""
    from types import SimpleNamespace

    from mini_gpt_inference_amd.ops import linear as L
    from mini_gpt_inference_amd.parts.base import Workspace

    g = torch.Generator().manual_seed(n + k)
    x, w, bias = rnd(g, n, k, scale=2.0).to(DEV), rnd(g, o, k, dtype="bfloat16", scale=k ** -0.5).to(DEV), rnd(g, o).to(DEV)
    gain, shift = 1.0 + rnd(g, k, scale=0.1).to(DEV), rnd(g, k, scale=0.1).to(DEV)
    assert kernels.linear_rows_plan(n, o, k) and L.folds_before_rows_apart(n, o, k) == (n in (16, 5, 10))
    want = _linear_want(P.plain_layer_norm(x.double().cpu(), gain.double().cpu(), shift.double().cpu(), 1e-5), w.cpu(), bias.cpu(), kernels.EPI_GELU, None)
    ctx = SimpleNamespace(exact=False, dtype=torch.bfloat16, n_rows=n, pending=None, copy_budget=None, workspace=Workspace(torch.device(DEV)))
    out = torch.empty(n, o, dtype=torch.bfloat16, device=DEV)
    norm = SimpleNamespace(weight=gain, bias=shift, eps=1e-5, fusable_layer_norm=True,
                           forward=lambda ctx, x, h, n, rows=None: kernels.layer_norm(x, gain, shift, h, n, 1e-5, rows))
    L.linear(ctx, L.LazyNorm(norm, x, n), w, bias, out, n, kernels.EPI_GELU)
    helpers.assert_close(out, want, "bfloat16", "LayerNorm and product")


def test_linear_skinny_refuses_what_it_cannot_do():
    w = torch.zeros(32, 64, dtype=torch.bfloat16, device=DEV)
    a = torch.zeros(65, 64, dtype=torch.bfloat16, device=DEV)
    assert not kernels.linear_skinny(a, w, None, torch.zeros(65, 32, dtype=torch.bfloat16, device=DEV), 65)
    assert not kernels.linear_skinny(a.float(), w, None, torch.zeros(65, 32, dtype=torch.bfloat16, device=DEV), 4)


# ----------------------------------------------------------------------------- cache write and attention
class PagedCase:
    """Random requests with part of their tokens already cached, laid out in scattered pages."""

    def __init__(self, seq_lens, q_lens, h, hk, d, page, dtype, seed=0, poison=True, spikes=()):
        """spikes: (request, query index within the step, key position, head): that query and that key
        are made long and parallel, so that this one score stands out among hundreds and the query's
        output is that key's value; a kernel that misses the key, or takes another for it, shows."""
        g = torch.Generator().manual_seed(seed)
        self.h, self.hk, self.d, self.page = h, hk, d, page
        self.seq_lens, self.q_lens = seq_lens, q_lens
        n_pages = sum(-(-s // page) for s in seq_lens) + 3
        order = torch.randperm(n_pages, generator=g).tolist()
        self.k = [rnd(g, s, hk, d, dtype=dtype) for s in seq_lens]
        self.v = [rnd(g, s, hk, d, dtype=dtype) for s in seq_lens]
        self.q = [rnd(g, ql, h, d, dtype=dtype) for ql in q_lens]
        for r, qi, key, head in spikes:
            assert key <= seq_lens[r] - q_lens[r] + qi, "a query sees no later key"
            u = torch.randn(d, generator=g)
            u = (3.0 * math.sqrt(d) * u / u.norm()).to(TDT[dtype])      # |u|^2 = 9 d: the score is 9 d * scale
            self.q[r][qi, head] = u
            self.k[r][key, head // (h // hk)] = u
        fill = float("nan") if poison else 0.0
        kp = torch.full((n_pages, hk, page, d), fill, dtype=TDT[dtype])
        vp = kp.clone()
        mb = max(-(-s // page) for s in seq_lens) + 1
        bt = torch.full((len(seq_lens), mb), -1, dtype=torch.int32)
        self.slots = []
        for r, s in enumerate(seq_lens):
            for b in range(-(-s // page)):
                bt[r, b] = order.pop()
            for t in range(s):
                pg, off = bt[r, t // page].item(), t % page
                kp[pg, :, off] = self.k[r][t]
                vp[pg, :, off] = self.v[r][t]
            self.slots += [bt[r, t // page].item() * page + t % page for t in range(s - q_lens[r], s)]
        self.kp, self.vp, self.bt = kp.to(DEV), vp.to(DEV), bt.to(DEV)
        self.n = sum(q_lens)
        self.cu = i32(np.concatenate([[0], np.cumsum(q_lens)]))
        self.sl = i32(seq_lens)
        self.q_req = i32([r for r, ql in enumerate(q_lens) for _ in range(ql)])
        self.q_flat = torch.cat([q.reshape(-1, h * d) for q in self.q]).to(DEV)

    def want(self, scale, window):
        outs = []
        for r, (s, ql) in enumerate(zip(self.seq_lens, self.q_lens)):
            # the plain attention over the whole sequence; the step's queries are its last q_len rows
            qfull = torch.zeros(self.h, s, self.d, dtype=P.DT)
            qfull[:, s - ql:] = self.q[r].double().transpose(0, 1)
            o = P.plain_causal_attention(qfull, self.k[r].double().transpose(0, 1),
                                         self.v[r].double().transpose(0, 1), scale=scale, window=window)
            outs.append(o[s - ql:])
        return torch.cat(outs)


ATTENTION_CASES = [
    # the reference's own cases (tests/test_triton.py:83-154): uniform, ragged around a page, one key
    dict(seq_lens=[16] * 4, q_lens=[1] * 4, h=4, hk=4, d=64, page=8),
    dict(seq_lens=[3, 8, 9, 17, 24], q_lens=[1] * 5, h=4, hk=4, d=64, page=8),
    dict(seq_lens=[1, 1], q_lens=[1, 1], h=2, hk=2, d=64, page=8),
    # other sizes: groups, head sizes in steps of 16, portions, pages of other sizes, long contexts
    dict(seq_lens=[40, 7, 130], q_lens=[5, 7, 2], h=6, hk=2, d=48, page=4),
    dict(seq_lens=[300, 65], q_lens=[1, 33], h=3, hk=1, d=16, page=16),
    dict(seq_lens=[77, 200], q_lens=[77, 1], h=2, hk=2, d=128, page=32),
    dict(seq_lens=[129], q_lens=[64], h=5, hk=5, d=80, page=16),
    dict(seq_lens=[333, 70, 200], q_lens=[333, 3, 130], h=4, hk=2, d=32, page=16),
    dict(seq_lens=[500], q_lens=[190], h=2, hk=1, d=96, page=8),
]


@pytest.mark.parametrize("window", [0, 90])
@pytest.mark.parametrize("d,h,hk", [(64, 12, 12), (64, 4, 1), (128, 8, 2)])
@pytest.mark.parametrize("seq_lens,q_lens", [([40, 513, 700], [1, 1, 130]), ([1, 64], [1, 63]), ([300] * 20 + [65, 1, 900], [1] * 20 + [65, 1, 640]),
                                             ([9] * 3 + [70] * 70, [1] * 3 + [66] * 70), ([500, 1000], [1, 1000])])
def test_single_tokens_and_portions_in_one_launch(seq_lens, q_lens, d, h, hk, window):
    """The launch that has a step's single tokens beside its prompt portions: both kinds against the plain attention, as the
    step's own requests (the leading ones are the single tokens) and as a padded step (which requests bring one token is
    read from cu_q, the last single token of the portions' part among them; requests and tokens of the padding are left
    alone), around a tile, few tiles and many, and with more requests than a wave numbers at a time."""
    c = PagedCase(seq_lens, q_lens, h=h, hk=hk, d=d, page=16, dtype="bfloat16", seed=d + len(q_lens))
    n, r = c.n, len(q_lens)
    lead = next(i for i, q in enumerate(q_lens) if q != 1)
    scale, want = d ** -0.5, c.want(d ** -0.5, window)
    positions = i32([s - q + t for s, q in zip(seq_lens, q_lens) for t in range(q)])
    out = torch.full((n, h * d), float("nan"), dtype=torch.bfloat16, device=DEV)
    args = (c.q_flat, out, c.kp, c.vp, c.bt, positions, c.q_req, c.cu, c.sl)
    took = lead * h <= 256
    assert kernels.mixed_attention_bf16(*args, lead, True, lead, r - lead, n - lead, 0, h, scale, window) == took
    if took:
        helpers.assert_close(out, want, "bfloat16", "the step's own requests")
    cap, rows = 16, n + 5
    pad = lambda t, size, fill: torch.cat([t, torch.full((size - t.shape[0], *t.shape[1:]), fill, dtype=t.dtype, device=DEV)])
    padded = torch.full((rows, h * d), 7.0, dtype=torch.bfloat16, device=DEV)
    took = kernels.mixed_attention_bf16(
        pad(c.q_flat, rows, 0.0), padded, c.kp, c.vp, pad(c.bt, r + 4, -1), pad(positions, rows, 0), pad(c.q_req, rows, -1),
        pad(c.cu, r + 5, n), pad(c.sl, r + 4, 0), min(cap, rows), False, 0, r + 4, rows, min(cap, rows), h, scale, window)
    assert took == (min(cap, rows) * h <= 256)
    if took:
        helpers.assert_close(padded[:n], want, "bfloat16", "a padded step")
        assert (padded[n:] == 7.0).all()


@pytest.mark.parametrize("portion", [97, 200])
def test_single_tokens_that_may_see_many_keys_beside_a_portion(portion):
    """Contexts of more than 1,024 keys and more workgroups than compute units: tiles of 64 queries in eight waves."""
    test_single_tokens_and_portions_in_one_launch([1100, 40] * 6 + [portion + 60], [1] * 12 + [portion], 64, 16, 16, 0)


MIXED_OPTIONS = {
    "sinks": (0, ["sinks"], {}), "cap": (0, [], {"softcap": 15.0}), "gate": (0, ["gate"], {}),
    "kept first keys": (90, [], {"keep_first": 70}), "sigmoid weights": (0, ["score_bias"], {}),
    "chunks": (96, [], {"chunked": True}), "sinks, cap and gate in a window": (90, ["sinks", "gate"], {"softcap": 15.0}),
    "sigmoid weights, gate and kept first keys": (90, ["score_bias", "gate"], {"keep_first": 5}),
    "sinks in chunks": (96, ["sinks"], {"chunked": True})}


@pytest.mark.parametrize("option", sorted(MIXED_OPTIONS))
@pytest.mark.parametrize("d,h,hk", [(64, 12, 12), (64, 4, 1), (128, 8, 2)])
@pytest.mark.parametrize("seq_lens,q_lens", [([40, 513, 700], [1, 1, 130]), ([300] * 20 + [65, 1, 900], [1] * 20 + [65, 1, 640])])
def test_single_tokens_and_portions_in_one_launch_with_every_option(seq_lens, q_lens, d, h, hk, option):
    """Each option that the launch passes on, for both kinds of tokens, as the step's own requests and as a padded step,
    against the general kernel in 32 bits on the same numbers."""
    window, tensors, mask = MIXED_OPTIONS[option]
    mask = dict(mask)
    c = PagedCase(seq_lens, q_lens, h=h, hk=hk, d=d, page=16, dtype="bfloat16", seed=d + len(q_lens))
    n, r = c.n, len(q_lens)
    lead = next(i for i, q in enumerate(q_lens) if q != 1)
    g = torch.Generator().manual_seed(d + h)
    gate = torch.randn(n, h, generator=g).to(DEV, torch.bfloat16) if "gate" in tensors else None
    for name in ("sinks", "score_bias"):
        if name in tensors:
            mask[name] = (torch.randn(h, generator=g) - (3.0 if name == "score_bias" else 0.0)).to(DEV)
    scale, positions = d ** -0.5, i32([s - q + t for s, q in zip(seq_lens, q_lens) for t in range(q)])
    want = torch.empty(n, h * d, device=DEV)
    kernels.paged_attention_generic(c.q_flat.float(), want, c.kp.float(), c.vp.float(), c.bt, c.cu, c.sl, c.q_req, n, r, h, scale,
                                    window, gate=None if gate is None else gate.float(), **mask)
    out = torch.full((n, h * d), float("nan"), dtype=torch.bfloat16, device=DEV)
    took = kernels.mixed_attention_bf16(c.q_flat, out, c.kp, c.vp, c.bt, positions, c.q_req, c.cu, c.sl, lead, True, lead,
                                        r - lead, n - lead, 0, h, scale, window, gate=gate, **mask)
    assert took == (lead * h <= 256)
    if took:
        helpers.assert_close(out, want, "bfloat16", "the step's own requests")
    rows, cap = n + 5, 16
    pad = lambda t, size, fill: torch.cat([t, torch.full((size - t.shape[0], *t.shape[1:]), fill, dtype=t.dtype, device=DEV)])
    padded = torch.full((rows, h * d), 7.0, dtype=torch.bfloat16, device=DEV)
    assert kernels.mixed_attention_bf16(
        pad(c.q_flat, rows, 0.0), padded, c.kp, c.vp, pad(c.bt, r + 4, -1), pad(positions, rows, 0), pad(c.q_req, rows, -1),
        pad(c.cu, r + 5, n), pad(c.sl, r + 4, 0), cap, False, 0, r + 4, rows, cap, h, scale, window,
        gate=None if gate is None else pad(gate, rows, 0.0), **mask)
    helpers.assert_close(padded[:n], want, "bfloat16", "a padded step")
    assert (padded[n:] == 7.0).all()


@pytest.mark.parametrize("d,h,hk,portion,keys,window", [(128, 4, 1, 30, 1204, 0), (128, 4, 1, 30, 1204, 1203),
                                                        (128, 4, 1, 30, 1204, 1204), (128, 4, 1, 30, 1204, 1250),
                                                        (128, 4, 1, 700, 4096, 0), (64, 12, 1, 2048, 16384, 0),
                                                        (128, 4, 1, 30, 1114, 0), (128, 4, 1, 30, 1114, 1113),
                                                        (128, 4, 1, 30, 1114, 1114), (128, 4, 1, 30, 1114, 1160),
                                                        (128, 4, 1, 700, 2560, 0)])
def test_single_tokens_behind_long_contexts_beside_a_portion(d, h, hk, portion, keys, window):
    """Where a token's workgroup has four waves, tokens that see more than so many keys have a second launch of their own:
    every token is done by one of the two, around that number, as the step's own requests and as a padded step, also with a
    window that keeps some of them or all below it."""
    seq_lens = [keys - 1, keys, keys + 1, 40, keys + 300, portion + 50]
    q_lens = [1] * 5 + [portion]
    c = PagedCase(seq_lens, q_lens, h=h, hk=hk, d=d, page=16, dtype="bfloat16", seed=portion)
    n, r, lead, scale = c.n, len(q_lens), 5, d ** -0.5
    positions = i32([s - q + t for s, q in zip(seq_lens, q_lens) for t in range(q)])
    for mask in ({}, {"keep_first": 10} if window else {"softcap": 20.0}):
        want = torch.empty(n, h * d, device=DEV)
        kernels.paged_attention_generic(c.q_flat.float(), want, c.kp.float(), c.vp.float(), c.bt, c.cu, c.sl, c.q_req, n, r, h,
                                        scale, window, **mask)
        out = torch.full((n, h * d), float("nan"), dtype=torch.bfloat16, device=DEV)
        assert kernels.mixed_attention_bf16(c.q_flat, out, c.kp, c.vp, c.bt, positions, c.q_req, c.cu, c.sl, lead, True, lead, 1,
                                            portion, 0, h, scale, window, **mask)
        helpers.assert_close(out, want, "bfloat16", "the step's own requests")
        padded = torch.full((n, h * d), float("nan"), dtype=torch.bfloat16, device=DEV)
        assert kernels.mixed_attention_bf16(c.q_flat, padded, c.kp, c.vp, c.bt, positions, c.q_req, c.cu, c.sl, 8, False, 0, r,
                                            n, 8, h, scale, window, **mask)
        helpers.assert_close(padded, want, "bfloat16", "a padded step")


@pytest.mark.parametrize("short", ["queries", "output"])
def test_single_tokens_and_portions_refuse_buffers_that_end_before_their_tokens(short):
    """The portions' tokens lie behind the single ones: their numbers add up.  Nothing is launched."""
    c = PagedCase([40, 50, 70], [1, 1, 70], h=4, hk=4, d=64, page=16, dtype="bfloat16", seed=3)
    out = torch.full((c.n, 4 * 64), 7.0, dtype=torch.bfloat16, device=DEV)
    q, o = (c.q_flat[:c.n - 1], out) if short == "queries" else (c.q_flat, out[:c.n - 1])
    with pytest.raises(kernels.KernelError, match="too small"):
        kernels.mixed_attention_bf16(q, o, c.kp, c.vp, c.bt, i32([39, 49] + list(range(70))), c.q_req, c.cu, c.sl, 2, True, 2, 1,
                                     70, 0, 4, 0.125)
    assert (out == 7.0).all()


@pytest.mark.parametrize("window", [0, 100])
@pytest.mark.parametrize("d,n", [(16, 129), (32, 129), (64, 128), (64, 129), (128, 64), (128, 65)])
def test_decode_attention_of_many_tokens(d, n, window):
    """More (token, head) pairs than the chip holds workgroups of eight waves: four a head, whose pass is 256 keys, for
    tokens behind few keys: around the line between the two, contexts around a chunk and around one and two passes."""
    lens = ([1, 63, 64, 65, 255, 256, 257, 511, 512, 513, 40] * 12)[:n]
    c = PagedCase(lens, [1] * n, h=4, hk=2, d=d, page=16, dtype="bfloat16", seed=d + n)
    out = torch.full((n, 4 * d), float("nan"), dtype=torch.bfloat16, device=DEV)
    assert kernels.paged_attention_decode_bf16(c.q_flat, out, c.kp, c.vp, c.bt, i32([x - 1 for x in lens]), c.q_req, n, 4,
                                               d ** -0.5, window, identity=True)
    helpers.assert_close(out, c.want(d ** -0.5, window), "bfloat16", "decode attention")


@pytest.mark.parametrize("window,mask", [(0, {}), (0, {"softcap": 15.0}), (300, {"keep_first": 3}), (300, {"chunked": True}),
                                         (600, {}), (256, {}), (250, {"keep_first": 7})])
@pytest.mark.parametrize("d,h,hk,n", [(16, 5, 1, 110), (32, 5, 5, 110), (64, 5, 1, 110), (64, 4, 2, 130), (128, 7, 7, 40),
                                      (128, 4, 1, 70)])
def test_decode_attention_of_many_tokens_short_ones_beside_long_ones(d, h, hk, n, window, mask):
    """Where a block table or window leaves room for long contexts, a token behind up to 256 keys (512 with heads of 128) has
    two heads in one workgroup, four waves each, and a token behind more a workgroup a head; so has an odd number's last
    head.  As requests' own tokens, and as a step in which some tokens are padding and some are another kernel's."""
    lens = ([1, 255, 256, 257, 40, 511, 512, 513, 700, 64, 1100, 3] * 11)[:n]
    c = PagedCase(lens, [1] * n, h=h, hk=hk, d=d, page=16, dtype="bfloat16", seed=d + n)
    want = torch.empty(n, h * d, device=DEV)
    kernels.paged_attention_generic(c.q_flat.float(), want, c.kp.float(), c.vp.float(), c.bt, c.cu, c.sl, c.q_req, n, n, h,
                                    d ** -0.5, window, **mask)
    out = torch.full((n, h * d), float("nan"), dtype=torch.bfloat16, device=DEV)
    positions = i32([x - 1 for x in lens])
    assert kernels.paged_attention_decode_bf16(c.q_flat, out, c.kp, c.vp, c.bt, positions, c.q_req, n, h, d ** -0.5, window,
                                               identity=True, **mask)
    helpers.assert_close(out, want, "bfloat16", "decode attention")
    q_req, cu = c.q_req.clone(), c.cu.clone()
    left = torch.zeros(n, dtype=torch.bool)
    left[[2, 3, 10, 11]] = True
    q_req[[2, 10]] = -1
    q_req[11] = q_req[12]                              # these two are one request's, as cu_q has it
    counts = torch.ones(n, dtype=torch.int32)
    counts[[3, 12]] = 2
    left[12] = True
    cu = i32(np.concatenate([[0], np.cumsum(counts.numpy())]))
    out = torch.full((n, h * d), 7.0, dtype=torch.bfloat16, device=DEV)
    assert kernels.paged_attention_decode_bf16(c.q_flat, out, c.kp, c.vp, c.bt, positions, q_req, n, h, d ** -0.5, window,
                                               cu_q=cu, **mask)
    assert (out[left.to(DEV)] == 7.0).all()
    helpers.assert_close(out[~left.to(DEV)], want[~left.to(DEV)], "bfloat16", "beside padding and portions")


@pytest.mark.parametrize("window,mask", [(0, {}), (100, {}), (100, {"keep_first": 70}), (96, {"chunked": True})])
@pytest.mark.parametrize("d", [16, 32, 64, 128])
def test_float32_attention_keeps_its_sums_whatever_the_portion(d, window, mask):
    """The matrix-core kernel of the 32-bit path has tiles of 16 queries and chunks of 64 keys dealt out over 8 waves (512
    keys a round): a query's output is the same bits as part of a whole prompt, of a portion and alone, around the ends of
    all of these, and with more requests than the 64 that a wave numbers the tiles of at a time."""
    lens = [1, 15, 16, 17, 63, 64, 65, 511, 512, 513, 600]
    c = PagedCase(lens, lens, h=4, hk=2, d=d, page=12, dtype="float32", seed=d)
    g = torch.Generator().manual_seed(d + 1)
    extra = {"sinks": torch.randn(4, generator=g).to(DEV), "softcap": 0.0 if mask else 20.0,
             "gate": torch.randn(c.n, 4, generator=g).to(DEV)}

    def attend(req, first, q_lens, rows):
        out = torch.full((len(rows), 4 * d), float("nan"), device=DEV)
        cu = i32(np.concatenate([[0], np.cumsum(q_lens)]))
        kernels.paged_attention_generic(
            c.q_flat[rows].contiguous(), out, c.kp, c.vp, c.bt[req].contiguous(), cu,
            i32([f + q for f, q in zip(first, q_lens)]), i32([i for i, q in enumerate(q_lens) for _ in range(q)]), len(rows),
            len(req), 4, d ** -0.5, window, **{**extra, "gate": extra["gate"][rows].contiguous()}, **mask)
        return out

    starts = np.concatenate([[0], np.cumsum(lens)])
    whole = attend(list(range(len(lens))), [0] * len(lens), lens, list(range(c.n)))
    if not mask:
        want = c.want(d ** -0.5, window)               # without sink, cap and gate
        plain = torch.empty_like(whole)
        kernels.paged_attention_generic(c.q_flat, plain, c.kp, c.vp, c.bt, c.cu, c.sl, c.q_req, c.n, len(lens), 4, d ** -0.5,
                                        window)
        helpers.assert_close(plain, want, "float32", "matrix-core attention")
    # every request's tokens from a third of it on, in one portion, with others before and behind it
    cut = [n // 3 for n in lens]
    rows = [starts[r] + t for r, n in enumerate(lens) for t in range(cut[r], n)]
    assert torch.equal(attend(list(range(len(lens))), cut, [n - x for n, x in zip(lens, cut)], rows), whole[rows])
    # single tokens, eighty requests' worth of them
    pick = [(r, t) for r, n in enumerate(lens) for t in sorted({0, n // 2, max(n - 2, 0), n - 1, min(64, n - 1)})]
    pick = (pick * 3)[:80]
    rows = [starts[r] + t for r, t in pick]
    assert torch.equal(attend([r for r, _ in pick], [t for _, t in pick], [1] * len(pick), rows), whole[rows])


@pytest.mark.parametrize("window,mask", [(0, {}), (100, {}), (100, {"keep_first": 70}), (96, {"chunked": True}), (0, {"dist_bias": 9}),
                                         (0, {"slopes": True})])
@pytest.mark.parametrize("page", [12, 16, 32])
@pytest.mark.parametrize("d", [16, 32, 64, 128])
def test_float32_attention_of_single_tokens_has_the_same_bits(d, page, window, mask):
    """The kernel for a step of single tokens against the one for any step: around the ends of groups (16), chunks (64) and
    rounds of eight waves (512), with padding, sinks, cap and gate, and with infinite and NaN values among the seen ones."""
    lens = [1, 2, 15, 16, 17, 63, 64, 65, 200, 511, 512, 513, 650]
    n = len(lens)
    c = PagedCase(lens, [1] * n, h=4, hk=2, d=d, page=page, dtype="float32", seed=d + page)
    g = torch.Generator().manual_seed(d)
    mask = dict(mask)
    if "dist_bias" in mask:
        mask["dist_bias"] = torch.randn(4, mask["dist_bias"], generator=g).to(DEV)
    if "slopes" in mask:
        mask["slopes"] = torch.rand(4, generator=g).to(DEV)
    extra = {"sinks": torch.randn(4, generator=g).to(DEV), "softcap": 20.0 if not mask else 0.0,
             "gate": torch.randn(n, 4, generator=g).to(DEV)}
    q_req = c.q_req.clone()
    q_req[[3, 9]] = -1

    def attend(single, **kw):
        out = torch.full((n, 4 * d), 7.0, device=DEV)
        kernels.paged_attention_generic(c.q_flat, out, c.kp, c.vp, c.bt, c.cu, c.sl, q_req, n, n, 4, d ** -0.5, window,
                                        single=single, **kw, **mask)
        return out

    for kw in ({}, extra):
        want = attend(False, **kw)
        assert torch.isfinite(want).all() and (want[[3, 9]] == 7.0).all()
        assert torch.equal(attend(True, **kw), want)
    for i, (r, s) in enumerate(zip(range(n), lens)):
        j = max(s - 1 - 5 * i, 0)
        c.vp[int(c.bt[r, j // page]), i % 2, j % page, i % d] = (float("inf"), float("nan"), float("-inf"))[i % 3]
    want = attend(False)
    assert not torch.isfinite(want).all()
    assert torch.equal(attend(True).nan_to_num(1e30, 2e30, 3e30), want.nan_to_num(1e30, 2e30, 3e30))


@pytest.mark.parametrize("window,mask", [(0, {}), (20, {}), (20, {"keep_first": 9}), (24, {"chunked": True})])
@pytest.mark.parametrize("d", [16, 32, 48, 64, 128])
def test_float32_attention_keeps_what_a_query_does_not_see_out_of_it(d, window, mask):
    """A value that is infinite or NaN reaches the queries that see its key, in its channel, and nobody else: every other
    output is the same bits as without it, also of the queries that share a tile with one that sees it.  (48: the general
    kernel; the others: the matrix-core kernel, prompts, portions and single tokens.)"""
    seq_lens, q_lens = [40, 65, 130, 7, 90, 150], [40, 65, 130, 7, 33, 1]
    c = PagedCase(seq_lens, q_lens, h=4, hk=2, d=d, page=12, dtype="float32", seed=d)

    def attend():
        out = torch.full((c.n, 4 * d), 7.0, device=DEV)
        kernels.paged_attention_generic(c.q_flat, out, c.kp, c.vp, c.bt, c.cu, c.sl, c.q_req, c.n, len(q_lens), 4, d ** -0.5,
                                        window, **mask)
        return out.view(c.n, 4, d)

    want = attend()
    assert torch.isfinite(want).all()
    unusual = []                                       # request, key, head of keys, channel, value
    for r, s in enumerate(seq_lens):
        for i, j in enumerate(sorted({s - 1, s - 2, s // 2, s // 2 + 1, 4})):
            unusual.append((r, j, i % 2, (5 * i + r) % d, (float("inf"), float("nan"), float("-inf"))[i % 3]))
    for r, j, hk, ch, value in unusual:
        c.vp[int(c.bt[r, j // 12]), hk, j % 12, ch] = value
    starts = c.cu.tolist()
    for r, j, hk, ch, value in unusual:
        for t in range(q_lens[r]):
            p = seq_lens[r] - q_lens[r] + t
            first = 0 if not window else (p - p % window if mask.get("chunked") else p - window + 1)
            if j <= p and (j >= first or j < mask.get("keep_first", 0)):
                want[starts[r] + t, 2 * hk:2 * hk + 2, ch] = value
    assert torch.equal(attend().nan_to_num(1e30, 2e30, 3e30), want.nan_to_num(1e30, 2e30, 3e30))


@pytest.mark.parametrize("d", [16, 48, 64, 128])
def test_float32_attention_leaves_other_tokens_alone(d):
    """Rows at or beyond n_tokens, which cu_q may still count, tokens without a request and a step without requests: the
    kernel on the matrix cores as the general one (48)."""
    seq_lens, q_lens = [20, 40, 9, 70], [20, 3, 9, 33]
    c = PagedCase(seq_lens, q_lens, h=4, hk=2, d=d, page=12, dtype="float32", seed=d)
    q_req = c.q_req.clone()
    q_req[[5, 19, 24]] = -1

    def attend(n, r, q_req):
        out = torch.full((c.n, 4 * d), 7.0, device=DEV)
        kernels.paged_attention_generic(c.q_flat, out, c.kp, c.vp, c.bt, c.cu, c.sl, q_req, n, r, 4, d ** -0.5)
        return out

    whole = attend(c.n, len(q_lens), c.q_req)
    assert not (whole == 7.0).all(1).any()
    for n in (c.n, c.n - 1, 49, 48, 33, 32, 24, 21, 20, 17, 16, 3):
        want = whole.clone()
        want[n:] = 7.0
        want[[5, 19, 24]] = 7.0
        assert torch.equal(attend(n, len(q_lens), q_req), want), n
    assert (attend(c.n, 0, torch.full_like(q_req, -1)) == 7.0).all()


@pytest.mark.parametrize("window", [0, 5, 70])
@pytest.mark.parametrize("case", range(len(ATTENTION_CASES)))
@pytest.mark.parametrize("kernel", ["generic-float32", "generic-bfloat16", "split-bfloat16", "splitfast-bfloat16",
                                    "prefill-bfloat16"])
def test_paged_attention(kernel, case, window):
    name, dtype = kernel.split("-")
    c = PagedCase(**ATTENTION_CASES[case], dtype=dtype, seed=case)
    scale = 0.37 if case % 2 else 1.0 / math.sqrt(c.d)
    out = torch.full((c.n, c.h * c.d), float("nan"), dtype=TDT[dtype], device=DEV)
    args = (c.q_flat, out, c.kp, c.vp, c.bt, c.cu, c.sl, c.q_req, c.n, len(c.seq_lens), c.h, scale, window)
    if name == "generic":
        kernels.paged_attention_generic(*args, fast_exp=dtype == "bfloat16")
    elif name == "prefill":
        if c.d not in (32, 64, 96, 128):
            pytest.skip("the MFMA tile kernel takes head sizes 32, 64, 96, 128")
        assert kernels.prefill_attention_bf16(c.q_flat, out, c.kp, c.vp, c.bt, c.cu, c.sl, len(c.seq_lens),
                                              max(c.q_lens), c.h, scale, window)
    else:
        if name == "splitfast" and c.d not in (16, 32, 64, 128):
            pytest.skip("the wide-load variant takes head sizes 16, 32, 64, 128")
        assert kernels.paged_attention_split_bf16(*args, fast=name == "splitfast")
    helpers.assert_close(out, c.want(scale, window), dtype, f"{kernel} case {case} window {window}")


@pytest.mark.parametrize("window", [0, 33, 290])
@pytest.mark.parametrize("q_lens,before,h", [([129, 1, 0], 415, 4),            # eight waves that share the keys of 32 queries
                                             ([1, 31, 32, 33, 64, 65, 127], 60, 4),    # four
                                             ([1, 31, 32, 33, 64, 65, 129] * 5, 200, 4)])   # two waves of queries, two that share
@pytest.mark.parametrize("d", [32, 64, 96, 128])
def test_prefill_attention_forms_at_the_edges_of_their_tiles(d, q_lens, before, h, window):
    """Tiles of 32 and 64 queries with their last queries missing, stretches of keys that end part way, waves without a query or
    without a key that one of their queries sees; pages beyond a request's tokens hold NaN."""
    lens = [q + (before + 37 * i) % 450 for i, q in enumerate(q_lens)]
    c = PagedCase(seq_lens=lens, q_lens=q_lens, h=h, hk=2, d=d, page=16, dtype="bfloat16", seed=d + window)
    out = torch.full((c.n, c.h * c.d), float("nan"), dtype=torch.bfloat16, device=DEV)
    assert kernels.prefill_attention_bf16(c.q_flat, out, c.kp, c.vp, c.bt, c.cu, c.sl, len(lens), max(c.q_lens), c.h, d ** -0.5, window)
    helpers.assert_close(out, c.want(d ** -0.5, window), "bfloat16", f"head size {d}, window {window}")


@pytest.mark.parametrize("window,mask", [(0, {}), (1650, {"keep_first": 50}), (900, {"chunked": True})])
@pytest.mark.parametrize("r,q_len,d,h,page", [(1, 70, 64, 2, 2), (1, 130, 128, 2, 1), (5, 70, 32, 16, 2), (6, 65, 64, 30, 2)])
def test_prefill_attention_behind_more_pages_than_lie_in_lds(r, q_len, d, h, page, window, mask):
    """A tile keeps 768 entries of the block table at a time: contexts of more pages than that, also behind a window that keeps the
    first keys, in each form of the kernel, against the general kernel in 32 bits on the same numbers."""
    lens = [2100 - 90 * i for i in range(r)]
    c = PagedCase(lens, [q_len] * r, h=h, hk=2, d=d, page=page, dtype="bfloat16", seed=d + window, poison=False)
    want = torch.empty(c.n, h * d, device=DEV)
    kernels.paged_attention_generic(c.q_flat.float(), want, c.kp.float(), c.vp.float(), c.bt, c.cu, c.sl, c.q_req, c.n, r, h, d ** -0.5,
                                    window, **mask)
    out = torch.full((c.n, h * d), float("nan"), dtype=torch.bfloat16, device=DEV)
    assert kernels.prefill_attention_bf16(c.q_flat, out, c.kp, c.vp, c.bt, c.cu, c.sl, r, q_len, h, d ** -0.5, window, **mask)
    helpers.assert_close(out, want, "bfloat16", f"{r} requests, window {window}")


@pytest.mark.parametrize("cap", [0.0, 12.0])
@pytest.mark.parametrize("q_lens,before", [([140, 1, 30], 300), ([1, 31, 32, 33, 65, 100] * 4, 60), ([65, 40, 129] * 10, 150)])
@pytest.mark.parametrize("d", [32, 64, 128])
def test_prefill_attention_with_slopes_in_each_form(d, q_lens, before, cap):
    """Slopes by distance, behind a cap and without one, with eight, four and two times two waves, against the general kernel in 32
    bits on the same numbers."""
    lens = [q + (before + 37 * i) % 450 for i, q in enumerate(q_lens)]
    c = PagedCase(lens, q_lens, h=4, hk=2, d=d, page=16, dtype="bfloat16", seed=d, poison=False)
    slopes = torch.tensor([0.5, 0.06, 0.004, 0.0], device=DEV)
    want = torch.empty(c.n, 4 * d, device=DEV)
    kernels.paged_attention_generic(c.q_flat.float(), want, c.kp.float(), c.vp.float(), c.bt, c.cu, c.sl, c.q_req, c.n, len(lens), 4,
                                    d ** -0.5, softcap=cap, slopes=slopes)
    out = torch.full((c.n, 4 * d), float("nan"), dtype=torch.bfloat16, device=DEV)
    assert kernels.prefill_attention_bf16(c.q_flat, out, c.kp, c.vp, c.bt, c.cu, c.sl, len(lens), max(q_lens), 4, d ** -0.5,
                                          softcap=cap, slopes=slopes)
    helpers.assert_close(out, want, "bfloat16", f"head size {d}, cap {cap}")


@pytest.mark.parametrize("r,h,longest", [(1, 1, 1), (1, 1, 300), (1, 3, 700), (1, 7, 256), (1, 8, 33), (3, 3, 290), (1, 15, 520), (2, 12, 64),
                                         (5, 5, 545)])
def test_prefill_attention_deals_every_tile_out_once(r, h, longest):
    """Heads that are no multiple of the eight dies, with fewer tiles than eight, whole eights of them and some over."""
    q_lens = [max(longest - 97 * i, 0) for i in range(r)]
    c = PagedCase([q + 5 * i for i, q in enumerate(q_lens)], q_lens, h=h, hk=1, d=64, page=16, dtype="bfloat16", seed=longest)
    out = torch.full((c.n, h * 64), float("nan"), dtype=torch.bfloat16, device=DEV)
    assert kernels.prefill_attention_bf16(c.q_flat, out, c.kp, c.vp, c.bt, c.cu, c.sl, r, longest, h, 0.125)
    helpers.assert_close(out, c.want(0.125, 0), "bfloat16", f"{r} requests x {h} heads")


def test_prefill_attention_of_more_heads_than_a_grid_is_wide():
    """129 requests x 65,535 heads, a token each behind two others."""
    r, h, d = 129, 65535, 32
    g = torch.Generator(device=DEV).manual_seed(3)
    q = torch.randn(r, h * d, generator=g, device=DEV, dtype=torch.bfloat16)
    kp, vp = (torch.randn(r, 1, 4, d, generator=g, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    out = torch.full((r, h * d), float("nan"), dtype=torch.bfloat16, device=DEV)
    bt = torch.arange(r, dtype=torch.int32, device=DEV).view(r, 1)
    cu, sl = torch.arange(r + 1, dtype=torch.int32, device=DEV), torch.full((r,), 3, dtype=torch.int32, device=DEV)
    assert kernels.prefill_attention_bf16(q, out, kp, vp, bt, cu, sl, r, 1, h, d ** -0.5)
    for i in (0, 1, 63, 127, 128):
        scores = q[i].float().view(h, d) @ kp[i, 0, :3].float().T * d ** -0.5
        helpers.assert_close(out[i].view(h, d), torch.softmax(scores, 1) @ vp[i, 0, :3].float(), "bfloat16", f"request {i}")
    assert torch.isfinite(out).all()


@pytest.mark.parametrize("window", [0, 33])
@pytest.mark.parametrize("d", [32, 64])
def test_prefill_attention_with_many_tiles(d, window):
    """More than 320 query tiles in the step: the tile kernel then takes 64 queries a workgroup, in two wave groups that
    split the keys, instead of 32 in four or eight."""
    lens = [130 + 7 * i for i in range(11)]
    c = PagedCase(seq_lens=lens, q_lens=[70 + (i % 3) for i in range(11)], h=16, hk=4, d=d, page=16,
                  dtype="bfloat16", seed=d)
    assert 11 * 2 * 16 > 320
    out = torch.full((c.n, c.h * c.d), float("nan"), dtype=torch.bfloat16, device=DEV)
    scale = 1.0 / math.sqrt(d)
    assert kernels.prefill_attention_bf16(c.q_flat, out, c.kp, c.vp, c.bt, c.cu, c.sl, len(lens), max(c.q_lens),
                                          c.h, scale, window)
    helpers.assert_close(out, c.want(scale, window), "bfloat16", f"many tiles, head size {d}")


LONG_PREFILL_CASES = {
    # the benchmarked prefill step: two whole prompts of 1,024 tokens, 8 heads of 64 (256 query tiles:
    # two wave groups split every 256 keys), and the same with more than 320 tiles (one wave group)
    "2x1024-d64": dict(seq_lens=[1024, 1024], q_lens=[1024, 1024], h=8, hk=8, d=64, page=16),
    "3x1024-d64": dict(seq_lens=[1024, 1000, 1024], q_lens=[1024, 1000, 1024], h=8, hk=8, d=64, page=16),
    "1x1024-d128": dict(seq_lens=[1024], q_lens=[1024], h=4, hk=4, d=128, page=16),
    "6x1024-d128": dict(seq_lens=[1024] * 6, q_lens=[1024] * 6, h=4, hk=2, d=128, page=32),
    # portions of 64 to 512 tokens over 512 and 900 cached keys, few tiles and many
    "portions-d64": dict(seq_lens=[576, 1024, 1024, 964], q_lens=[64, 124, 512, 64], h=8, hk=8, d=64, page=16),
    "portions-d64-many": dict(seq_lens=[576, 1024, 1024, 964], q_lens=[64, 124, 512, 64], h=32, hk=8, d=64, page=16),
    "portions-d128": dict(seq_lens=[1024, 612, 1000], q_lens=[512, 100, 100], h=4, hk=4, d=128, page=8),
    "portions-d128-many": dict(seq_lens=[1024, 612, 1000], q_lens=[512, 100, 100], h=32, hk=4, d=128, page=8),
}


@pytest.mark.parametrize("name", sorted(LONG_PREFILL_CASES))
def test_prefill_attention_at_the_benchmarked_lengths(name):
    """The MFMA tile kernel with whole prompts of 1,024 tokens and with portions over 512 and 900
    cached keys, head sizes 64 and 128, in both of its modes (two wave groups that split every 256
    keys while the step has at most 320 query tiles, one wave group beyond), pages scattered over a
    NaN-poisoned pool.  Random scores alone are nearly flat over so many keys: in every request a
    few queries get one key that stands out (the first key, one a few blocks back, the last key of a
    128-key block, the query's own), and the query's output must be that key's value."""
    spec = LONG_PREFILL_CASES[name]
    tiles = sum(-(-q // 64) for q in spec["q_lens"]) * spec["h"]
    assert (tiles > 320) == (name.startswith(("3x", "6x")) or name.endswith("many")), tiles
    spikes = []
    for r, (s, ql) in enumerate(zip(spec["seq_lens"], spec["q_lens"])):
        first = s - ql
        for j, (qi, key) in enumerate([(ql - 1, 0), (ql - 1 - 7, max(first + ql - 8 - 300, 1)), (ql // 2, 127),
                                       (ql // 3, first + ql // 3), (1, first + 1), (ql - 2, 383)]):
            if key <= first + qi:
                spikes.append((r, qi, key, (r + j) % spec["h"]))
    assert len({(r, key) for r, _, key, _ in spikes}) == len({(r, qi) for r, qi, _, _ in spikes}) == len(spikes)
    c = PagedCase(**spec, dtype="bfloat16", seed=len(name), spikes=spikes)
    scale = 1.0 / math.sqrt(c.d)
    out = torch.full((c.n, c.h * c.d), float("nan"), dtype=torch.bfloat16, device=DEV)
    assert kernels.prefill_attention_bf16(c.q_flat, out, c.kp, c.vp, c.bt, c.cu, c.sl, len(c.seq_lens),
                                          max(c.q_lens), c.h, scale, 0)
    want = c.want(scale, 0)
    helpers.assert_close(out, want, "bfloat16", name)
    # the spiked queries really are decided by one key (so the comparison above pins the lookup)
    offs = np.concatenate([[0], np.cumsum(c.q_lens)])
    for r, qi, key, head in spikes:
        row = want[offs[r] + qi, head * c.d:(head + 1) * c.d]
        helpers.assert_close(row, c.v[r][key, head // (c.h // c.hk)].double(), "bfloat16", f"{name}: spike {r, qi, key}")


@pytest.mark.parametrize("window", [0, 20])
def test_single_tokens_and_portions_told_apart_on_the_device(window):
    """What a padded graph of a step with prompt portions launches: the decode kernel over the first 16
    tokens, leaving out those of requests with several tokens; the tile kernel over all requests
    (padded to 8, the padding bringing no tokens), leaving out the single tokens among the first 16.
    Together they write every token's row once: single tokens before and after the 16th, portions
    that start before it."""
    q_lens = [1, 1, 1, 9, 1, 1, 30]            # tokens 0, 1, 2 | 3..11 | 12 | 13 | 14..43: token 13 < 16 <= 14 + 30
    seq_lens = [50, 1, 77, 40, 200, 18, 64]
    c = PagedCase(seq_lens=seq_lens, q_lens=q_lens, h=4, hk=2, d=64, page=16, dtype="bfloat16", seed=3)
    scale = 0.125
    r_cap, n_cap = 8, 48
    cu = torch.full((r_cap + 1,), c.n, dtype=torch.int32)
    cu[:len(q_lens) + 1] = c.cu.cpu()
    sl = torch.zeros(r_cap, dtype=torch.int32)
    sl[:len(q_lens)] = c.sl.cpu()
    bt = torch.full((r_cap, c.bt.shape[1]), -1, dtype=torch.int32)
    bt[:len(q_lens)] = c.bt.cpu()
    q_req = torch.full((n_cap,), -1, dtype=torch.int32)
    q_req[:c.n] = c.q_req.cpu()
    pos = torch.zeros(n_cap, dtype=torch.int32)
    pos[:c.n] = torch.tensor([s - ql + j for s, ql in zip(seq_lens, q_lens) for j in range(ql)], dtype=torch.int32)
    qp = torch.zeros(n_cap, c.q_flat.shape[1], dtype=torch.bfloat16, device=DEV)
    qp[:c.n] = c.q_flat
    out = torch.full((n_cap, c.h * c.d), float("nan"), dtype=torch.bfloat16, device=DEV)
    cu, sl, bt, q_req, pos = (t.to(DEV) for t in (cu, sl, bt, q_req, pos))
    assert kernels.paged_attention_decode_bf16(qp, out, c.kp, c.vp, bt, pos, q_req, 16, c.h, scale, window, cu_q=cu)
    singles = [0, 1, 2, 12, 13]
    others = [t for t in range(c.n) if t not in singles]
    assert torch.isnan(out[others].float()).all(), "the decode kernel wrote a portion's token"
    assert not torch.isnan(out[singles].float()).any()
    assert kernels.prefill_attention_bf16(qp, out, c.kp, c.vp, bt, cu, sl, r_cap, n_cap, c.h, scale, window,
                                          single_below=16)
    helpers.assert_close(out[:c.n], c.want(scale, window), "bfloat16", "single tokens and portions together")
    assert torch.isnan(out[c.n:].float()).all(), "a padded row was written"


DECODE_CASES = [
    dict(seq_lens=[600, 1, 64, 65, 513, 300], q_lens=[1] * 6, h=4, hk=2, d=64, page=16),
    dict(seq_lens=[130, 1030, 7], q_lens=[1] * 3, h=3, hk=3, d=128, page=32),
    dict(seq_lens=[257, 31, 512, 511], q_lens=[1] * 4, h=6, hk=2, d=32, page=8),
    dict(seq_lens=[90, 700], q_lens=[1] * 2, h=2, hk=1, d=16, page=4),
    dict(seq_lens=[100, 550, 13], q_lens=[1] * 3, h=2, hk=2, d=64, page=12),   # a page size that is no power of two
]


@pytest.mark.parametrize("window", [0, 5, 70])
@pytest.mark.parametrize("case", range(len(ATTENTION_CASES) + len(DECODE_CASES)))
def test_paged_attention_decode(case, window):
    """The decode step's kernel: by position and block table row, for any token; with identity=True
    where every request brings one token.  Unused block table entries hold numbers far outside the
    pool, and a padded token leaves its output row alone."""
    spec = (ATTENTION_CASES + DECODE_CASES)[case]
    if spec["d"] not in (16, 32, 64, 128):
        pytest.skip("head sizes 16, 32, 64, 128")
    c = PagedCase(**spec, dtype="bfloat16", seed=case)
    scale = 0.37 if case % 2 else 1.0 / math.sqrt(c.d)
    bt = c.bt.clone()
    bt[bt < 0] = 10 ** 6
    positions = i32([p for s, ql in zip(c.seq_lens, c.q_lens) for p in range(s - ql, s)] + [0])
    q_req = torch.cat([c.q_req, i32([-1])])
    q = torch.cat([c.q_flat, c.q_flat[:1]])
    want = c.want(scale, window)
    modes = [False, True] if all(ql == 1 for ql in c.q_lens) else [False]
    for identity in modes:
        out = torch.full((c.n + 1, c.h * c.d), 7.0, dtype=torch.bfloat16, device=DEV)
        if identity:   # the padded token's row of the block table exists, as in a padded step
            bt_i = torch.cat([bt, torch.full_like(bt[:1], 10 ** 6)])
        else:
            bt_i = bt
        took = kernels.paged_attention_decode_bf16(q, out, c.kp, c.vp, bt_i, positions, q_req, c.n + 1, c.h, scale,
                                                   window, identity=identity)
        if c.page & (c.page - 1):
            assert not took, "page sizes that are no power of two go to the general kernels"
            return
        assert took
        helpers.assert_close(out[:c.n], want, "bfloat16", f"decode case {case} window {window} identity {identity}")
        assert (out[c.n] == 7.0).all(), "a padded token's row was written"


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_kv_write_and_padding(dtype):
    g = torch.Generator().manual_seed(7)
    n, hk, d, page, pages = 5, 3, 16, 4, 6
    qkv = rnd(g, n, 7 + 2 * hk * d, dtype=dtype).to(DEV)
    kp = torch.full((pages, hk, page, d), float("nan"), dtype=TDT[dtype], device=DEV)
    vp = kp.clone()
    slots = [9, 0, -1, 23, 10]
    kernels.kv_write(qkv, 7, 7 + hk * d, kp, vp, i32(slots), n)
    for t, s in enumerate(slots):
        if s < 0:
            continue
        assert torch.equal(kp[s // page, :, s % page].reshape(-1), qkv[t, 7:7 + hk * d])
        assert torch.equal(vp[s // page, :, s % page].reshape(-1), qkv[t, 7 + hk * d:])
    assert torch.isnan(kp.float()).sum().item() == (pages * page - 4) * hk * d
    # a padded token (q_req = -1) is skipped by attention: its output row is left alone
    c = PagedCase(seq_lens=[9], q_lens=[2], h=3, hk=3, d=16, page=4, dtype=dtype)
    out = torch.full((3, 48), 7.0, dtype=TDT[dtype], device=DEV)
    q = torch.cat([c.q_flat, c.q_flat[:1]])
    kernels.paged_attention_generic(q, out, c.kp, c.vp, c.bt, c.cu, c.sl, i32([0, 0, -1]), 3, 1, 3, 0.25, 0)
    assert (out[2] == 7.0).all() and torch.isfinite(out[:2].float()).all()


# ----------------------------------------------------------------------------- sampling
def _sample(logits, temperature, top_k=None, top_p=None, seeds=None, idx=None, engine_seed=0, real_vocab=None):
    m, v = logits.shape
    out = torch.full((m,), -1, dtype=torch.int32, device=DEV)
    kernels.sample(logits.to(DEV), m, real_vocab or v, torch.tensor(temperature, dtype=torch.float32, device=DEV),
                   None if top_k is None else i32(top_k),
                   None if top_p is None else torch.tensor(top_p, dtype=torch.float32, device=DEV),
                   None if seeds is None else torch.tensor(seeds, dtype=torch.int64, device=DEV),
                   None if idx is None else i32(idx), engine_seed, out)
    return out.cpu().tolist()


def test_greedy_is_argmax_with_the_lowest_index_on_ties_and_respects_the_vocabulary_mask():
    g = torch.Generator().manual_seed(8)
    logits = rnd(g, 6, 50304)
    logits[1, 777] = logits[1, 40000] = 50.0
    logits[2, 50300] = 99.0                       # beyond the real vocabulary
    got = _sample(logits, [0.0] * 6, real_vocab=50257)
    want = [P.plain_sample(row.numpy(), 0.0, None, None, 0.0, 50257)[0] for row in logits]
    assert got == want and got[1] == 777 and got[2] < 50257


def test_greedy_ties_at_every_distance_and_rows_that_are_not_aligned():
    """Equal maxima in one vector of four, in one thread's vectors, in different waves; the last id that
    may be chosen; a vocabulary that leaves rows unaligned and a tail of one to three logits."""
    g = torch.Generator().manual_seed(12)
    for rows, vocab, real in ((6, 50304, 50257), (3, 50257, 50257), (7, 9003, 9001), (3, 300, 300)):
        logits = rnd(g, rows, vocab)
        logits[0, real - 5] = logits[0, 11] = 60.0
        logits[1, real - 1] = 70.0
        far = 4096 + 5 if real > 4101 else 200
        logits[-1, 5] = logits[-1, 6] = logits[-1, far] = 65.0
        got = _sample(logits, [0.0] * rows, real_vocab=real)
        want = [P.plain_sample(row.numpy(), 0.0, None, None, 0.0, real)[0] for row in logits]
        assert got == want and got[0] == 11 and got[1] == real - 1 and got[-1] == 5


@pytest.mark.parametrize("rows,n_out,k_dim,limit,packed,bias", [(1, 1008, 96, 1001, True, False), (5, 50304, 512, 50257, True, False),
                                                             (16, 208, 64, 208, False, True), (8, 4096, 1600, 4090, True, True),
                                                             (3, 2000, 768, 1999, False, False)])
def test_head_leaves_the_best_column_of_every_tile_and_greedy_rows_choose_from_them(rows, n_out, k_dim, limit, packed, bias):
    """The logits are those of the plain product; every tile's best is the plain argmax over the
    tile's columns below the limit (the lowest column among equals: two rows of the matrix are the
    same, inside a tile and across tiles); and greedy rows that read the tiles' bests choose what
    they choose from the logits themselves, beside seeded rows that still read the logits."""
    g = torch.Generator().manual_seed(rows * 7 + n_out)
    a = rnd(g, rows, k_dim, dtype="bfloat16")
    w = rnd(g, n_out, k_dim, dtype="bfloat16", scale=0.1)
    w[17] = w[21]                          # equal logits within a tile
    w[n_out - 40] = w[3]                   # and in two tiles far apart
    a[0] = (w[3].float() * 8).bfloat16()   # row 0 points at them: its largest logits are the equal pair
    if rows > 1:
        a[-1] = (w[n_out - 1].float() * 8).bfloat16()   # the last row's largest logit lies past the limit (if limit < n_out)
    b = rnd(g, n_out, scale=0.1) if bias else None
    if bias:
        b[17], b[n_out - 40] = b[21], b[3]
    out = torch.full((rows, n_out), float("nan"), device=DEV)
    tiles = n_out // 16
    bv = torch.full((rows + 2, tiles), float("nan"), device=DEV)
    bi = torch.full((rows + 2, tiles), -3, dtype=torch.int32, device=DEV)
    wd = w.to(DEV)
    assert kernels.linear_head_best(a.to(DEV), wd, None if b is None else b.to(DEV), out, rows, bv, bi, limit,
                                    w_packed=kernels.pack_weight(wd) if packed else None)
    want = _linear_want(a, w, b, kernels.EPI_NONE, None)
    helpers.assert_close(out, want, "bfloat16", "head")
    # the tiles' bests are exact statements about the logits that were stored
    got = out.cpu()
    masked = got.clone()
    masked[:, limit:] = -float("inf")
    per_tile = masked.view(rows, tiles, 16)
    want_val, want_off = per_tile.max(dim=2)
    first = (per_tile == want_val.unsqueeze(2)).int().argmax(dim=2)     # the lowest column among equals
    want_idx = first + 16 * torch.arange(tiles).unsqueeze(0)
    live = torch.isfinite(want_val)       # a tile wholly past the limit holds -inf and no column
    assert torch.equal(bv[:rows].cpu()[live], want_val[live])
    assert torch.equal(bi[:rows].cpu()[live].long(), want_idx[live])
    assert (bv[:rows].cpu()[~live] == -float("inf")).all()
    assert torch.isnan(bv[rows:]).all() and (bi[rows:] == -3).all()
    # choosing from them
    temps = [0.0] * rows
    if rows > 2:
        temps[1] = 0.8
    tk = torch.tensor(temps, device=DEV)
    seeds = torch.arange(rows, dtype=torch.int64, device=DEV)
    idx = torch.zeros(rows, dtype=torch.int32, device=DEV)
    from_logits = torch.full((rows,), -1, dtype=torch.int32, device=DEV)
    from_tiles = torch.full((rows,), -1, dtype=torch.int32, device=DEV)
    kernels.sample(out, rows, limit, tk, None, None, seeds, idx, 5, from_logits)
    kernels.sample(out, rows, limit, tk, None, None, seeds, idx, 5, from_tiles, tile_best=(bv, bi))
    assert torch.equal(from_logits, from_tiles)
    plain = [P.plain_sample(got[r].numpy(), 0.0, None, None, 0.0, limit)[0] for r in range(rows) if temps[r] == 0.0]
    assert [t for t, temp in zip(from_tiles.cpu().tolist(), temps) if temp == 0.0] == plain
    assert from_tiles[0].item() == 3 and from_tiles[-1].item() < limit


def test_head_with_tile_bests_refuses_what_its_kernel_does_not_take():
    g = torch.Generator().manual_seed(4)
    for rows, n_out, k_dim in ((17, 208, 64), (4, 200, 64), (4, 208, 48)):
        a, w = rnd(g, rows, k_dim, dtype="bfloat16").to(DEV), rnd(g, n_out, k_dim, dtype="bfloat16").to(DEV)
        out = torch.zeros(rows, n_out, device=DEV)
        tiles = max(n_out // 16, 1)
        bv, bi = torch.zeros(rows, tiles, device=DEV), torch.zeros(rows, tiles, dtype=torch.int32, device=DEV)
        assert not kernels.linear_head_best(a, w, None, out, rows, bv, bi, n_out)
        assert (out == 0).all()


def test_sampling_prepares_the_next_decode_step_on_the_device():
    """Greedy and seeded rows; two cache groups with pages of 4 and 8 slots; a padded row is left alone;
    a position past the block table's end gets slot -1."""
    g = torch.Generator().manual_seed(21)
    rows, vocab, n_stride, r_stride, max_blocks = 5, 300, 8, 6, 4
    page_sizes = [4, 8]
    positions = [3, 7, 0, 15, 9]
    q_req = [0, 1, -1, 3, 4]
    bt = torch.randint(0, 50, (2, r_stride, max_blocks), generator=g, dtype=torch.int32)
    bt[0, 1, 2] = -1                     # request 1 has no page yet for position 8 in group 0
    tok0 = torch.randint(0, vocab, (n_stride,), generator=g, dtype=torch.int32)
    d = dict(token_ids=tok0.clone().to(DEV), positions=i32(positions + [0] * 3),
             seq_lens=i32([p + 1 for p in positions] + [0]), q_req=i32(q_req + [-1] * 3),
             slot_mapping=torch.full((2, n_stride), -7, dtype=torch.int32, device=DEV), block_tables=bt.to(DEV),
             page_sizes=i32(page_sizes), history=torch.full((3, 6), -5, dtype=torch.int32, device=DEV),
             history_pos=torch.zeros(6, dtype=torch.int32, device=DEV))
    out_index = i32([0, 4, 2, 9, 1])
    temps = torch.tensor([0.0, 0.9, 0.0, 1.3, 0.0], device=DEV)
    seeds = torch.tensor([5, 6, 7, 8, 9], dtype=torch.int64, device=DEV)
    out = torch.full((rows,), -1, dtype=torch.int32, device=DEV)
    advance = tuple(d[k] for k in ("token_ids", "positions", "seq_lens", "q_req", "slot_mapping", "block_tables",
                                   "page_sizes", "history", "history_pos"))
    want_tokens = []
    for step in range(2):
        logits = rnd(g, rows, vocab, scale=2.0)
        idx_before = out_index.cpu().tolist()
        kernels.sample(logits.to(DEV), rows, vocab, temps, None, None, seeds, out_index, 3, out, advance=advance)
        plain = torch.full((rows,), -1, dtype=torch.int32, device=DEV)
        kernels.sample(logits.to(DEV), rows, vocab, temps, None, None, seeds, i32(idx_before), 3, plain)
        assert torch.equal(out, plain), "advancing must not change what is sampled"
        want_tokens.append(plain.cpu().tolist())
        for r in range(rows):
            if q_req[r] < 0:
                assert d["token_ids"][r].item() == tok0[r].item() and d["positions"][r].item() == positions[r]
                assert d["history_pos"][r].item() == 0 and out_index[r].item() == 2
                assert d["slot_mapping"][:, r].cpu().tolist() == [-7, -7]
                continue
            pos = positions[r] + step + 1
            assert d["token_ids"][r].item() == want_tokens[step][r]
            assert d["positions"][r].item() == pos and d["seq_lens"][r].item() == pos + 1
            assert out_index[r].item() == idx_before[r] + 1
            assert d["history_pos"][r].item() == step + 1 and d["history"][step, r].item() == want_tokens[step][r]
            for grp, ps in enumerate(page_sizes):
                page = bt[grp, r, pos // ps].item() if pos // ps < max_blocks else -1
                assert d["slot_mapping"][grp, r].item() == (page * ps + pos % ps if page >= 0 else -1)
    assert (d["history"][2] == -5).all() and (d["history"][:, 5] == -5).all()


@pytest.mark.parametrize("vocab", [257, 503, 5000])
def test_seeded_sampling_matches_the_plain_sampler(vocab):
    g = torch.Generator().manual_seed(9)
    m = 24
    logits = rnd(g, m, vocab, scale=2.0)
    temps = [0.8, 1.0, 0.3, 1.7] * (m // 4)
    top_k = [0, 5, 0, 40, 1, 0] * (m // 6)
    top_p = [1.0, 1.0, 0.7, 0.9, 1.0, 0.2] * (m // 6)
    seeds, idx = list(range(100, 100 + m)), [3 * i for i in range(m)]
    got = _sample(logits, temps, top_k, top_p, seeds, idx, engine_seed=42)
    assert got == _sample(logits, temps, top_k, top_p, seeds, idx, engine_seed=42)       # deterministic
    for r in range(m):
        u = P.plain_uniform(42, seeds[r], idx[r])
        tok, lo, hi, total = P.plain_sample(logits[r].numpy(), temps[r], top_k[r] or None,
                                            top_p[r] if top_p[r] < 1 else None, u)
        if got[r] != tok:
            # float32 prefix sums may move a boundary by rounding: then u must sit on that boundary
            edge = min(abs(u * total - lo), abs(u * total - hi))
            assert edge <= 1e-4 * total, f"row {r}: kernel {got[r]}, plain {tok}, u {u}"


@pytest.mark.parametrize("vocab", [1, 3, 1023, 1025, 16384, 16385, 32769, 50257, 53249, 65536, 65537])
def test_sampling_from_held_rows(vocab):
    """Rows of up to 65,536 logits are held in registers, 1 to 64 a thread; longer ones are read again.  The lists of the
    two searches, their ends, ties, infinities and a temperature that makes different logits equal."""
    g = torch.Generator().manual_seed(vocab)
    opts = [(0.8, 0, 1.0), (0.7, 50, 0.95), (1.0, 1, 1.0), (1.3, 0, 0.9), (0.5, 0, 0.05), (3.9, 512, 0.99), (1.0, 513, 1.0),
            (5.0, 20, 1.0), (1e9, 3, 1.0), (0.9, vocab, 0.5), (0.9, max(vocab - 1, 1), 0.5), (1.0, 40, 1.0)]
    m = 3 * len(opts)
    logits = rnd(g, m, vocab, scale=2.0)
    logits[len(opts):2 * len(opts)] = (logits[len(opts):2 * len(opts)] * 4).round() / 4          # ties, lists too long
    low = logits[2 * len(opts):]
    low[torch.rand(low.shape, generator=g) < 0.5] = float("-inf")                                # masked rows
    low[:, -1] = 1.5
    temps, top_k, top_p = (list(x) * 3 for x in zip(*opts))
    seeds, idx = list(range(7, 7 + m)), [5 * i for i in range(m)]
    got = _sample(logits, temps, top_k, top_p, seeds, idx, engine_seed=11)
    assert got == _sample(logits, temps, top_k, top_p, seeds, idx, engine_seed=11)
    for r in range(m):
        u = P.plain_uniform(11, seeds[r], idx[r])
        tok, lo, hi, total = P.plain_sample(logits[r].numpy(), temps[r], top_k[r] or None,
                                            top_p[r] if top_p[r] < 1 else None, u)
        if got[r] != tok:      # sums of float32: u must sit on a boundary, as above
            edge = min(abs(u * total - lo), abs(u * total - hi))
            assert edge <= 1e-4 * total, f"row {r}: kernel {got[r]}, plain {tok}, u {u}, options {opts[r % len(opts)]}"


@pytest.mark.parametrize("top_p", [0.0, -0.5, float("-inf")])
@pytest.mark.parametrize("vocab,top_k", [(50, 20), (3000, 512), (3000, 0), (70000, 40)])
def test_a_top_p_of_nothing_keeps_the_largest_logit(vocab, top_k, top_p):
    """As the reference, which drops a token for the mass before it and never the first; over the list of candidates, all
    registers, and a row that is read again."""
    logits = rnd(torch.Generator().manual_seed(vocab), 4, vocab)
    got = _sample(logits, [0.9] * 4, [top_k] * 4, [top_p] * 4, list(range(4)), [1] * 4)
    assert got == logits.argmax(dim=1).tolist()


@pytest.mark.parametrize("logit,keeps", [(-0.46050000190734863, False), (-0.41769999265670776, True)])
def test_top_p_of_a_long_list_adds_masses_up_without_a_drift(logit, keeps):
    """One logit, 400 equal ones below it and 100 below those, of which the mass above ends 0.75e-6 beside top-p: additions one by one
    in float32 are off by 1.5e-6 here (expf by up to 1e-7, the mass of all that is kept and p by 1e-7)."""
    logits = torch.full((64, 600), -30.0)
    logits[:, 0], logits[:, 1:401], logits[:, 401:501] = 0.0, logit, logit - 0.01
    mass = logits[0, :501].double().exp()
    above = mass[:401].sum().item()
    p = above * (1 + (0.75e-6 if keeps else -0.75e-6)) / mass.sum().item()
    got = _sample(logits, [1.0] * 64, [501] * 64, [p] * 64, list(range(64)), [1] * 64)
    assert any(token > 400 for token in got) == keeps and max(got) < 501


def test_reference_vectors_top_k_top_p():
    # reference tests/test_sampling.py:25-38
    logits = torch.tensor([[1.0, 5.0, 3.0, 2.0, 4.0]] * 64)
    got = set(_sample(logits, [1.0] * 64, top_k=[2] * 64, seeds=list(range(64)), idx=[0] * 64))
    assert got == {1, 4}
    logits = torch.tensor([[10.0, 0.0, 0.0, 0.0]] * 64)
    assert set(_sample(logits, [1.0] * 64, top_p=[1e-6] * 64, seeds=list(range(64)), idx=[0] * 64)) == {0}
    # mixed rows: greedy beside stochastic (reference test_sampling.py:56-63)
    g = torch.Generator().manual_seed(10)
    logits = rnd(g, 2, 30)
    assert _sample(logits, [0.0, 1.0], seeds=[1, 2], idx=[0, 0])[0] == int(torch.argmax(logits[0]))


def test_sampling_follows_the_distribution():
    probs = torch.tensor([0.5, 0.25, 0.125, 0.125])
    m = 4096
    logits = probs.log().repeat(m, 1)
    got = np.bincount(_sample(logits, [1.0] * m, seeds=[7] * m, idx=list(range(m))), minlength=4) / m
    assert np.abs(got - probs.numpy()).max() < 0.03
