"""The products of many rows (``csrc/tile_gemm.hip``) alone: every tile at its edges, every epilogue, shares, and the
error beside the library's float32 product."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    from nanoinfer_amd import kernels
    return kernels


def operands(M, N, Kd, seed=0, spread=0):
    g = torch.Generator().manual_seed(seed)
    x, w = torch.randn(M, Kd, generator=g), torch.randn(N, Kd, generator=g)
    if spread:      # rows of very different size: powers of two, so that the sums' relative errors stay what they are
        x *= 2.0 ** torch.randint(-spread, spread + 1, (M, 1), generator=g)
    return x.cuda(), w.cuda()


def close(got, x, w, whole=None):
    """Every number within the bound of a float32 sum of 6 K exact products: (6 K + 8) roundings of at most 2^-24 of
    sum |x||w| each (the three products left out are together at most one of them).  And all of them together within
    ``whole`` of what such sums come to, the root of sum x^2 w^2."""
    want, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    assert bool(((got.double() - want).abs() <= (6 * x.shape[1] + 8) * 2.0 ** -24 * size).all())
    if whole is not None:
        assert float((got.double() - want).norm() / ((x.double() ** 2) @ (w.double() ** 2).t()).sqrt().norm()) <= whole
    return float((got.double() - want).norm() / want.norm())


# With any one of the six products left out, results are off as a whole by 2.4e-6 (the two with a last part), 2.7e-6 (the
# middle parts) or 1.6e-3 and more, worked out in 64 bits for operands like those here; a float32 sum of 100 to 2,048 products
# by 1.8e-7 to 3.2e-7.  In between, for sums of so many:
WHOLE = 2.0 ** -20


@pytest.mark.parametrize("tile", [0, 1, 2, 3])
@pytest.mark.parametrize("M,N,Kd,shares", [(1, 1, 4, 1), (63, 255, 20, 1), (64, 256, 16, 1), (65, 257, 36, 1), (129, 130, 100, 1),
                                           (257, 513, 132, 1), (300, 258, 300, 2), (70, 77, 1036, 3), (256, 128, 2048, 16)])
def test_split_gemm_at_the_edges_of_its_tiles(K, tile, M, N, Kd, shares):
    x, w = operands(M, N, Kd, seed=M + N + Kd, spread=30)
    out = torch.full((M + 1, N), 7.0, device="cuda")
    K.split_gemm(x, w, out[:M], plan=(tile, shares))
    close(out[:M], x, w, WHOLE)
    assert bool((out[M] == 7.0).all())                       # nothing behind the last row


@pytest.mark.parametrize("tile", [0, 1, 2, 3])
def test_a_single_product(K, tile):
    """Rows with one number each, so that a result is one product: off by what is left out (2^-24 of it at most) and by the
    sums of the six, the last of which the matrix cores may cut (2^-23) and the others are of numbers 2^-7 as large.
    Measured up to 2.7 times 2^-24.  The mantissas are those that leave the most out and random ones."""
    g = torch.Generator().manual_seed(tile)
    worst = torch.tensor([0x3f807fc0, 0x3f80ff80, 0x3f80ffff, 0x3f807fff, 0x3fffffff, 0x3f800001], dtype=torch.int32).view(torch.float32)

    def numbers(n):
        bits = torch.randint(0, 1 << 23, (n,), generator=g, dtype=torch.int32) + 0x3f800000
        v = bits.view(torch.float32).clone()
        v[:len(worst)] = worst
        return v * torch.where(torch.rand(n, generator=g) < 0.5, -1.0, 1.0) * 2.0 ** torch.randint(-40, 41, (n,), generator=g)

    M, N, Kd = 300, 270, 36
    x, w = torch.zeros(M, Kd), numbers(N)[:, None].expand(N, Kd).contiguous()
    x[torch.arange(M), torch.arange(M) % Kd] = numbers(M)
    want = x.double() @ w.double().t()
    got = K.split_gemm(x.cuda(), w.cuda(), plan=(tile, 1)).cpu().double()
    assert bool(((got - want).abs() <= 3.1 * 2.0 ** -24 * want.abs()).all())


@pytest.mark.parametrize("tile", [0, 1, 2, 3])
@pytest.mark.parametrize("M,inter", [(65, 1), (64, 32), (130, 100), (129, 129), (257, 300)])
def test_split_gemm_gated_and_squared(K, tile, M, inter):
    x, w = operands(M, 2 * inter, 68, seed=inter)
    z = K.split_gemm(x, w, plan=(tile, 1))
    for act in ("silu", "gelu_tanh"):
        # the epilogue applies what the kernel of its own applies to the same float32 sums
        got = K.split_gemm(x, w, gated=act, plan=(tile, 1))
        assert torch.allclose(got, K.swiglu(z, torch.empty_like(got), act), rtol=1e-6, atol=0)
    assert torch.equal(K.split_gemm(x, w, squared=True, plan=(tile, 1)), torch.relu(z) ** 2)
    assert torch.equal(K.split_gemm(x, w, squared=True, plan=(tile, 2)), torch.relu(K.split_gemm(x, w, plan=(tile, 2))) ** 2)


@pytest.mark.parametrize("M,N,Kd", [(65, 16384, 2048), (512, 2048, 8192), (512, 3072, 3072), (1000, 2500, 700)])
def test_products_of_many_float32_rows_are_no_less_exact_than_the_librarys(K, M, N, Kd):
    x, w = operands(M, N, Kd)
    assert K.split_wins(x, w)
    calls = K.library_calls()
    ours = close(K.linear(x, w), x, w, 2 * WHOLE)
    assert K.library_calls() == calls
    assert ours <= 1.05 * close(torch.mm(x, w.t()), x, w)     # measured 0.6 to 0.9
    g = K.linear_swiglu(x, w)
    want = torch.nn.functional.silu(x.double() @ w[:N // 2].double().t()) * (x.double() @ w[N // 2:].double().t())
    assert float((g.double() - want).norm() / want.norm()) <= 1e-5
    assert K.library_calls() == calls


def test_rows_that_are_not_finite_stay_so_and_touch_no_other(K):
    x, w = operands(130, 300, 64)
    x[3, 5], x[70, 0], x[129, 63] = float("inf"), float("nan"), float("-inf")
    got = K.split_gemm(x, w)
    bad = torch.zeros(130, dtype=torch.bool)
    bad[[3, 70, 129]] = True
    assert not bool(torch.isfinite(got[bad.cuda()]).any())
    close(got[~bad.cuda()], x[~bad.cuda()], w)


def same(got, want, rtol=1e-5):
    """The same infinities with the same signs, NaN in the same places, the finite rest within rtol of its largest in a row."""
    got, want = got.double().cpu(), want.double().cpu()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(torch.isinf(got) * torch.sign(got), torch.isinf(want) * torch.sign(want))
    fine = torch.isfinite(want)
    a, b = torch.where(fine, got, 0.0), torch.where(fine, want, 0.0)
    assert bool(((a - b).abs() <= rtol * b.abs().amax(dim=1, keepdim=True)).all())


def not_finite(M, N, Kd, seed=3, huge=True):
    """Operands with infinities of both signs, NaN, zeros that meet an infinity and (``huge``) numbers near the type's
    largest, whose bfloat16 is infinite; with the exact products, as float32 holds them."""
    x, w = operands(M, N, Kd, seed=seed)
    inf, nan = float("inf"), float("nan")
    x[3, 5], x[70, 0], x[M - 1, Kd - 1], x[9, 8], x[9, 9] = inf, nan, -inf, inf, -inf
    w[11, 2], w[N // 2 + 11, 7], w[N - 1, 3], w[41, 5] = -inf, inf, nan, 0.0
    if huge:
        x[20], x[21], w[40] = 3.4e38, 3.4e38 * torch.sign(x[21]), 1e-30
    return x, w, (x.cpu().double() @ w.cpu().double().t()).float()


@pytest.mark.parametrize("tile", [0, 1, 2, 3])
@pytest.mark.parametrize("M,N,Kd", [(130, 300, 64), (300, 130, 132)])
def test_what_is_not_finite_stays_what_a_float32_product_makes_of_it(K, tile, M, N, Kd):
    x, w, z = not_finite(M, N, Kd)
    same(K.split_gemm(x, w, plan=(tile, 1)), z)
    # cut along K: the shares' sums, each as float32 holds it (two that overflow may cancel to NaN where one sum would not)
    parts = K.split_gemm(x, w, plan=(tile, 2), addends=True)
    per = -(-Kd // 32) * 16
    for p, at in zip(parts, (0, per)):
        same(p, (x[:, at:at + per].cpu().double() @ w[:, at:at + per].cpu().double().t()).float())
    same(K.split_gemm(x, w, plan=(tile, 2)), parts[0] + parts[1])
    same(K.split_gemm(x, w, squared=True, plan=(tile, 1)), torch.relu(z) ** 2)
    same(K.split_gemm(x, w, squared=True, plan=(tile, 2)), torch.relu(parts[0] + parts[1]) ** 2)
    for act in ("silu", "gelu_tanh"):
        same(K.split_gemm(x, w, gated=act, plan=(tile, 1)), K.swiglu(z.cuda(), torch.empty(M, N // 2, device="cuda"), act), 1e-4)


def test_feed_forwards_of_rows_that_are_not_finite(K):
    """The same through the entry points, where the rule sends such products to these kernels."""
    x, w, z = not_finite(300, 4096, 1024, huge=False)
    calls = K.library_calls()
    assert K.split_wins(x, w)
    same(K.linear(x, w), z)
    same(K.linear_relu2(x, K.Weight(w)), torch.relu(z) ** 2)
    same(K.linear_swiglu(x, w), K.swiglu(z.cuda(), torch.empty(300, 2048, device="cuda")), 1e-4)
    assert K.library_calls() == calls


@pytest.mark.parametrize("tile", [0, 1, 2, 3])
def test_experts_of_tokens_that_are_not_finite(K, monkeypatch, tile):
    """An infinity in a token, in an expert's rows: as all experts run as two float32 products would have it, but for the
    experts that a token did not choose, which it does not meet."""
    from nanoinfer_amd.kernels import tile as tiles
    monkeypatch.setattr(tiles, "_grouped_plan", lambda *a: (0.0, tile))
    T, d, ff, E, top = 150, 64, 36, 5, 2
    g = torch.Generator().manual_seed(5)
    x, up, down = torch.randn(T, d, generator=g), torch.randn(E * ff, d, generator=g), torch.randn(d, E * ff, generator=g)
    chosen = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(T)]).int()
    mix = torch.rand(T, top, generator=g) + 0.1
    inf = float("inf")
    x[4, 3], x[77, 0], x[149, 63], up[2 * ff + 5, 9], down[7, 3 * ff + 1] = inf, float("nan"), -inf, -inf, inf
    want = torch.zeros(T, d, dtype=torch.float64)
    for t in range(T):
        for k in range(top):
            e = int(chosen[t, k])
            hid = mix[t, k].double() * torch.relu(up[e * ff:(e + 1) * ff].double() @ x[t].double()) ** 2
            want[t] += (down[:, e * ff:(e + 1) * ff].double() * hid).sum(dim=1)
    got = K.experts_grouped(x.cuda(), up.cuda(), down.cuda(), chosen.cuda(), mix.cuda(), E, lambda z, w: K.experts_act(z, w, ff, "relu2"))
    same(got, want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_addends_go_with_nothing_else(K, dtype):
    """A product that leaves its addends would leave an ``out`` unwritten and an activation undone: refused, and a linear
    product with an ``out`` writes it."""
    x, w = (t.to(dtype) for t in operands(300, 2048, 4096))
    weight, out = K.Weight(w), torch.full((300, 2048), 7.0, device="cuda", dtype=dtype)
    product = (lambda **k: K.split_gemm(x, w, plan=(1, 2), **k)) if dtype == torch.float32 else (lambda **k: K.tiled_gemm(x, weight, plan=(1, 2), **k))
    assert product(addends=True).shape == (2, 300, 2048)
    for more in ({"out": out}, {"squared": True}, {"gated": "silu"}):
        with pytest.raises(K.KernelError):
            product(addends=True, **more)
    assert K.linear(x, weight, addends=True).dim() == 3
    assert torch.equal(K.linear(x, weight, out=out, addends=True), K.linear(x, weight)) and torch.equal(out, K.linear(x, weight))


def test_what_split_gemm_does_not_take(K):
    x, w = operands(70, 64, 64)
    for bad in (lambda: K.split_gemm(x[:, :62].contiguous(), w[:, :62].contiguous()), lambda: K.split_gemm(x.bfloat16(), w.bfloat16()),
                lambda: K.split_gemm(x, w[:, :60].contiguous()), lambda: K.split_gemm(x.view(-1)[1:1 + 69 * 64].view(69, 64), w),
                lambda: K.split_gemm(x, w[:63], gated="silu"), lambda: K.split_gemm(x.t(), w)):
        with pytest.raises(K.KernelError):
            bad()
    big, wide = operands(600, 1024, 2048)
    calls = K.library_calls()                                 # rows that are no whole run of memory, or not aligned: the library's product
    assert K.linear(big.t().contiguous().t(), wide).shape == (600, 1024)
    assert K.linear(torch.randn(600 * 2048 + 1, device="cuda")[1:].view(600, 2048), wide).shape == (600, 1024)
    assert K.library_calls() == calls + 2


@pytest.mark.parametrize("offset", [1, 2, 3])
def test_results_that_start_at_any_number(K, offset):
    """A caller's ``out`` need not start at 16 bytes: whole, added up from shares, and the experts' sum."""
    x, w = operands(512, 1056, 2048)
    aside = torch.full((512 * 1056 + 8,), 7.0, device="cuda")
    for plan in ((1, 1), (1, 3)):
        out = aside[offset:offset + 512 * 1056].view(512, 1056)
        assert torch.equal(K.split_gemm(x, w, out, plan=plan), K.split_gemm(x, w, plan=plan))
        assert bool((aside[:offset] == 7.0).all()) and bool((aside[offset + 512 * 1056:] == 7.0).all())
    calls = K.library_calls()
    assert K.linear(x, w, out=out).data_ptr() == out.data_ptr() and K.library_calls() == calls
    g = torch.Generator().manual_seed(offset)
    chosen = torch.stack([torch.randperm(5, generator=g)[:2] for _ in range(70)]).int().cuda()
    tokens, up, down, mix = (torch.randn(s, generator=g).cuda() for s in ((70, 64), (5 * 36, 64), (64, 5 * 36), (70, 2)))
    out = aside[offset:offset + 70 * 64].view(70, 64)
    act = lambda z, weights: K.experts_act(z, weights, 36, "relu2")     # noqa: E731
    assert torch.equal(K.experts_grouped(tokens, up, down, chosen, mix, 5, act, out=out), K.experts_grouped(tokens, up, down, chosen, mix, 5, act))
    assert bool((aside[:offset] == 7.0).all())


@pytest.mark.parametrize("T,d,ff,E,top,kind", [(1, 4, 4, 1, 1, "any"), (65, 36, 20, 5, 2, "any"), (300, 64, 132, 16, 4, "any"), (257, 68, 64, 7, 3, "one"),
                                               (130, 40, 36, 6, 2, "identity"), (1500, 128, 64, 16, 4, "any")])
@pytest.mark.parametrize("tile", [0, 1, 2, 3])
def test_every_expert_multiplies_its_own_tokens(K, monkeypatch, tile, T, d, ff, E, top, kind):
    """Lists of every shape (an expert without tokens, one with all, entries that name no expert), whole against 64 bits."""
    from nanoinfer_amd.kernels import tile as tiles
    monkeypatch.setattr(tiles, "_grouped_plan", lambda *a: (0.0, tile))
    g = torch.Generator().manual_seed(T + d)
    x, up, down = torch.randn(T, d, generator=g), torch.randn(E * ff, d, generator=g), torch.randn(d, E * ff, generator=g)
    total = E + (3 if kind == "identity" else 0)
    chosen = torch.stack([torch.randperm(total, generator=g)[:top] for _ in range(T)]).int()
    if kind == "one":                  # one expert has every token, the last has none
        chosen[:, 0] = 2
        chosen[:, 1:] = torch.tensor([0, 4])
    mix = torch.rand(T, top, generator=g)
    want, size = torch.zeros(T, d, dtype=torch.float64), torch.zeros(T, d, dtype=torch.float64)
    for t in range(T):
        for k in range(top):
            e = int(chosen[t, k])
            if e < E:
                u, n = up[e * ff:(e + 1) * ff].double(), down[:, e * ff:(e + 1) * ff].double()
                hid = mix[t, k].double() * torch.relu(u @ x[t].double()) ** 2
                want[t] += n @ hid
                size[t] += n.abs() @ (mix[t, k].double() * (u.abs() @ x[t].double().abs()) ** 2)
    got = K.experts_grouped(x.cuda(), up.cuda(), down.cuda(), chosen.cuda(), mix.cuda(), E,
                            lambda z, w: K.experts_act(z, w, ff, "relu2")).cpu().double()
    # two products and a square, each a float32 sum: (2 (6 d + 8) + (6 ff + 8) + top + 4) roundings of the sums of sizes
    assert bool(((got - want).abs() <= (12 * d + 6 * ff + 28 + top) * 2.0 ** -24 * size + 1e-30).all())
    # and as a whole: the second product's error and twice the first's, as its sums are squared
    assert float((got - want).norm() / want.norm()) <= 1.5 * WHOLE


@pytest.mark.parametrize("tile", [0, 1, 2, 3])
@pytest.mark.parametrize("M,N,Kd,shares", [(1, 4, 64, 1), (63, 60, 128, 1), (65, 68, 192, 1), (129, 260, 256, 1), (257, 132, 320, 1),
                                           (130, 516, 448, 2), (200, 96, 1024, 3), (64, 256, 2048, 8)])
def test_tiled_gemm_at_the_edges_of_its_tiles(K, tile, M, N, Kd, shares):
    x, w = (t.bfloat16() for t in operands(M, N, Kd, seed=M + N + Kd, spread=20))
    weight = K.Weight(w)
    for dtype in (torch.float32, torch.bfloat16):
        out = torch.full((M + 1, N), 7.0, device="cuda", dtype=dtype)
        K.tiled_gemm(x, weight, dtype, out[:M], plan=(tile, shares))
        want, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
        # K exact products in a float32 sum (K + 8 roundings), and the rounding of the result
        bound = (Kd + 8) * 2.0 ** -24 * size + (2.0 ** -8 * want.abs() if dtype == torch.bfloat16 else 0)
        assert bool(((out[:M].double() - want).abs() <= bound).all()), dtype
        assert bool((out[M] == 7.0).all())
    if shares > 1:
        parts = K.tiled_gemm(x, weight, plan=(tile, shares), addends=True)
        assert parts.dtype == torch.float32 and parts.dim() == 3
        total = parts[0].clone()
        for p in parts[1:]:
            total += p
        assert torch.equal(total, K.tiled_gemm(x, weight, torch.float32, plan=(tile, shares)))


@pytest.mark.parametrize("tile", [0, 1, 2])
@pytest.mark.parametrize("M,inter", [(65, 16), (64, 32), (130, 112), (129, 144)])
def test_tiled_gemm_gated_and_squared(K, tile, M, inter):
    x, w = (t.bfloat16() for t in operands(M, 2 * inter, 192, seed=inter))
    weight = K.Weight(w)
    z = K.tiled_gemm(x, weight, torch.float32, plan=(tile, 1))
    for act in ("silu", "gelu_tanh"):
        want = K.swiglu(z, torch.empty(M, inter, device="cuda"), act)
        got = K.tiled_gemm(x, weight, gated=act, plan=(tile, 1)).float()
        # one rounding to bfloat16, and the hardware's exponential (2^-20 of the value)
        assert bool(((got - want).abs() <= (2.0 ** -8 + 2.0 ** -18) * want.abs() + 1e-30).all())
    for shares in (1, 2):
        whole = K.tiled_gemm(x, weight, torch.float32, plan=(tile, shares))
        assert torch.equal(K.tiled_gemm(x, weight, torch.float32, squared=True, plan=(tile, shares)), torch.relu(whole) ** 2)


def test_where_bfloat16_products_go(K):
    """65 to 512 rows (1,024 with SwiGLU) of a re-tiled matrix are multiplied here, the library is not asked; what the kernel
    cannot take goes to the library as before."""
    x, w = (t.bfloat16() for t in operands(600, 2080, 256))
    weight, odd = K.Weight(w), K.Weight(w[:2079].contiguous())
    calls = K.library_calls()
    K.linear(x[:65], weight), K.linear(x[:512], weight, out_dtype=torch.float32), K.linear_swiglu(x, weight), K.linear_relu2(x[:200], weight)
    assert K.library_calls() == calls
    aside = torch.empty(600 * 2080 + 1, device="cuda", dtype=torch.bfloat16)[1:].view(600, 2080)
    for n, f in enumerate((lambda: K.linear(x, weight), lambda: K.linear(x[:200], odd), lambda: K.linear(x[:100], w),
                           lambda: K.linear(x[:100], K.Weight(w, tiled=False)), lambda: K.linear(x[:200, :200].contiguous(), K.Weight(w[:, :200].contiguous())),
                           lambda: K.linear(x[:200], weight, out=aside[:200]), lambda: K.linear(x[:70], weight, out=aside[:70]),
                           lambda: K.linear(x.view(-1)[1:1 + 70 * 256].view(70, 256), weight))):
        got = f()
        assert K.library_calls() == calls + n + 1 and bool(torch.isfinite(got).all()), n
    for bad in (lambda: K.tiled_gemm(x.float(), weight), lambda: K.tiled_gemm(x, w), lambda: K.tiled_gemm(x[:, :128].contiguous(), weight),
                lambda: K.tiled_gemm(x, odd), lambda: K.tiled_gemm(x, K.Weight(w[:48].contiguous()), gated="silu"),
                lambda: K.tiled_gemm(x[:100], weight, out=aside[:100])):
        with pytest.raises(K.KernelError):
            bad()
