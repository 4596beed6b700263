"""A norm between two products of many bfloat16 rows, half done by each (``csrc/row_norm.h``): what the product onto the residual stream
leaves, and what the products behind it make of that."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    from nanoinfer_amd import kernels
    return kernels


def draw(*shape, seed, scale=1.0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale


# rows and columns: one, the edges of the tiles, several groups of tiles; K: fewer stages than the rings have, and more
@pytest.mark.parametrize("tile", [0, 1, 2, 3])
@pytest.mark.parametrize("M,N,Kd", [(1, 64, 64), (127, 256, 128), (129, 192, 320), (257, 320, 64), (1100, 512, 384), (600, 2048, 640)])
def test_what_is_left_beside_the_stream(K, tile, M, N, Kd):
    x, w = draw(M, Kd, seed=M).bfloat16().cuda(), draw(N, Kd, seed=N).bfloat16().cuda()
    h, weight = draw(M, N, seed=1, scale=8.0).cuda(), draw(N, seed=2).cuda()
    product, size = x.cpu().double() @ w.cpu().double().t(), x.cpu().double().abs() @ w.cpu().double().abs().t()
    want = h.cpu().double() + product
    guarded = torch.full((M + 1, N), 7.0, device="cuda")
    guarded[:M] = h
    left, ss = K.wide_stream(x, w, guarded[:M], weight, tile=tile)
    got = guarded[:M].cpu().double()
    # a float32 sum of K products of bfloat16 numbers (exact in float32), and the one onto the stream
    assert bool(((got - want).abs() <= (Kd + 1) * 2.0 ** -24 * (size + h.cpu().double().abs())).all()) and bool((guarded[M] == 7.0).all())
    assert torch.equal(left, (guarded[:M] * weight).bfloat16())
    sums = (got ** 2).view(M, N // 64, 64).sum(2)
    assert bool(((ss.cpu().double() - sums).abs() <= 66 * 2.0 ** -24 * sums).all())
    again = h.clone()
    assert K.wide_stream(x, w, again, tile=tile) == (None, None) and torch.equal(again, guarded[:M])


@pytest.mark.parametrize("tile", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("M,inter,Kd", [(1, 32, 256), (129, 96, 512), (300, 160, 1024), (600, 512, 2048), (257, 64, 4096)])
def test_rows_are_divided_in_the_product_behind(K, tile, M, inter, Kd):
    """By a factor a row: as good as the product of rows that were divided before, in float32, and gated."""
    h, weight = draw(M, Kd, seed=M, scale=3.0).cuda(), draw(Kd, seed=3).cuda()
    h *= 2.0 ** torch.arange(M, device="cuda").remainder(9)[:, None]
    left, ss = (h * weight).bfloat16(), (h ** 2).view(M, Kd // 64, 64).sum(2)
    eps = 1e-5
    w = draw(2 * inter, Kd, seed=inter, scale=Kd ** -0.5).bfloat16().cuda()
    got = K.wide_gemm(K.ScaledInput(left, ss, K.NormSpec(weight, eps)), w, gated="silu", tile=tile).cpu().double()
    f = ((h.cpu().double() ** 2).mean(1, keepdim=True) + eps).rsqrt()
    z = (left.cpu().double() @ w.cpu().double().t()) * f
    off = (Kd + 48) * 2.0 ** -24 * (left.cpu().double().abs() @ w.cpu().double().abs().t()) * f      # of gate and of up
    gate, up = z[:, :inter], z[:, inter:]
    # |d act| <= 1.1 |d gate|, |act| <= |gate|; the quick exponential is within 2^-20; rounded to bfloat16 once
    bound = 1.1 * off[:, :inter] * up.abs() + gate.abs() * off[:, inter:] + (2.0 ** -8 + 2.0 ** -20) * (gate * up).abs() + 1e-30
    assert bool(((got - torch.nn.functional.silu(gate) * up).abs() <= bound).all())


@pytest.mark.parametrize("tile", [0, 1, 2, 3])
@pytest.mark.parametrize("M,H,KVH,hd,Kd", [(65, 1, 1, 64, 256), (300, 3, 1, 128, 512), (1100, 6, 2, 64, 768)])
def test_rotated_behind_the_division(K, tile, M, H, KVH, hd, Kd):
    """The rotation is linear: a row that is divided by a power of two comes out divided by it, bit for bit."""
    x, w = draw(M, Kd, seed=M).bfloat16().cuda(), draw((H + 2 * KVH) * hd, Kd, seed=5).bfloat16().cuda()
    half = draw(M, hd // 2, seed=6).cuda()
    cos, sin = half.cos().contiguous(), half.sin().contiguous()
    positions = torch.arange(M, device="cuda", dtype=torch.int32)
    pools = [torch.full(((M + 15) // 16, KVH, 16, hd), 7.0, device="cuda", dtype=torch.bfloat16) for _ in range(4)]
    weight = K.Weight(w, tiled=False)
    q = K.qkv_rope(x, weight, positions, cos, sin, positions, pools[0], pools[1], H, KVH, hd, (False, tile))
    power = 2.0 ** torch.arange(M, device="cuda").remainder(5).float()
    ss = torch.zeros(M, Kd // 64, device="cuda")
    ss[:, ::2] = (power ** 2 * Kd / ((Kd // 64 + 1) // 2))[:, None]
    got = K.qkv_rope(K.ScaledInput(x, ss, K.NormSpec(torch.ones(Kd, device="cuda"), 0.0)), weight, positions, cos, sin, positions, pools[2], pools[3], H, KVH, hd,
                     (False, tile))
    assert torch.equal(got.float() * power[:, None], q.float())
    for a, b in ((pools[0], pools[2]), (pools[1], pools[3])):
        rows = [t.permute(0, 2, 1, 3).reshape(-1, KVH * hd)[:M].float() for t in (a, b)]
        assert torch.equal(rows[1] * power[:, None], rows[0])


def test_what_they_do_not_take(K):
    x, w, h = (torch.zeros(s, device="cuda", dtype=t) for s, t in (((70, 64), torch.bfloat16), ((128, 64), torch.bfloat16), ((70, 128), torch.float32)))
    scaled = K.ScaledInput(x, torch.zeros(70, 1, device="cuda"), K.NormSpec(torch.ones(64, device="cuda"), 1e-5))
    for bad in (lambda: K.wide_stream(x, w[:100], h[:, :100].contiguous()), lambda: K.wide_stream(x, w, h.bfloat16()), lambda: K.wide_stream(x[:, :32].contiguous(), w[:, :32].contiguous(), h),
                lambda: K.wide_stream(x, w, h, torch.ones(64, device="cuda")), lambda: K.wide_gemm(scaled, w, gated="silu"),
                lambda: K.linear(x, K.Weight(w), residual=h), lambda: K.linear_swiglu(scaled, K.Weight(w, tiled=False))):
        with pytest.raises(K.KernelError):
            bad()


def test_rows_and_weights_that_are_not_aligned(K):
    """Rows with a stride, or off sixteen bytes, are copied; a norm's weight off them leaves the norm to its kernel."""
    M, N, Kd = 1999, 2048, 2048
    wide, w = draw(M, Kd + 8, seed=1).bfloat16().cuda(), K.Weight(draw(N, Kd, seed=2).bfloat16().cuda())
    flat = draw(M * Kd + 1, seed=3).bfloat16().cuda()
    weight = draw(N + 1, seed=4).cuda()
    for x in (wide[:, :Kd], flat[1:].view(M, Kd)):
        a, b = torch.zeros(M, N, device="cuda"), torch.zeros(M, N, device="cuda")
        left = K.linear(x, w, residual=a, leave=K.NormSpec(weight[:N], 1e-5))
        assert K.linear(x.clone(memory_format=torch.contiguous_format), w, residual=b, leave=K.NormSpec(weight[1:], 1e-5)) is None
        assert torch.equal(a, b) and torch.equal(left.x, (a * weight[:N]).bfloat16())


def test_a_prompt_with_its_norms_in_halves(K, monkeypatch):
    """A prompt of 1,700 tokens at the 1B layer sizes in one portion, launched and recorded, against the plain implementation; every
    product onto the stream but the last one leaves the next norm's input, and the products behind those take it."""
    from gpu_common import assert_close, model_folder, plain_logits, random_tokens
    from nanoinfer_amd.engine.runner import ModelRunner, StepEntry
    from test_gpu_family_shapes import ALL

    left = []
    stream = K.wide_stream
    monkeypatch.setattr(K, "wide_stream", lambda *a: left.append(len(a)) or stream(*a))
    folder = model_folder("1B", stored="bfloat16")
    tokens, at = random_tokens(ALL["1B"]["vocab_size"], 1700, 5), list(range(1684, 1700))
    for graphs in (False, True):
        runner = ModelRunner(folder, dtype="bfloat16", page_size=16, max_tokens=2048, max_step_tokens=2048, max_requests=2, use_graphs=graphs)
        left.clear()
        got = runner.step([StepEntry(0, tokens, at)]).clone()
        layers = len(runner.model.blocks)
        assert left[:2 * layers] == [4] * (2 * layers - 1) + [3]
        runner.release(0)
        assert_close(got, plain_logits(folder, tokens, "bfloat16")[at], "bfloat16", f"graphs {graphs}")


def test_a_stream_that_is_not_aligned(K):
    """Off sixteen bytes there are no whole vectors to add to: the product goes out alone, and nothing is left for the norm."""
    M, N, Kd = 1999, 2048, 2048
    x, w = draw(M, Kd, seed=1).bfloat16().cuda(), K.Weight(draw(N, Kd, seed=2).bfloat16().cuda())
    h, a = torch.zeros(M * N + 1, device="cuda")[1:].view(M, N), torch.zeros(M, N, device="cuda")
    for t in (h, a):
        t.copy_(draw(M, N, seed=3))
    assert K.linear(x, w, residual=h, leave=K.NormSpec(torch.ones(N, device="cuda"), 1e-5)) is None
    K.linear(x, w, residual=a)
    assert torch.equal(h, a)
    with pytest.raises(K.KernelError):
        K.linear(x, w, residual=h.bfloat16())
