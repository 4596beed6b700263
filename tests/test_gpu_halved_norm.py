"""The norm that leaves its rows as pairs of halves too (``ni_add_rmsnorm_halves``) against the norm and the pass over its rows, which
it stands for, to the bit; and the products that read such rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    from nanoinfer_amd import kernels
    return kernels


# one row and many; the fewest columns, every size of the workgroup, the most; widths that go the long way (no whole stages of 32
# columns, too wide for the registers)
@pytest.mark.parametrize("T,d", [(1, 32), (3, 512), (70, 544), (129, 1056), (130, 2048), (5, 4128), (2, 8192), (3, 2052), (2, 8224)])
@pytest.mark.parametrize("addends", [None, 0, 1, 6])      # none, one [T, d], one and six [S, T, d]
def test_rows_and_halves_are_those_of_the_two_passes(K, T, d, addends):
    g = torch.Generator().manual_seed(T + d)
    h = torch.randn(T, d, generator=g) * 2.0 ** torch.randint(-20, 20, (T, 1), generator=g)
    w = torch.randn(d, generator=g)
    if T > 2:
        h[0] = 0.0                                         # a row of zeros, and rows that are no numbers
        h[1, d - 1] = float("inf")
        h[2, 0] = float("nan")
    h, w = h.cuda(), w.cuda()
    pending = None
    if addends is not None:
        pending = torch.randn(*((T, d) if addends == 0 else (addends, T, d)), generator=g).cuda()
        if T > 2:
            pending.view(-1, T, d)[:, 0] = 0.0
    one, two = h.clone(), h.clone()
    rows = K.add_rmsnorm(one, pending, w, 1e-5, torch.empty(T, d, device="cuda"))
    planes, info = K.pair_rows(rows)
    got = K.add_rmsnorm_halved(two, pending, w, 1e-5)
    assert torch.equal(got.x.view(torch.int32), rows.view(torch.int32)) and torch.equal(one.view(torch.int32), two.view(torch.int32))
    assert torch.equal(got.info, info)
    finite = info[:, 1].cpu() >= 0                         # (the halves of a row with infinities are never read)
    assert torch.equal(got.planes.view(torch.int32).view(T, -1)[finite], planes.view(torch.int32).view(T, -1)[finite])


@pytest.mark.parametrize("T", [65, 600])       # (of [16384, 2048], from 65 rows on)
def test_products_of_halved_rows_are_those_of_rows(K, T):
    g = torch.Generator().manual_seed(T)
    h, w = torch.randn(T, 2048, generator=g).cuda(), torch.ones(2048).cuda()
    weight = K.Weight((torch.randn(16384, 2048, generator=g) / 45).cuda())
    small = K.Weight((torch.randn(64, 2048, generator=g) / 45).cuda())       # goes to another product, which reads the rows
    assert weight.pairs is not None and K.takes_halved(T, 2048, torch.float32, weight) and not K.takes_halved(T, 2048, torch.float32, small)
    x = K.add_rmsnorm_halved(h, None, w, 1e-5)
    for product in (K.linear, K.linear_swiglu, K.linear_relu2):
        assert torch.equal(product(x, weight), product(x.x, weight))
    assert torch.equal(K.linear(x, small), K.linear(x.x, small))


def test_halved_rows_take_less_work_to_go_there(K):
    g = torch.Generator().manual_seed(1)
    weight = K.Weight((torch.randn(3072, 2048, generator=g) / 45).cuda())
    x = K.add_rmsnorm_halved(torch.randn(164, 2048, generator=g).cuda(), None, torch.ones(2048, device="cuda"), 1e-5)
    assert K.pair_wins(x, weight) and not K.pair_wins(x.x, weight)
    assert torch.equal(K.linear(x, weight), K.pair_gemm(x.x, weight))


def test_parts_say_which_rows_they_read(K):
    """A layer that replaces a stage, and a part that knows nothing of halves, are given rows."""
    from nanoinfer_amd.parts import standard

    class Norm(standard.RMSNorm):
        def forward(self, h, pending, rows=None):
            return h

    class Part:
        pass

    h = torch.zeros(600, 64, device="cuda")
    norm = Norm.__new__(Norm)
    norm.rt = type("Runtime", (), {"dtype": torch.float32})()
    assert standard.normed_rows(norm, h, None, (Part(),)) is h
    part = Part()
    part.takes_halved = lambda T: True
    assert standard.normed_rows(norm, h, None, (part,)) is h       # its forward is its own

    class Projects(standard.Attention):
        def project(self, x, ctx):
            return None

    assert not Projects.__new__(Projects).takes_halved(600)


# widths of every size of the workgroup's chunks, and one that is no whole stage of 32 columns; one run and many; runs without a key (sum
# and rows zero, a finite maximum) and rows that are no numbers
@pytest.mark.parametrize("T,H,hd,runs", [(1, 1, 64, 1), (70, 32, 64, 4), (3, 24, 128, 3), (66, 5, 80, 2), (2, 3, 24, 7), (65, 32, 256, 5)])
def test_merged_runs_and_their_halves_are_those_of_the_two_passes(K, T, H, hd, runs):
    g = torch.Generator().manual_seed(T + hd)
    part_o = torch.randn(T, H, runs, hd, generator=g) * 2.0 ** torch.randint(-10, 10, (T, 1, 1, 1), generator=g)
    part_ml = torch.rand(T, H, runs, 2, generator=g) * 20 + 0.1
    if runs > 1:
        part_o[0, 0, 1], part_ml[0, 0, 1] = 0.0, torch.tensor([-1e30, 0.0])
    if T > 2:
        part_o[1] = 0.0
        part_o[2, H - 1, runs - 1, hd - 1] = float("nan")
    part_o, part_ml = part_o.cuda(), part_ml.cuda()
    rows = torch.empty(T, H * hd, device="cuda")
    if hd % 16 == 0:
        K._check(K.attention_lib(hd).ni_merge_splits(K._ptr(part_o), K._ptr(part_ml), K._ptr(rows), T, H, runs, 0, K._stream()), "merge_splits")
    got = K.merge_pair_rows(part_o.view(-1), part_ml.view(-1), torch.empty(T, H * hd, device="cuda"), H, hd, runs)
    if hd % 16 == 0:
        assert torch.equal(got.x.view(torch.int32), rows.view(torch.int32))
    weight = torch.exp(part_ml[..., :1].double() - part_ml[..., :1].double().amax(2, keepdim=True))
    below = (part_ml[..., 1:].double() * weight).sum(2)
    want, size = (((v * weight).sum(2) / below).view(T, H * hd) for v in (part_o.double(), part_o.double().abs()))
    sure = torch.isfinite(want)                            # (an exponential off by two places, a rounding or two a run)
    assert bool(((got.x.double() - want).abs()[sure] <= (2 * runs + 8) * 2.0 ** -23 * size[sure]).all())
    planes, info = K.pair_rows(got.x)
    assert torch.equal(got.info, info)
    finite = info[:, 1].cpu() >= 0
    assert torch.equal(got.planes.view(torch.int32).view(T, -1)[finite], planes.view(torch.int32).view(T, -1)[finite])
    for bad in (lambda: K.merge_pair_rows(part_o.view(-1)[:-8], part_ml.view(-1), got.x, H, hd, runs),
                lambda: K.merge_pair_rows(part_o.view(-1), part_ml.view(-1), got.x[:, :-8].contiguous(), H, hd, runs)):
        with pytest.raises(K.KernelError):
            bad()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,d", [(9, 4), (9, 252), (9, 260), (1024, 2048), (1025, 2048), (3, 2052), (3, 4096), (3, 4100)])
def test_a_norm_on_both_sides_of_a_vector_a_thread(K, dtype, T, d):
    """Against 64 bits: a sum of d squares (at most d + 2 roundings), the root and the division, two products, and one rounding to the type."""
    g = torch.Generator().manual_seed(T + d)
    h, w, parts = torch.randn(T, d, generator=g), torch.randn(d, generator=g), torch.randn(5, T, d, generator=g)
    hd = h.cuda()
    out = K.add_rmsnorm(hd, parts.cuda(), w.cuda(), 1e-5, torch.empty(T, d, device="cuda", dtype=dtype))
    stream = h
    for p in parts:
        stream = stream + p                                    # in their order
    assert torch.equal(hd.cpu(), stream)
    want = stream.double() * ((stream.double() ** 2).mean(1, keepdim=True) + 1e-5).rsqrt() * w.double()
    off = ((d + 2) / 2 + 5) * 2.0 ** -24 + (2.0 ** -8 if dtype == torch.bfloat16 else 0.0)
    assert bool(((out.cpu().double() - want).abs() <= off * want.abs() + 1e-30).all())
