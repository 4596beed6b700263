"""The rules by which a product goes to a kernel here or to the library, without a GPU."""
import pytest
import torch

from nanoinfer_amd import kernels as K


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M", [1, 20, 64, 65, 100, 512, 1000])
@pytest.mark.parametrize("N,Kd", [(64, 0), (0, 64)])
def test_products_over_nothing_are_the_librarys(dtype, M, N, Kd):
    """No kernel here takes rows of no elements (it would read the last piece of a row that has none) or none of them."""
    x, weight = torch.empty(M, Kd, dtype=dtype), K.Weight(torch.empty(N, Kd, dtype=dtype))
    if Kd == 0:
        assert not K.skinny_ok(M, Kd, dtype) and not K.skinny_wins(M, Kd, dtype, weight) and not K.skinny_deals(M, N, Kd, dtype, weight)
    assert not K.tiled_wins(x, weight) and not K.tiled_wins(x, weight, gated=True) and not K.split_wins(x, weight.rows)


def test_what_the_tiled_product_cannot_address_is_the_librarys():
    """Bytes of x and of W are counted in 32 bits: what tiled_gemm refuses, the rule does not send there."""
    class Stored:                                      # a matrix that is only looked at
        tiles = torch.empty(0)

        def __init__(self, N, Kd):
            self.rows = torch.empty(N, Kd, dtype=torch.bfloat16, device="meta")

    for M, N, Kd in ((1024, 32, 1 << 20), (512, 4, 1 << 21), (65, 1 << 14, 1 << 16)):
        x = torch.empty(M, Kd, dtype=torch.bfloat16, device="meta")
        assert not K.tiled_wins(x, Stored(N, Kd)) and not K.tiled_wins(x, Stored(N, Kd), gated=True)


def test_a_plan_is_made_once_for_64_rows():
    """Steps of every number of rows weigh the tiles and shares of a product eight times up to 512 rows, not 448 times."""
    from nanoinfer_amd.kernels import tile
    for plan, made in ((K.tiled_plan, tile._tiled_plan), (K.split_plan, tile._split_plan), (lambda M, N, Kd: tile._grouped_plan(M, N, Kd, 7), tile._grouped_tiles)):
        before = made.cache_info().misses
        plans = [plan(M, 3075, 2047) for M in range(65, 513)]
        assert made.cache_info().misses - before <= 8
        assert plans[0] == plan(128, 3075, 2047) and plans[-1] == plan(449, 3075, 2047)


@pytest.mark.parametrize("N,Kd,kind,here,there", [
    (2048, 2048, "addends", (65, 512), (64, 513)), (4096, 14336, "addends", (65, 512), (513,)),      # shares left to the norm
    (4096, 14336, "plain", (65, 320, 512), (513,)), (3072, 8192, "plain", (65, 356), (505, 512)),     # cut along K, or not often enough
    (3072, 2048, "plain", (65, 300, 512), (513,)), (6144, 4096, "plain", (65, 256), (257, 320, 512)),
    (16384, 2048, "gated", (65, 320, 512), (513, 640, 1024)), (16384, 3072, "gated", (65, 256, 512), (320, 384, 600)),
    (28672, 4096, "gated", (65, 128), (129, 192, 512, 1024)), (4096, 2048, "gated", (65, 512, 600, 1024), (1025,)),
    (8192, 2048, "gated", (512,), (701, 767))])
def test_where_bfloat16_products_of_many_rows_go(N, Kd, kind, here, there):
    """Both sides of the lines that the rule draws, at the sizes measured beside it; the plan is one that the kernel takes."""
    class Stored:
        tiles = torch.empty(0)
        rows = torch.empty(N, Kd, dtype=torch.bfloat16, device="meta")

    more = {kind: True} if kind != "plain" else {}
    for M in here + there:
        x = torch.empty(M, Kd, dtype=torch.bfloat16, device="meta")
        assert K.tiled_wins(x, Stored(), **more) == (M in here), M
        tile, shares = K.tiled_plan(M, N, Kd, kind == "gated", kind == "addends")
        assert 0 <= tile < (3 if kind == "gated" else 4) and 1 <= shares <= (1 if kind == "gated" else 8) and (shares == 1 or Kd // shares >= 256)


@pytest.mark.parametrize("N,Kd,gated,here,there", [
    (16384, 2048, True, (400, 512, 900, 1024, 1999, 4096), (256, 600)), (4096, 2048, True, (600, 1024, 1999), (512,)),
    (2048, 8192, False, (1600, 1999, 2048), (512, 1024, 2049)), (2048, 2048, False, (1024, 1600, 1999), (512, 640, 2049)),
    (3072, 2048, False, (1024, 1999), (512, 1300, 1600, 3000)), (2040, 2048, False, (), (1999,)), (2048, 2080, False, (), (1999,)),
    (16, 1 << 27, False, (), (1024,)), (1 << 25, 64, True, (), (1024,))])
def test_where_bfloat16_products_of_many_rows_on_the_stored_matrix_go(N, Kd, gated, here, there):
    """Both sides of the lines; what the kernel refuses (columns that are no whole vectors, bytes past 31 bits) the rule does not send there."""
    rows = torch.empty(N, Kd, dtype=torch.bfloat16, device="meta")
    for M in here + there:
        assert K.wide_wins(torch.empty(M, Kd, dtype=torch.bfloat16, device="meta"), rows, gated) == (M in here), M
    x = torch.empty(1024, Kd, device="meta")
    assert not K.wide_wins(x, rows, gated) and not K.wide_wins(x, rows.float(), gated)
    if Kd < 1 << 20:
        assert not K.wide_wins(torch.empty(Kd, 1024, dtype=torch.bfloat16, device="meta").t(), rows, gated)


@pytest.mark.parametrize("N,Kd,to,here,there", [
    (5120, 3072, "bfloat16", (600, 1200), (1024,)), (5120, 3072, "float32", (600,), (1024,)), (5120, 3072, "epilogue", (600, 1024, 1200), ()),
    (8192, 4096, "bfloat16", (1024,), (700, 2048)), (4096, 14336, "bfloat16", (1700, 2048), (900, 1300, 1400)), (4096, 14336, "epilogue", (900, 1300, 2048), ()),
    (8192, 2048, "bfloat16", (1024,), (2048,)), (8192, 2048, "float32", (2048,), (700,)), (2048, 2048, "float32", (1300, 2048), ()),
    (16384, 3072, "gated", (350, 400, 512), (300,)), (16384, 2048, "gated", (300, 350, 512), ())])
def test_no_products_on_the_stored_matrix_where_the_librarys_are_faster(N, Kd, to, here, there):
    """By where the results go: beside the sizes above, those where a product here was measured to take 3 to 15 % longer."""
    rows = torch.empty(N, Kd, dtype=torch.bfloat16, device="meta")
    for M in here + there:
        assert K.wide_takes(M, Kd, rows, True) == (M in here) if to == "gated" else K.wide_takes(M, Kd, rows, to=to) == (M in here), M


@pytest.mark.parametrize("N,Kd,M,adds,leaves", [(2048, 2048, 1999, True, True), (2048, 8192, 1999, True, True), (2048, 2048, 1100, True, True), (2048, 8192, 1100, False, False),
                                                (2048, 2048, 512, False, False), (2048, 2048, 2049, False, False), (4160, 2048, 1200, True, False), (3136, 4096, 1024, True, False), (2064, 2048, 1999, False, False)])
def test_which_products_go_onto_the_stream_in_their_epilogue(N, Kd, M, adds, leaves):
    """Those that go to the product on the stored matrix at all; sums of squares are left in whole vectors of parts of 64 columns, at most 64."""
    class Stored:
        tiles = torch.empty(0)
        rows = torch.empty(N, Kd, dtype=torch.bfloat16, device="meta")

    assert K.wide_stream_ok(M, Kd, torch.bfloat16, Stored()) == adds and K.wide_leaves_ok(M, Kd, torch.bfloat16, Stored()) == leaves
    assert not K.wide_stream_ok(M, Kd, torch.float32, Stored()) and not K.wide_stream_ok(M, Kd, torch.bfloat16, Stored.rows)


@pytest.mark.parametrize("N,Kd,hd,here,there", [(3072, 2048, 64, (600, 1024, 1300, 1999, 2500, 4096), ()), (5120, 3072, 128, (600, 800, 1024, 1500, 2500), (1600, 1664)),
                                                (6144, 4096, 128, (600, 1024, 1200, 2500), (1300, 1400, 3000)), (3072, 2048, 96, (), (1999,))])
def test_where_products_of_many_rows_rotate_and_store(N, Kd, hd, here, there):
    """Both sides of the line at the sizes measured beside it."""
    class Stored:
        tiles = None
        rows = torch.empty(N, Kd, dtype=torch.bfloat16, device="meta")

    for M in here + there:
        plan = K.qkv_rope_plan(torch.empty(M, Kd, dtype=torch.bfloat16, device="meta"), Stored(), hd, hd)
        assert plan == K.wide_rope_plan(M, Kd, torch.bfloat16, Stored(), hd, hd) and (plan is not None) == (M in here), M


@pytest.mark.parametrize("N,Kd,hd,whole,shares,inside", [(5120, 3072, 128, (), (65, 256, 300, 384), (400, 512)), (6144, 4096, 128, (300, 400, 512), (65, 256, 352, 384), ()),
                                                         (3072, 2048, 64, (), (65, 192, 224, 320), (352, 512)), (2048, 2048, 64, (), (65, 256), (257, 300, 384, 512)),
                                                         (2560, 2048, 128, (), (65, 256, 300, 384), (400, 512)), (1536, 1024, 64, (), (65, 128), (160, 512))])
def test_where_stacked_products_of_65_to_512_rows_rotate_and_store(N, Kd, hd, whole, shares, inside):
    """In the epilogue, in the pass that adds a cut product's shares, or in that pass over float32 results: the fastest of those, which all round once."""
    class Stored:
        tiles = torch.empty(0)
        rows = torch.empty(N, Kd, dtype=torch.bfloat16, device="meta")

    for M in whole + shares + inside:
        x = torch.empty(M, Kd, dtype=torch.bfloat16, device="meta")
        assert (K.qkv_rope_plan(x, Stored(), hd, hd) is not None) == (M in inside), M
        assert M in inside or K.qkv_whole(x, Stored()) == (M in whole), M
    assert not K.qkv_whole(x, Stored.rows) and not K.qkv_whole(torch.empty(300, Kd), Stored()) and not K.qkv_whole(x[:, :32], Stored())


@pytest.mark.parametrize("stage", ["forward", "output"])
def test_a_replaced_stage_of_attention_is_given_no_stream_of_many_rows(stage):
    """Past the skinny products' rows a class that has its own ``forward`` or ``output``, which may know of no ``residual``, is run without one."""
    from types import SimpleNamespace

    from nanoinfer_amd.parts.standard import Attention

    def part(cls):
        p = cls.__new__(cls)
        p.H, p.hd, p.rt = 32, 64, SimpleNamespace(dtype=torch.bfloat16)
        p.w_o = SimpleNamespace(tiles=None, rows=torch.empty(2048, 2048, dtype=torch.bfloat16, device="meta"))
        return p

    assert part(Attention).adds_residual(1999) and part(Attention).leaves_scaled(1999)
    own = part(type("Own", (Attention,), {stage: lambda self, x, ctx, cache: x}))
    assert not own.adds_residual(1999) and not own.leaves_scaled(1999)


def test_a_norm_whose_input_a_product_cannot_leave_is_ignored(monkeypatch):
    """As with few rows: 4,160 columns are 65 parts of sums of squares, more than the product behind takes; the sum onto the stream goes out alone."""
    went = []
    monkeypatch.setattr(K, "wide_stream", lambda *a, **k: went.append((len(a), k)) or (None, None))
    x, w, h = torch.empty(1200, 2048, dtype=torch.bfloat16), K.Weight(torch.empty(4160, 2048, dtype=torch.bfloat16), tiled=False), torch.empty(1200, 4160)
    assert K.linear(x, w, residual=h, leave=K.NormSpec(torch.empty(4160), 1e-5)) is None and went == [(3, {})]
    for bad in (x.view(1, 1200, 2048).expand(65, 1200, 2048), x[:, :64]):
        with pytest.raises(K.KernelError):
            K.linear(bad, w, residual=h)


def test_float32_steps_ask_nothing_that_is_for_bfloat16(monkeypatch):
    """A step of more than 64 float32 tokens is launched kernel by kernel by a host that takes longer than they do: what its type decides it asks no rule."""
    from types import SimpleNamespace

    from nanoinfer_amd.parts.standard import Attention, SwiGLU

    for name in ("wide_stream_ok", "wide_rope_plan", "wide_leaves_ok", "wide_takes", "swiglu_takes_scaled"):
        monkeypatch.setattr(K, name, lambda *a, **k: pytest.fail("asked"))
    w = SimpleNamespace(rows=torch.empty(192, 192), shape=(192, 192), tiles=None)
    for cls in (Attention, SwiGLU):
        part = cls.__new__(cls)
        part.rt, part.H, part.hd, part.intermediate_size = SimpleNamespace(dtype=torch.float32), 6, 32, 192
        part.w_o = part.w_qkv = part.w_gate_up = part.w_down = w
        part.position = SimpleNamespace(tables=lambda: pytest.fail("asked"))
        assert not part.adds_residual(100) and not part.takes_scaled(100) and not part.leaves_scaled(100)


def test_squares_are_of_sums_that_were_not_rounded(monkeypatch):
    """The product whose epilogue squares goes by the line of those, not by a plain one's, whose rounded results a kernel would square."""
    monkeypatch.setattr(K, "wide_gemm", lambda x, rows, **k: k)
    x, w = torch.empty(1024, 3072, dtype=torch.bfloat16), K.Weight(torch.empty(5120, 3072, dtype=torch.bfloat16), tiled=False)
    assert not K.wide_wins(x, w.rows) and K.wide_wins(x, w.rows, to="epilogue")
    assert K.linear_relu2(x, w) == {"squared": True}
