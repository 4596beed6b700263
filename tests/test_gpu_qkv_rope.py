"""The products of many bfloat16 rows that rotate queries and keys and store keys and values in their epilogue, against the product
and the rotating kernel one behind the other."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    from nanoinfer_amd import kernels
    return kernels


# rows at the edges of tiles; heads whose halves are one, two and four blocks of a wavefront's columns; a last tile of columns that is not
# whole; slots that are left out, and none at all
@pytest.mark.parametrize("plan", [(True, 0), (True, 1), (True, 2), (False, 0), (False, 1), (False, 2), (False, 3)])
@pytest.mark.parametrize("M,Kd,H,KVH,hd,page", [(65, 64, 1, 1, 64, 16), (129, 128, 6, 2, 64, 5), (300, 192, 3, 1, 128, 16), (257, 320, 2, 1, 192, 7),
                                                (1100, 128, 4, 4, 64, 16), (200, 64, 5, 5, 32, 16)])
def test_rotated_and_stored_as_by_the_kernel_behind_the_product(K, plan, M, Kd, H, KVH, hd, page):
    if not plan[0] and hd % 64:
        pytest.skip("on the stored matrix: heads of whole 64")
    g = torch.Generator().manual_seed(M + hd)
    N = (H + 2 * KVH) * hd
    x, w = torch.randn(M, Kd, generator=g).bfloat16().cuda(), torch.randn(N, Kd, generator=g).bfloat16().cuda()
    weight = K.Weight(w)
    angle = torch.rand(2000, hd // 2, generator=g) * 6.28
    cos, sin = angle.cos().cuda(), angle.sin().cuda()
    positions = torch.randint(0, 2000, (M,), generator=g, dtype=torch.int32).cuda()
    pages = M // page + 3
    slots = torch.randperm(pages * page, generator=g)[:M].to(torch.int32)
    slots[3] = -1
    slots = slots.cuda()
    sums = x.double() @ w.double().t()
    size = (x.double().abs() @ w.double().abs().t()).view(M, H + 2 * KVH, 2, hd // 2)
    heads = sums.view(M, H + 2 * KVH, 2, hd // 2)
    c, s = cos.double()[positions.long()][:, None], sin.double()[positions.long()][:, None]
    turned = torch.stack((heads[:, :, 0] * c - heads[:, :, 1] * s, heads[:, :, 0] * s + heads[:, :, 1] * c), dim=2)
    want = torch.cat((turned[:, :H + KVH], heads[:, H + KVH:]), dim=1).reshape(M, H + 2 * KVH, hd)
    # K roundings of a sum, three of the rotation, one to bfloat16
    off = ((Kd + 12) * 2.0 ** -24 * size.sum(2, keepdim=True).expand_as(size)).reshape(M, H + 2 * KVH, hd) + 2.0 ** -8 * want.abs()
    kept = slots >= 0
    at = slots[kept].long()

    def check(q, kpool, vpool):
        assert bool(((q.double().view(M, H, hd) - want[:, :H]).abs() <= off[:, :H]).all())
        for pool, first in ((kpool, H), (vpool, H + KVH)):
            got = pool.permute(0, 2, 1, 3).reshape(-1, KVH, hd)[at].double()
            assert bool(((got - want[kept, first:first + KVH]).abs() <= off[kept, first:first + KVH]).all())
            untouched = torch.ones(pages * page, dtype=torch.bool, device="cuda")
            untouched[at] = False
            assert bool((pool.permute(0, 2, 1, 3).reshape(-1, KVH, hd)[untouched] == 7.0).all())

    kpool, vpool = (torch.full((pages, KVH, page, hd), 7.0, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    q = K.qkv_rope(x, weight, positions, cos, sin, slots, kpool, vpool, H, KVH, hd, plan)
    check(q, kpool, vpool)
    assert torch.equal(K.qkv_rope(x, weight, positions, cos, sin, None, None, None, H, KVH, hd, plan), q)
    # the product and the kernel behind it: its rows are rounded before they are rotated (2^-9 of a pair's two), both results are rounded (2^-9 each of
    # no more than the pair's two), and the sums' order may be another
    pools = [torch.full((pages, KVH, page, hd), 7.0, device="cuda", dtype=torch.bfloat16) for _ in range(2)]
    behind = K.wide_gemm(x, w)
    K.rope_kv_write(behind, positions, cos, sin, slots, *pools, H, KVH, hd)
    pair = heads.abs().sum(2, keepdim=True).expand_as(heads).reshape(M, H + 2 * KVH, hd)
    apart = 2 * (off - 2.0 ** -8 * want.abs()) + 2.0 ** -7 * pair
    assert bool(((behind[:, :H * hd].double().view(M, H, hd) - q.double().view(M, H, hd)).abs() <= apart[:, :H]).all())
    for one, other, first in ((kpool, pools[0], H), (vpool, pools[1], H + KVH)):
        one, other = (t.permute(0, 2, 1, 3).reshape(-1, KVH, hd) for t in (one, other))
        assert bool(((one[at].double() - other[at].double()).abs() <= apart[kept, first:first + KVH]).all())
        untouched = torch.ones(pages * page, dtype=torch.bool, device="cuda")
        untouched[at] = False
        assert torch.equal(one[untouched], other[untouched])


def test_what_it_does_not_take(K):
    x, weight = torch.zeros(100, 64, device="cuda", dtype=torch.bfloat16), K.Weight(torch.zeros(3 * 96, 64, device="cuda", dtype=torch.bfloat16))
    pos, half = torch.zeros(100, device="cuda", dtype=torch.int32), torch.zeros(8, 48, device="cuda")
    K.qkv_rope(x, weight, pos, half, half, None, None, None, 1, 1, 96, (True, 2))
    pool = torch.zeros(8, 1, 16, 96, device="cuda", dtype=torch.bfloat16)
    for bad in (lambda: K.qkv_rope(x, weight, pos, half, half, None, None, None, 1, 1, 96, (False, 3)),                # heads of 96 on the stored matrix
                lambda: K.qkv_rope(x, weight, pos, half[:, :32].contiguous(), half[:, :32].contiguous(), None, None, None, 1, 1, 96, (True, 2)),
                lambda: K.qkv_rope(x, weight, pos, half, half, None, None, None, 2, 1, 96, (True, 2)),
                lambda: K.qkv_rope(x, weight, pos, half, half, pos, pool, None, 1, 1, 96, (True, 2)),
                lambda: K.qkv_rope(x, weight, pos, half, half, pos, pool.float(), pool, 1, 1, 96, (True, 2)),
                lambda: K.qkv_rope(x, weight, pos, half, half, None, None, None, 1, 1, 96, (True, 3))):
        with pytest.raises(K.KernelError):
            bad()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,S,H,KVH,hd,rot,page", [(1, 1, 1, 1, 64, 64, 16), (67, 2, 6, 2, 64, 64, 5), (130, 3, 3, 1, 80, 48, 16), (70, 4, 2, 2, 20, 8, 16), (65, 2, 4, 2, 64, 0, 7), (66, 6, 2, 1, 64, 64, 16)])
def test_the_shares_of_a_cut_product_added_rotated_and_stored(K, dtype, T, S, H, KVH, hd, rot, page):
    """In float32 bit for bit what adding them in their order and the rotating kernel make."""
    g = torch.Generator().manual_seed(T + hd)
    parts = torch.randn(S, T, (H + 2 * KVH) * hd, generator=g).cuda()
    cos = sin = None
    if rot:
        angle = torch.rand(300, rot // 2, generator=g) * 6.28
        cos, sin = angle.cos().cuda(), angle.sin().cuda()
    positions = torch.randint(0, 300, (T,), generator=g, dtype=torch.int32).cuda()
    pages = T // page + 3
    slots = torch.randperm(pages * page, generator=g)[:T].to(torch.int32)
    slots[T // 2] = -1
    slots = slots.cuda()
    pools = [torch.full((pages, KVH, page, hd), 7.0, device="cuda", dtype=dtype) for _ in range(2)]
    q = K.rope_kv_write_shares(parts, positions, cos, sin, slots, *pools, H, KVH, hd, dtype)
    whole = parts[0].clone()
    for p in range(1, S):
        whole += parts[p]
    want = [torch.full((pages, KVH, page, hd), 7.0, device="cuda") for _ in range(2)]
    K.rope_kv_write(whole, positions, cos, sin, slots, *want, H, KVH, hd)
    for got, true in ((q, whole[:, :H * hd].contiguous()), *zip(pools, want)):
        assert torch.equal(got, true.to(dtype))                # both round to nearest
    assert torch.equal(K.rope_kv_write_shares(parts, positions, cos, sin, None, None, None, H, KVH, hd, dtype), q)
    for bad in (lambda: K.rope_kv_write_shares(parts[:, :, :-4], positions, cos, sin, None, None, None, H, KVH, hd, dtype),
                lambda: K.rope_kv_write_shares(parts, positions, cos, sin, slots, pools[0], None, H, KVH, hd, dtype)):
        with pytest.raises(K.KernelError):
            bad()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("S", [5, 8, 10, 12, 13])
def test_as_many_shares_as_plans_have(K, dtype, S):
    """The numbers of shares that are compiled and their neighbours, whose places in a sum differ by bits where one is left out or taken twice."""
    T, H, KVH, hd = 70, 3, 1, 64
    g = torch.Generator().manual_seed(S)
    parts, angle = torch.randn(S, T, (H + 2 * KVH) * hd, generator=g).cuda(), torch.rand(T, hd // 2, generator=g) * 6.28
    cos, sin, at = angle.cos().cuda(), angle.sin().cuda(), torch.arange(T, dtype=torch.int32).cuda()
    pools, want = ([torch.zeros(5, KVH, 16, hd, device="cuda", dtype=t) for _ in range(2)] for t in (dtype, torch.float32))
    q = K.rope_kv_write_shares(parts, at, cos, sin, at, *pools, H, KVH, hd, dtype)
    whole = parts[0].clone()
    for p in range(1, S):
        whole += parts[p]
    K.rope_kv_write(whole, at, cos, sin, at, *want, H, KVH, hd)
    for got, true in ((q, whole[:, :H * hd].contiguous()), *zip(pools, want)):
        assert torch.equal(got, true.to(dtype))


def off_vectors(t):
    """The same numbers four bytes behind a multiple of sixteen, as a view into a program's own buffer may stand."""
    by = 4 // t.element_size()
    flat = torch.zeros(t.numel() + by, dtype=t.dtype, device=t.device)
    flat[by:] = t.reshape(-1)
    return flat[by:].view(t.shape)


@pytest.mark.parametrize("pools_off,tables_off", [(True, False), (False, True), (True, True)])
@pytest.mark.parametrize("kind", ["tiled", "stored", "shares", "shares float32"])
def test_pools_and_tables_off_sixteen_bytes(K, kind, pools_off, tables_off):
    """They were taken by the rotating kernel behind a product, and are by what stands in its place; queries are the same, keys and values up to the one
    rounding more of a kernel behind rounded rows."""
    M, Kd, H, KVH, hd = 300, 256, 3, 1, 64
    dtype = torch.float32 if "float32" in kind else torch.bfloat16
    g = torch.Generator().manual_seed(3)
    x, w = torch.randn(M, Kd, generator=g).bfloat16().cuda(), torch.randn((H + 2 * KVH) * hd, Kd, generator=g).bfloat16().cuda()
    parts, angle = torch.randn(3, M, (H + 2 * KVH) * hd, generator=g).cuda(), torch.rand(M, hd // 2, generator=g) * 6.28
    tables, at = (angle.cos().cuda(), angle.sin().cuda()), torch.arange(M, dtype=torch.int32).cuda()
    at[5] = -1
    made = []
    for off in (False, True):
        pools = [torch.full((20, KVH, 16, hd), 7.0, device="cuda", dtype=dtype) for _ in range(2)]
        cos, sin = (off_vectors(t) for t in tables) if off and tables_off else tables
        pools = [off_vectors(p) for p in pools] if off and pools_off else pools
        positions = torch.arange(M, dtype=torch.int32).cuda()
        if kind.startswith("shares"):
            q = K.rope_kv_write_shares(parts, positions, cos, sin, at, *pools, H, KVH, hd, dtype)
        else:
            q = K.qkv_rope(x, K.Weight(w), positions, cos, sin, at, *pools, H, KVH, hd, (kind == "tiled", 2 if kind == "tiled" else 3))
        made.append((q, *pools))
    for one, other in zip(*made):
        if kind.startswith("shares"):
            # a c - b s with either product inside the sum's rounding: apart by at most 2^-23 (|a c| + |b s|) <= 2^-22 of the row's largest, as the rotation
            # leaves a pair's length; in bfloat16 the rounded row is rotated (2^-8 of it), and the result rounded once more
            off = 2.0 ** -22 if dtype == torch.float32 else 2.0 ** -6
            assert bool(((one.float() - other.float()).abs() <= off * one.float().abs().amax(-1, keepdim=True)).all())
        else:
            assert torch.equal(one, other)


@pytest.mark.parametrize("M,H,KVH,hd,Kd,way", [(320, 32, 8, 128, 4096, "whole"), (352, 32, 8, 128, 4096, "shares"), (257, 16, 8, 64, 2048, "inside"), (256, 16, 8, 64, 2048, "shares")])
def test_whichever_way_a_layer_takes_rounds_once(K, M, H, KVH, hd, Kd, way):
    """Past 64 rows a layer's queries, keys and values are sums in float32, rotated, and rounded once, by the epilogue as by the pass behind a product."""
    from types import SimpleNamespace

    from nanoinfer_amd.parts.standard import Attention
    g = torch.Generator().manual_seed(M)
    x, w = torch.randn(M, Kd, generator=g).bfloat16().cuda(), (torch.randn((H + 2 * KVH) * hd, Kd, generator=g) * Kd ** -0.5).bfloat16().cuda()
    weight, angle = K.Weight(w), torch.rand(M, hd // 2, generator=g) * 6.28
    cos, sin, at = angle.cos().cuda(), angle.sin().cuda(), torch.arange(M, dtype=torch.int32).cuda()
    assert ("inside" if K.qkv_rope_plan(x, weight, hd, hd) else "whole" if K.qkv_whole(x, weight) else "shares") == way
    part = Attention.__new__(Attention)
    part.H, part.KVH, part.hd, part.w_qkv, part.position = H, KVH, hd, weight, SimpleNamespace(tables=lambda: (cos, sin))
    pools = [torch.zeros(M // 16 + 1, KVH, 16, hd, device="cuda", dtype=torch.bfloat16) for _ in range(2)]
    cache = SimpleNamespace(writes=True, slot_mapping=at, kpool=pools[0], vpool=pools[1])
    q = part._project_many(x, SimpleNamespace(positions=at), cache)
    sums, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    heads, c, s = sums.view(M, H + 2 * KVH, 2, hd // 2), cos.double()[:, None], sin.double()[:, None]
    turned = torch.stack((heads[:, :, 0] * c - heads[:, :, 1] * s, heads[:, :, 0] * s + heads[:, :, 1] * c), dim=2)
    want = torch.cat((turned[:, :H + KVH], heads[:, H + KVH:]), dim=1).reshape(M, H + 2 * KVH, hd)
    got = torch.cat((q.view(M, H, hd), *(p.permute(0, 2, 1, 3).reshape(-1, KVH, hd)[:M] for p in pools)), dim=1).double()
    # K roundings of a sum and three of the rotation in float32, one to bfloat16
    off = (Kd + 12) * 2.0 ** -24 * size.view(M, H + 2 * KVH, 2, hd // 2).sum(2, keepdim=True).expand(-1, -1, 2, -1).reshape(M, H + 2 * KVH, hd) + 2.0 ** -8 * want.abs()
    assert bool(((got - want).abs() <= off).all())


@pytest.mark.parametrize("M", [257, 320, 400, 512])
def test_float32_results_of_the_library_recorded(K, M):
    """The library's product with float32 results and the pass behind it in a graph: every replay, with other work between, is what they give launched."""
    H, KVH, hd, Kd = 32, 8, 128, 4096
    g = torch.Generator().manual_seed(M)
    x, w = torch.randn(M, Kd, generator=g).bfloat16().cuda(), K.Weight((torch.randn((H + 2 * KVH) * hd, Kd, generator=g) * Kd ** -0.5).bfloat16().cuda())
    angle, at = torch.rand(M, hd // 2, generator=g) * 6.28, torch.arange(M, dtype=torch.int32).cuda()
    cos, sin = angle.cos().cuda(), angle.sin().cuda()
    pools = [torch.zeros(M // 16 + 1, KVH, 16, hd, device="cuda", dtype=torch.bfloat16) for _ in range(2)]

    def run():
        return K.rope_kv_write_shares(K.linear(x, w, torch.float32).unsqueeze(0), at, cos, sin, at, *pools, H, KVH, hd, torch.bfloat16)

    def stored():
        return [p.permute(0, 2, 1, 3).reshape(-1, KVH, hd)[:M].clone() for p in pools]

    assert K.qkv_whole(x, w)
    want = [run(), *stored()]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        q = run()
    for turn in range(4):
        for t in (q, *pools):
            t.fill_(float(turn))
        K.linear(x, w)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for got, true in zip((q, *stored()), want):
            assert torch.equal(got, true)
