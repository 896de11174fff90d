"""Expert products on the matrix cores where their tiles can go wrong: rows an expert from none to one past a tile, one and
many stages, output blocks that end early -- against fp32 products of the same bf16 operands."""
import pytest
import torch

from kubernetes_cloud_amd.ops import moe

pytestmark = pytest.mark.gpu
# the activation and the result are rounded to bf16 once each (2^-9), the products are summed in fp32
TOL = 2.5 * 2.0 ** -9


def _case(counts, top, d, F, seed=0):
    """Ids with ``counts[e]`` rows of expert e, shuffled."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    flat = torch.cat([torch.full((c,), e) for e, c in enumerate(counts)])
    assert flat.numel() % top == 0
    ids = flat[torch.randperm(flat.numel(), generator=torch.Generator().manual_seed(seed))].view(-1, top).int().cuda()
    T, E = ids.shape[0], len(counts)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    return (r(T, d).bfloat16(), ids, torch.rand(T, top, device="cuda", generator=g), (r(E, 2 * F, d) * d ** -0.5).bfloat16(),
            (r(E, d, F) * F ** -0.5).bfloat16())


@pytest.mark.parametrize("mt", [moe.STREAM_ROWS, 128, 192, moe.GEMM_ROWS])
@pytest.mark.parametrize("scale_in", [True, False])
@pytest.mark.parametrize("counts,top,d,F", [([0, 1, 16, 17, 32, 33, 15], 2, 64, 64), ([31, 64, 65, 0, 8], 3, 320, 192),
                                            ([1], 1, 128, 64), ([129, 127, 256, 2], 2, 192, 320), ([65, 96, 97, 160, 161, 193, 257, 191], 4, 72, 200), ([40, 40], 4, 64, 576),
                                            ([193, 256, 225, 255, 512, 449], 2, 128, 192), ([449, 191, 200, 224], 4, 704, 320)])
def test_products(mt, scale_in, counts, top, d, F):
    if mt == moe.STREAM_ROWS and (d % 64 or F % 64):
        pytest.skip("the stream takes whole stages")
    h, ids, wts, gu, dn = _case(counts, top, d, F)
    g = moe.group(ids, len(counts), mt)
    y = moe.experts(h, ids, wts, gu, dn, g, scale_in)[g.inv.long()]
    e = ids.long()
    u = torch.einsum("td,tkfd->tkf", h.float(), gu.float()[e])
    w = wts[..., None]
    u = u * w if scale_in else u
    a = (torch.nn.functional.silu(u[..., :F]) * u[..., F:]).bfloat16().float()
    want = torch.einsum("tkf,tkdf->tkd", a, dn.float()[e]) * (1 if scale_in else w)
    assert (y.float() - want).norm() <= TOL * want.norm()


@pytest.mark.parametrize("d,F", [(64, 128), (192, 256), (320, 576), (1088, 64), (64, 1216)])
def test_stream_rows(d, F):
    """Every number of rows a tile's forms end at, with fewer stages of K than waves, one more, and a remainder of them; row by row."""
    counts = [1, 7, 8, 9, 15, 16, 0, 17, 31, 32, 33, 65, 2]
    h, ids, wts, gu, dn = _case(counts, 1, d, F)
    g = moe.group(ids, len(counts), moe.STREAM_ROWS)
    y = moe.experts(h, ids, wts, gu, dn, g, False)[g.inv.view(-1).long()].float()
    e = ids.view(-1).long()
    u = torch.bmm(gu.float()[e], h.float()[:, :, None])[..., 0]
    a = (torch.nn.functional.silu(u[:, :F]) * u[:, F:]).bfloat16().float()
    want = torch.bmm(dn.float()[e], a[..., None])[..., 0] * wts
    assert ((y - want).norm(dim=1) <= 2 * TOL * want.norm(dim=1)).all()  # (a row has few outputs: twice the whole's bound)


@pytest.mark.parametrize("counts,mt", [([64, 65, 1, 0, 128, 320, 321], 128), ([257, 288, 289, 40, 513, 256, 130], 256), ([5, 70] * 40, 128), ([3] * 70, 192)])
def test_short_tiles_run_last(counts, mt):
    """Tiles that are alone and at most half full stand behind the rest; every row has one tile, and the products are right."""
    h, ids, wts, gu, dn = _case(counts, 1, 64, 64)
    g = moe.group(ids, len(counts), mt)
    tiles = g.tiles[:int(g.ntiles)].tolist()
    late = [t[4] == 1 and 2 * t[2] <= mt for t in tiles]
    assert late == sorted(late)
    for i, (e, at, rows, first, n) in enumerate(tiles):
        assert 0 < rows <= mt and first <= i < first + n and all(t[0] == e and t[3:] == [first, n] for t in tiles[first:first + n])
    rows = sorted((t[0], t[1] + j) for t in tiles for j in range(t[2]))
    assert rows == [(e, sum(counts[:e]) + j) for e, c in enumerate(counts) for j in range(c)]
    y = moe.experts(h, ids, wts, gu, dn, g, False)[g.inv.view(-1).long()]
    u = torch.bmm(gu.float()[ids.view(-1).long()], h.float()[:, :, None])[..., 0]
    a = (torch.nn.functional.silu(u[:, :64]) * u[:, 64:]).bfloat16().float()
    want = torch.bmm(dn.float()[ids.view(-1).long()], a[..., None])[..., 0] * wts
    assert (y.float() - want).norm() <= TOL * want.norm()


@pytest.mark.parametrize("counts,d,F", [([250, 64, 577, 1, 0, 129, 300, 65], 128, 320), ([70, 300, 10, 150] * 18, 64, 640), ([130] * 9 + [769, 513], 192, 1152),
                                        ([257, 320, 63], 1088, 64)])
def test_wide_tiles(counts, d, F):
    """Rows of an expert in even tiles, largest first; blocks of all four sizes, fewer than a round, several rounds, 1, 2, 3 and 17 stages, weight
    rows that end within a block."""
    h, ids, wts, gu, dn = _case(counts, 1, d, F)
    g = moe.group(ids, len(counts), moe.GEMM_ROWS)
    tiles = g.tiles[:int(g.ntiles)].tolist()
    for e, c in enumerate(counts):
        units = [-(-t[2] // 64) for t in tiles if t[0] == e]
        assert sum(t[2] for t in tiles if t[0] == e) == c and len(units) == -(-c // 256) and sum(units) == -(-c // 64)
        assert not units or max(units) - min(units) <= 1
    most = [-(-tiles[t[3]][2] // 64) for t in tiles]
    assert most == sorted(most, reverse=True)
    for scale_in in (True, False):
        y = moe.experts(h, ids, wts, gu, dn, g, scale_in)[g.inv.view(-1).long()].float()
        want = torch.empty_like(y)
        for e in range(len(counts)):
            k = ids.view(-1) == e
            w = wts.view(-1)[k, None]
            u = h[k].float() @ gu[e].float().T * (w if scale_in else 1)
            a = (torch.nn.functional.silu(u[:, :F]) * u[:, F:]).bfloat16().float()
            want[k] = a @ dn[e].float().T * (1 if scale_in else w)
        assert (y - want).norm() <= TOL * want.norm()


@pytest.mark.parametrize("d,F,counts,kernels", [
    (64, 128, [1, 5, 8, 9, 16, 17, 31, 32, 33, 0, 64, 65], "bb"), (640, 576, [3, 4, 2, 0, 33, 2, 1], "bb"), (192, 64, [2, 1, 3], "bb"),
    (1088, 64, [3, 8, 1, 9, 2, 0, 33, 16], "sb"), (1152, 1088, [8, 9, 16, 17, 1, 0, 7, 12], "ss"), (512, 1216, [9, 5, 31, 8, 12, 7], "bs"), (1024, 8256, [8, 9, 7, 6, 5], "bs"),
    (1024, 8256, [8, 1, 7, 6, 5], "ss"), (2112, 1984, [0, 1, 8, 9, 16, 17, 32, 33, 40, 64], "ss")])
def test_stream_and_blocks(d, F, counts, kernels):
    """The two kernels of up to 32 rows a tile, which the rows of an expert and the length of the walk choose between; 1 to 33 stages, weight rows that
    end within a block of 128."""
    h, ids, wts, gu, dn = _case(counts, 1, d, F)
    g = moe.group(ids, len(counts), moe.STREAM_ROWS)
    for scale_in in (True, False):
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
            y = moe.experts(h, ids, wts, gu, dn, g, scale_in)
            torch.cuda.synchronize()
        names = [e.key for e in prof.key_averages() if "expert_" in e.key]
        for up, k in zip(("true", "false"), kernels):
            assert any(f"expert_{'block' if k == 'b' else 'stream'}_kernel<{up}>" in n for n in names), names
        y = y[g.inv.view(-1).long()].float()
        want = torch.empty_like(y)
        for e in range(len(counts)):
            k = ids.view(-1) == e
            w = wts.view(-1)[k, None]
            u = h[k].float() @ gu[e].float().T * (w if scale_in else 1)
            a = (torch.nn.functional.silu(u[:, :F]) * u[:, F:]).bfloat16().float()
            want[k] = a @ dn[e].float().T * (1 if scale_in else w)
        assert (y - want).norm() <= TOL * want.norm()


@pytest.mark.parametrize("tiles", [511, 512, 513, 577, 1088])
def test_many_wide_tiles(tiles):
    """Blocks count the tiles of each size 512 and 64 at a time; one size ends within the last of them, or all stand past the first 512."""
    few = [250, 64, 577, 1, 0, 129, 300]
    counts = few + [(tiles - sum(-(-c // 256) for c in few)) * 256 - 100]
    d, F = 64, 128
    h, ids, wts, gu, dn = _case(counts, 1, d, F)
    g = moe.group(ids, len(counts), moe.GEMM_ROWS)
    assert int(g.ntiles) == tiles
    y = moe.experts(h, ids, wts, gu, dn, g, False)[g.inv.view(-1).long()].float()
    for e in range(len(counts)):
        k = ids.view(-1) == e
        u = h[k].float() @ gu[e].float().T
        want = (torch.nn.functional.silu(u[:, :F]) * u[:, F:]).bfloat16().float() @ dn[e].float().T * wts.view(-1)[k, None]
        assert (y[k] - want).norm() <= TOL * want.norm() and torch.isfinite(y[k]).all()


@pytest.mark.parametrize("tiles", [65535, 65536, 66000])
def test_more_tiles_than_16_bits_count(tiles):
    """Tiles of up to 256 rows: the counts of a size are packed in 16 bits, up to as many."""
    few = [300, 64, 1, 0, 700]
    counts = few + [(tiles - len(few) - 1) * 256 - sum(few)]  # (a call's most tiles: experts and whole tiles)
    n = sum(counts)
    assert len(counts) + n // 256 == tiles
    ids = torch.cat([torch.full((c,), e, device="cuda", dtype=torch.int32) for e, c in enumerate(counts)])
    ids = ids[torch.randperm(n, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))][:, None]
    g = moe.group(ids, len(counts), moe.GEMM_ROWS)
    t = g.tiles[:int(g.ntiles)].long()
    assert len(t) == sum(-(-c // 256) for c in counts) and int(t[:, 2].min()) >= 1 and int(t[:, 2].max()) <= 256
    assert torch.bincount(t[:, 0], t[:, 2].double(), minlength=len(counts)).long().tolist() == counts
    t = t[t[:, 1].argsort()]  # the tiles' rows follow each other, by experts
    assert torch.equal(t[:, 1], t[:, 2].cumsum(0) - t[:, 2]) and (t[1:, 0] >= t[:-1, 0]).all()
    sorted_ids = ids.view(-1)[g.perm.long()]
    assert (sorted_ids[1:] >= sorted_ids[:-1]).all() and torch.equal(g.perm[g.inv.view(-1).long()].long(), torch.arange(n, device="cuda"))
    of = g.tiles[:int(g.ntiles)].long()
    first = of[:, 3]  # an expert's tiles stand together
    assert torch.equal(of[first, 0], of[:, 0]) and (torch.arange(len(of), device="cuda") - first < of[:, 4]).all()


def test_more_blocks_than_a_dimension_holds():
    """The stream's launch for 21900 tiles of 12288 outputs: 16.8 million blocks of 256 threads; the rows of the last ones."""
    T, F = 32 * 21900, 12288
    h, ids, wts, gu, dn = _case([T], 1, 64, F)
    g = moe.group(ids, 1, moe.STREAM_ROWS)
    y = moe.experts(h, ids, wts, gu, dn, g, False)
    for rows in (slice(0, 64), slice(T // 2, T // 2 + 64), slice(T - 64, T)):
        t = g.perm[rows].long()
        u = h[t].float() @ gu[0].float().T
        a = (torch.nn.functional.silu(u[:, :F]) * u[:, F:]).bfloat16().float()
        want = a @ dn[0].float().T * wts[t]
        assert (y[rows].float() - want).norm() <= TOL * want.norm()


def _far(T, d, F, E):
    """Sizes past the 32-bit offsets, and some tokens' outputs in fp32."""
    g = torch.Generator(device="cuda").manual_seed(1)
    r = lambda *s, std=1.0: torch.empty(s, device="cuda", dtype=torch.bfloat16).normal_(0, std, generator=g)  # noqa: E731
    h, gu, dn = r(T, d), r(E, 2 * F, d, std=d ** -0.5), r(E, d, F, std=F ** -0.5)
    ids = torch.randint(0, E, (T, 1), device="cuda", generator=g).int()
    wts = torch.rand(T, 1, device="cuda", generator=g)
    mt = moe.tile_rows(T, 1, E, d, F, torch.bfloat16)
    assert mt == 128
    groups = moe.group(ids, E, mt)
    y = moe.experts(h, ids, wts, gu, dn, groups, True)
    at = torch.cat([torch.arange(T)[:20], torch.arange(T)[-20:], torch.randint(0, T, (40,), generator=torch.Generator().manual_seed(2))]).cuda()
    got = y[groups.inv.view(-1)[at].long()].float()
    want = torch.empty_like(got)
    for e in range(E):
        k = ids[at, 0] == e
        u = (h[at[k]].float() @ gu[e].float().T) * wts[at[k]]
        want[k] = (torch.nn.functional.silu(u[:, :F]) * u[:, F:]).bfloat16().float() @ dn[e].float().T
    assert (got - want).norm() <= TOL * want.norm()


def test_activations_past_2_gib():
    _far(130960, 8200, 72, 4)


def test_expert_weights_past_4_gib():
    _far(40, 16384, 65536, 1)


@pytest.mark.parametrize("mt", [moe.STREAM_ROWS, 128])
def test_rows_off_16_bytes(mt):
    """Tokens or weights that 16-byte loads do not fit."""
    h, ids, wts, gu, dn = _case([20, 0, 33, 19], 2, 128, 192)
    g = moe.group(ids, 4, mt)
    want = moe.experts(h, ids, wts, gu, dn, g, True)

    def off(t):
        big = torch.empty(t.numel() + 8, device="cuda", dtype=t.dtype)
        return big[1:1 + t.numel()].view(t.shape).copy_(t)

    for args in ((off(h), gu, dn), (h, off(gu), dn), (h, gu, off(dn))):
        y = moe.experts(args[0], ids, wts, *args[1:], g, True)
        assert torch.equal(y, want)


@pytest.mark.parametrize("scale_in", [True, False])
@pytest.mark.parametrize("which", ["gate_up", "down"])
def test_few_rows_of_weights_off_16_bytes(which, scale_in):
    """One to two rows an expert: no copy of the stacks, the vector product's results in the order of the stream's groups; identity experts too."""
    E, d, F = 32, 256, 512
    h, ids, wts, gu, dn = _case([1, 2, 3, 0] * 8 + [9], 3, d, F)  # (the last id has no weights)
    gu, dn = gu[:E].contiguous(), dn[:E].contiguous()
    off = lambda t: torch.empty(t.numel() + 8, device="cuda", dtype=t.dtype)[1:1 + t.numel()].view(t.shape).copy_(t)  # noqa: E731
    gu, dn = (off(gu), dn) if which == "gate_up" else (gu, off(dn))
    g, own = moe.group(ids, E, moe.STREAM_ROWS), moe.group(ids, E, 8)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    y = moe.experts(h, ids, wts, gu, dn, g, scale_in)
    assert torch.cuda.max_memory_allocated() - before < dn.numel()  # (half of the smaller stack's bytes)
    want = moe.experts(h, ids, wts, gu, dn, own, scale_in)
    i, j = g.inv.view(-1), own.inv.view(-1)
    assert torch.equal(i < 0, j < 0) and torch.equal(y[i[i >= 0].long()], want[j[j >= 0].long()])
