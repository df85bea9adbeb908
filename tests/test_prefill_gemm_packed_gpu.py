"""Prefill GEMM over the packed decode-weight layout (csrc/kernels/prefill_gemm_packed.hip)
vs a plain PyTorch fp32 reference of the same op: plain store (+ bias), residual add and
the SiLU / GELU GLU epilogues, both workgroup shapes (wm = 1: 128 x 512, wm = 2: 256 x 256),
ragged M (not a multiple of the row tile, and fewer rows than one tile), N that is not a
multiple of 128 (zero-padded packed rows) or of the workgroup's 512 / 256 columns (waves
past the last weight tile), K from one 256-deep packed step up. Asymmetric random
operands catch transposed fragments and swizzles."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(autouse=True, scope="module")
def _lib():
    from hipserve.ops import load_library

    load_library()


def _rnd(g, *s, scale=1.0):
    return ((torch.rand(*s, device=DEV, generator=g) * 2 - 1) * scale).to(torch.bfloat16)


def _pack(w, glu=False):
    N, K = w.shape
    wp = torch.empty(-(-N // 128) * 128 * K, device=DEV, dtype=torch.bfloat16)
    torch.ops.hipserve.pack_decode_weight(wp, w, glu)
    return wp


SHAPES = [(256, 512, 256), (300, 640, 1024), (1000, 200, 512), (77, 1536, 768), (2049, 384, 2048),
          (1, 128, 256), (8192, 512, 4096)]


# grid: 0 = persistent (one workgroup per CU walking the tiles), 3 = three workgroups
# walking many tiles each (uneven counts), 1 << 30 = one tile per workgroup
@pytest.mark.parametrize("rw", [2, 4])  # weight slots in flight
@pytest.mark.parametrize("grid", [0, 3, 1 << 30])
@pytest.mark.parametrize("wm", [1, 2])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_packed_store(M, N, K, wm, grid, rw):
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x, w = _rnd(g, M, K), _rnd(g, N, K, scale=0.05)
    out = torch.full((M, N), float("nan"), device=DEV, dtype=torch.bfloat16)
    torch.ops.hipserve.prefill_gemm_packed(out, x, _pack(w), N, 0, None, wm, grid, rw)
    want = x.float() @ w.float().t()
    torch.testing.assert_close(out.float(), want, rtol=1e-2, atol=1e-2 * want.abs().max().item())


@pytest.mark.parametrize("wm", [1, 2])
def test_packed_store_bias_and_strided_x(wm):
    g = torch.Generator(device=DEV).manual_seed(5)
    M, N, K = 700, 896, 512
    xb = _rnd(g, M, K + 64)
    x = xb[:, 32:32 + K]  # row stride K + 64
    w, b = _rnd(g, N, K, scale=0.05), _rnd(g, N)
    out = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
    torch.ops.hipserve.prefill_gemm_packed(out, x, _pack(w), N, 0, b, wm)
    want = x.float() @ w.float().t() + b.float()
    torch.testing.assert_close(out.float(), want, rtol=1e-2, atol=1e-2 * want.abs().max().item())


@pytest.mark.parametrize("wm", [1, 2])
@pytest.mark.parametrize("M,N,K", [(300, 512, 1024), (1000, 384, 512), (2049, 1024, 256)])
def test_packed_residual_add(M, N, K, wm):
    g = torch.Generator(device=DEV).manual_seed(7 + M)
    x, w = _rnd(g, M, K), _rnd(g, N, K, scale=0.05)
    res0 = _rnd(g, M, N)
    res = res0.clone()
    torch.ops.hipserve.prefill_gemm_packed(res, x, _pack(w), N, 1, None, wm, 7, 4)  # 7 workgroups: many tiles each
    h = (x.float() @ w.float().t()).to(torch.bfloat16).float()
    want = (h + res0.float()).to(torch.bfloat16).float()
    torch.testing.assert_close(res.float(), want, rtol=1e-2, atol=2e-2)


@pytest.mark.parametrize("rw", [2, 4])
@pytest.mark.parametrize("grid", [0, 5])
@pytest.mark.parametrize("wm,act", [(1, "silu"), (2, "silu"), (1, "gelu"), (2, "gelu")])
@pytest.mark.parametrize("M,I,K", [(300, 256, 1024), (1000, 192, 512), (2049, 64, 256), (513, 1344, 768)])
def test_packed_glu(M, I, K, wm, act, grid, rw):
    g = torch.Generator(device=DEV).manual_seed(11 + M)
    x, w = _rnd(g, M, K), _rnd(g, 2 * I, K, scale=0.05)
    out = torch.full((M, I), float("nan"), device=DEV, dtype=torch.bfloat16)
    torch.ops.hipserve.prefill_gemm_packed(out, x, _pack(w, glu=True), 2 * I, 2 if act == "silu" else 3, None, wm,
                                           grid, rw)
    gu = (x.float() @ w.float().t()).to(torch.bfloat16).float()
    f = torch.nn.functional.silu if act == "silu" else (lambda t: torch.nn.functional.gelu(t, approximate="tanh"))
    want = f(gu[:, :I]) * gu[:, I:]
    torch.testing.assert_close(out.float(), want, rtol=2e-2, atol=2e-2 * want.abs().max().item())


def test_packed_rejects_bad_shapes():
    g = torch.Generator(device=DEV).manual_seed(3)
    x, w = _rnd(g, 64, 320), _rnd(g, 128, 320)
    out = torch.empty(64, 128, device=DEV, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError):  # K % 256
        torch.ops.hipserve.prefill_gemm_packed(out, x, torch.empty(128 * 320, device=DEV, dtype=torch.bfloat16),
                                               128, 0, None, 1)


@pytest.mark.parametrize("gather", [False, True])
@pytest.mark.parametrize("wm", [1, 2])
@pytest.mark.parametrize("E,I,K,glu", [(8, 512, 1024, True), (8, 256, 512, False), (16, 128, 256, True)])
def test_packed_grouped_moe(E, I, K, glu, wm, gather):
    """Grouped expert GEMM over moe_align's expert-sorted (128 * wm)-row tiles with each
    expert's weight in the packed decode layout (moe_packed: w13 GLU-interleaved), the
    valid tile count read on the device, vs a per-expert fp32 reference."""
    g = torch.Generator(device=DEV).manual_seed(E + I + K)
    T, k = 700, 2
    ids = torch.stack([torch.randperm(E, device=DEV, generator=g)[:k] for _ in range(T)]).int()
    N = 2 * I if glu else I
    w = _rnd(g, E, N, K, scale=0.05)
    wp = torch.stack([_pack(w[e], glu) for e in range(E)])
    x = _rnd(g, T, K)
    op = torch.ops.hipserve
    P, tile = T * k, 128 * wm
    cap = -(-(P + E * (tile - 1)) // tile) * tile
    slots = torch.empty(cap, dtype=torch.int32, device=DEV)
    tile_expert = torch.empty(cap // tile, dtype=torch.int32, device=DEV)
    ntiles = torch.empty(1, dtype=torch.int32, device=DEV)
    pair_slot = torch.empty(P, dtype=torch.int32, device=DEV)
    ends = torch.empty(E, dtype=torch.int32, device=DEV)
    op.moe_align(ids, E, tile, slots, tile_expert, ntiles, pair_slot, ends)
    xs = torch.empty(cap, K, dtype=torch.bfloat16, device=DEV)
    op.moe_gather(xs, x, slots, k)
    out = torch.full((cap, I), float("nan"), device=DEV, dtype=torch.bfloat16)
    op.prefill_gemm_packed_grouped(out, xs, wp, N, 2 if glu else 0, tile_expert, ntiles, wm)
    if gather:  # token rows read through the slot table inside the GEMM (moe_gather fused): bit-identical
        used = torch.arange(cap, device=DEV) < int(ntiles.item()) * tile
        fused = torch.full_like(out, float("nan"))
        op.prefill_gemm_packed_grouped(fused, x, wp, N, 2 if glu else 0, tile_expert, ntiles, wm, 4, slots, k)
        assert torch.equal(fused[used], out[used])
        assert bool((fused[used & (slots < 0)] == 0).all())  # padding slots multiply zero rows
    ps = pair_slot.long()
    for p in range(0, P, 37):  # a spread of pairs
        t, j = p // k, p % k
        e = int(ids[t, j])
        h = x[t].float() @ w[e].float().t()
        if glu:
            h = h.to(torch.bfloat16).float()
            want = torch.nn.functional.silu(h[:I]) * h[I:]
        else:
            want = h
        torch.testing.assert_close(out[ps[p]].float(), want, rtol=2e-2, atol=2e-2 * max(1.0, want.abs().max().item()))


@pytest.mark.parametrize("T,k,E,tile", [(700, 2, 8, 128), (8192, 8, 128, 128), (20000, 2, 8, 128), (9000, 8, 60, 16)])
def test_moe_align_layout(T, k, E, tile):
    """moe_align (single workgroup below 16K pairs, per-block histograms + scatter above):
    every pair has exactly one slot inside its expert's tile-padded segment, segments are in
    expert order, padding slots are -1, and the tile table / tile count / group ends match
    a host recount."""
    g = torch.Generator(device=DEV).manual_seed(T + E)
    logits = torch.randn(T, E, device=DEV, generator=g)
    ids = logits.topk(k, dim=-1).indices.int().contiguous()
    P = T * k
    cap = -(-(P + E * (tile - 1)) // tile) * tile
    op = torch.ops.hipserve
    slots = torch.empty(cap, dtype=torch.int32, device=DEV)
    tile_expert = torch.empty(cap // tile, dtype=torch.int32, device=DEV)
    ntiles = torch.empty(1, dtype=torch.int32, device=DEV)
    pair_slot = torch.empty(P, dtype=torch.int32, device=DEV)
    ends = torch.empty(E, dtype=torch.int32, device=DEV)
    op.moe_align(ids, E, tile, slots, tile_expert, ntiles, pair_slot, ends)
    flat = ids.view(-1).long().cpu()
    cnt = torch.bincount(flat, minlength=E)
    padded = (cnt + tile - 1) // tile * tile
    off = torch.cumsum(padded, 0) - padded
    assert int(ntiles.item()) == int(padded.sum()) // tile
    assert torch.equal(ends.cpu().long(), off + padded)
    s, ps, te = slots.cpu().long(), pair_slot.cpu().long(), tile_expert.cpu().long()
    assert torch.equal(s[ps], torch.arange(P))  # slots[pair_slot[p]] == p: a bijection on the real slots
    e_of = flat
    assert bool(((ps >= off[e_of]) & (ps < off[e_of] + cnt[e_of])).all())  # inside its expert's segment
    real = torch.zeros(cap, dtype=torch.bool)
    real[ps] = True
    assert bool((s[~real] == -1).all())
    want_te = torch.full((cap // tile,), -1, dtype=torch.long)
    for e in range(E):
        want_te[int(off[e]) // tile:int(off[e] + padded[e]) // tile] = e
    assert torch.equal(te, want_te)


@pytest.mark.parametrize("tiles,N,K,epi", [(66, 2048, 1536, 4), (65, 2000, 1792, 0), (35, 1024, 2048, 2), (16, 2048, 1536, 4), (300, 512, 1536, 0),
                                                 (100, 512, 1536, 4), (66, 2048, 1280, 0)])
@pytest.mark.parametrize("gather", [False, True])
def test_packed_grouped_left_over(tiles, N, K, epi, gather):
    """Tiles that whole rounds leave over (quarters of K per wave, their sums in LDS): some, all, too many; a weight tile cut off; odd
    counts of stages per wave; padding rows; K that is too short."""
    g, op, E, M = torch.Generator(device=DEV).manual_seed(tiles + N), torch.ops.hipserve, 3, tiles * 128
    w, x = _rnd(g, E, N, K, scale=0.05), _rnd(g, M // 2, K)
    wp = torch.stack([_pack(w[e], epi == 2) for e in range(E)])
    tile_expert = torch.randint(0, E, (tiles + 2,), device=DEV, generator=g, dtype=torch.int32)
    ntiles = torch.tensor([tiles], dtype=torch.int32, device=DEV)
    slots = torch.randperm(M + 256, device=DEV, generator=g).int()
    slots[(slots >= M) | (slots % 97 == 5)] = -1
    No = N // 2 if epi == 2 else N
    out = torch.full((M + 256, No), 7.0, device=DEV, dtype=torch.bfloat16)
    rows = torch.where((slots >= 0)[:, None], x[(slots.clamp(min=0) // 2).long()], 0.0).bfloat16()
    if gather:
        op.prefill_gemm_packed_grouped(out, x, wp, N, epi, tile_expert, ntiles, 1, 4, slots, 2)
    else:
        op.prefill_gemm_packed_grouped(out, rows, wp, N, epi, tile_expert, ntiles, 1)
    assert bool((out[M:] == 7.0).all())   # past the counted tiles nothing is written
    for e in range(E):
        mine = (tile_expert[:tiles] == e).repeat_interleave(128).nonzero()[:, 0]
        h = rows[mine].double() @ w[e].double().t()
        want = h.clamp(min=0).square() if epi == 4 else torch.nn.functional.silu(h[:, :No]) * h[:, No:] if epi == 2 else h
        # sums of K products in 32 bits and the result's rounding. In the gate three more: of the gate (which silu takes up at most
        # threefold for gates above -3), of silu and of the up projection: 6 x 2^-9
        rel = 2.0 ** -6 if epi == 2 else 2.0 ** -7
        assert ((out[mine].double() - want).abs() <= rel * want.abs() + 2.0 ** -9 * want.abs().mean()).all()


@pytest.mark.parametrize("tiles,counted,N", [(5, 0, 512), (300, 3, 1024), (40, 40, 1024), (64, 33, 2048)])
def test_packed_grouped_in_one_launch(tiles, counted, N, tmp_path):
    """Whatever is counted on the device, a grouped product is one launch; of a bound far above the count, and of a grid of which some
    workgroups have no whole tile, every counted row is written and no other."""
    g, op, E, K, M = torch.Generator(device=DEV).manual_seed(tiles), torch.ops.hipserve, 2, 1536, tiles * 128
    w, x = _rnd(g, E, N, K, scale=0.05), _rnd(g, M, K)
    wp = torch.stack([_pack(w[e]) for e in range(E)])
    tile_expert = torch.randint(0, E, (tiles,), device=DEV, generator=g, dtype=torch.int32)
    ntiles = torch.tensor([counted], dtype=torch.int32, device=DEV)
    out = torch.full((M, N), 7.0, device=DEV, dtype=torch.bfloat16)
    op.prefill_gemm_packed_grouped(out, x, wp, N, 0, tile_expert, ntiles, 1)
    got = out.clone()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    graph.enable_debug_mode()
    with torch.cuda.graph(graph):
        op.prefill_gemm_packed_grouped(out, x, wp, N, 0, tile_expert, ntiles, 1)
    graph.debug_dump(str(tmp_path / "graph.dot"))
    assert (tmp_path / "graph.dot").read_text().count("KERNEL") == 1
    rows = counted * 128
    assert bool((got[rows:] == 7.0).all())
    want = torch.cat([x[t * 128:(t + 1) * 128].double() @ w[int(tile_expert[t])].double().t() for t in range(counted)] + [x.new_zeros(0, N).double()])
    # sums of K products in 32 bits and the result's rounding
    assert ((got[:rows].double() - want).abs() <= 2.0 ** -7 * want.abs() + 2.0 ** -9 * K ** 0.5 * 0.05).all()


@pytest.mark.parametrize("counts,N,K,epi", [([5, 200, 64], 512, 256, 0), ([128, 33, 0, 17], 1024, 512, 4), ([129, 97, 1], 640, 768, 2),
                                            ([30] * 16 + [1000, 4096], 2048, 1024, 0), ([128 * 16 + 40, 128 * 15 + 31, 128], 4096, 1536, 4)])
@pytest.mark.parametrize("gather", [False, True])
def test_packed_grouped_by_order(counts, N, K, epi, gather):
    """Tiles in the order that the alignment leaves for rounds of them, what they leave over by columns: one to 128 rows, a weight tile cut off, fewer stages
    than are in flight, as whole rounds and as the only ones; K too short for quarters."""
    from hipserve.ops import get_ops

    g, op, E, k = torch.Generator(device=DEV).manual_seed(len(counts) + N), torch.ops.hipserve, len(counts), 2
    P = -(-sum(counts) // k) * k
    ids = torch.repeat_interleave(torch.arange(E, device=DEV), torch.tensor(counts, device=DEV))
    ids = torch.cat([ids, ids.new_full((P - len(ids),), E - 1)])[torch.randperm(P, device=DEV, generator=g)].int()
    cnt = torch.bincount(ids, minlength=E)
    cap = -(-(P + E * 127) // 128) * 128
    table, tokens = ids.view(-1, 1).contiguous(), torch.arange(P, device=DEV)   # a token per pair
    slots, te, nt, ps = (torch.empty(n, dtype=torch.int32, device=DEV) for n in (cap, cap // 128, 1, P))
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    per_round = [max(1, cus // -(-N // 512)), 3]
    orders = torch.full((2, cap // 128), -1, dtype=torch.int32, device=DEV)
    get_ops("cuda").moe_table_align(table, tokens, E, 128, slots, te, ps, nt, orders, per_round)
    n, rows = int(nt), (slots.view(-1, 128) >= 0).sum(1).cpu()
    for o, r in zip(orders[:, :n].cpu(), per_round):
        place = o >> 16
        assert torch.equal(place.sort().values, torch.arange(n)) and torch.equal(te.cpu()[place.long()], o >> 8 & 255)
        assert torch.equal(rows[place.long()], (o & 255).long() + 1)
        left = n % r if 16 * (n % r) <= 3 * r else 0
        few = sorted(x for x in rows[:n].tolist() if x < 128)[:left]
        assert rows[place.long()][n - len(few):].tolist() == few
        assert torch.equal(place[:n - len(few)], place[:n - len(few)].sort().values)   # the others as they lie
    assert torch.equal(cnt.cpu(), torch.bincount(torch.repeat_interleave(te[:n].cpu().long(), rows[:n]), minlength=E))
    w, x = _rnd(g, E, N, K, scale=0.05), _rnd(g, P, K)
    wp = torch.stack([_pack(w[e], epi == 2) for e in range(E)])
    No = N // 2 if epi == 2 else N
    xs = torch.full((cap, K), float("nan"), device=DEV, dtype=torch.bfloat16)   # rows of no pair may hold anything
    xs[ps.long()] = x
    out = torch.full((cap, No), 7.0, device=DEV, dtype=torch.bfloat16)
    if gather:
        op.prefill_gemm_packed_grouped(out, x, wp, N, epi, te, nt, 1, 4, slots, 1, order=orders[0])
    else:
        op.prefill_gemm_packed_grouped(out, xs, wp, N, epi, te, nt, 1, order=orders[0])
    assert bool((out[n * 128:] == 7.0).all())
    got = out[ps.long()]
    for e in range(E):
        mine = (ids == e).nonzero()[:, 0]
        h = x[mine].double() @ w[e].double().t()
        want = h.clamp(min=0).square() if epi == 4 else torch.nn.functional.silu(h[:, :No]) * h[:, No:] if epi == 2 else h
        rel = 2.0 ** -6 if epi == 2 else 2.0 ** -7   # as above
        assert len(mine) == 0 or ((got[mine].double() - want).abs() <= rel * want.abs() + 2.0 ** -9 * want.abs().mean()).all()


def _left_over(n, across, per_round):
    """The m-tiles that the tiles behind whole rounds are of, as the kernel walks them: groups of 8 m-tiles, column by column."""
    walk = [tm for g in range(0, n, 8) for _ in range(across) for tm in range(g, min(g + 8, n))]
    return sorted(set(walk[len(walk) // per_round * per_round:])), len(walk) % per_round


@pytest.mark.parametrize("across,per_round", [(1, 16), (2, 16), (3, 16), (3, 32), (6, 64), (5, 48), (8, 256), (3, 256)])
@pytest.mark.parametrize("counts", [[5, 200, 64], [1000, 129, 40, 300, 0, 257, 33, 1], [128] * 9, [20, 130] * 12, [700, 65, 193, 90, 321, 511, 66, 1200], [10] * 60])
def test_order_of_tiles_for_whole_rounds(counts, across, per_round):
    """Tiles of few pairs last where what whole rounds of the GEMM's tiles leave over goes by columns, which it does not for three sixteenths of a round with
    longer ones; numbers of tiles beside each other that divide a round, and that do not."""
    from hipserve.ops import get_ops

    E, P = len(counts), sum(counts)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(P, generator=torch.Generator().manual_seed(P))].int().to(DEV)
    cap = -(-(P + E * 127) // 128) * 128
    slots, te, nt, ps = (torch.empty(n, dtype=torch.int32, device=DEV) for n in (cap, cap // 128, 1, P))
    orders = torch.full((2, cap // 128), -1, dtype=torch.int32, device=DEV)
    get_ops("cuda").moe_table_align(ids.view(-1, 1), torch.arange(P, device=DEV), E, 128, slots, te, ps, nt, orders, [7, per_round], [1, across])
    n, rows = int(nt), (slots.view(-1, 128) >= 0).sum(1).cpu()
    o = orders[1, :n].cpu().long()
    place = o >> 16
    assert torch.equal(te.cpu()[place].long(), o >> 8 & 255) and torch.equal(rows[place], (o & 255) + 1)
    left, over = _left_over(n, across, per_round)
    partial = sorted((int(rows[t]), t) for t in range(n) if rows[t] < 128)
    moved = partial[:len(left)]
    short = len(moved) == len(left) and all(r <= 64 for r, _ in moved)
    if 16 * over > (3 if short else 2) * per_round:
        moved = []
    gone = {t for _, t in moved}
    assert place.tolist() == [t for t in range(n) if t not in gone] + [t for _, t in moved]
    assert not moved or left == list(range(left[0], n))   # they are the last places


@pytest.mark.parametrize("P", [1, 65, 1024, 1025, 4096, 4097, 16384, 65537])
@pytest.mark.parametrize("E", [1, 2, 16, 100, 128])
def test_alignments_for_the_packed_gemm_repeat(P, E):
    """A pair has the same place in every run, whatever the order of the waves, and every pair one of its expert's: with a table and without one."""
    from hipserve.ops import get_ops

    op, g = torch.ops.hipserve, torch.Generator(device=DEV).manual_seed(P + E)
    ids = (torch.randint(0, E, (P,), device=DEV, generator=g) if E < 100 else (torch.rand(P, device=DEV, generator=g) ** 3 * E).long()).int()
    cap = -(-(P + E * 127) // 128) * 128
    first = None
    for _ in range(6):
        runs = []
        for table in (False, True) if P <= 16384 else (False,):
            slots, te, nt, ps = (torch.full((n,), -7, dtype=torch.int32, device=DEV) for n in (cap, cap // 128, 1, P))
            if table:
                get_ops("cuda").moe_table_align(ids.view(-1, 1), torch.arange(P, device=DEV), E, 128, slots, te, ps, nt)
            else:
                op.moe_align(ids, E, 128, slots, te, nt, ps)
            runs.append((slots, te, nt, ps))
        first = first or runs
        assert all(torch.equal(a, b) for x, y in zip(first, runs) for a, b in zip(x, y))
    for slots, te, nt, ps in first:
        assert torch.equal(slots[ps.long()], torch.arange(P, device=DEV).int()) and int((slots >= 0).sum()) == P
        assert torch.equal(te[ps.long() // 128], ids)
        live = slots.view(-1, 128) >= 0   # a tile is filled from its first slot on
        assert bool((live[:, 1:] <= live[:, :-1]).all())
        assert int(nt) == int((-(-torch.bincount(ids, minlength=E) // 128)).sum())


@pytest.mark.parametrize("T,E,H,ff,ordered", [(3000, 4, 512, 512, 2), (8192, 8, 512, 512, 0), (8192, 8, 2048, 512, 1), (8192, 8, 512, 2048, 1), (16384, 8, 1024, 512, 1),
                                              (6145, 1, 512, 512, 0), (6144, 1, 512, 512, 2)])
def test_packed_experts_ordered_where_it_matters(T, E, H, ff, ordered, monkeypatch):
    """Products whose tiles are all taken alike get no order of them, with the bits that they have in one."""
    from hipserve.config import TableMoESpec
    from hipserve.models.mixers import TableMoE
    from hipserve.ops import get_ops, gemm

    ops, op, g = get_ops("cuda"), torch.ops.hipserve, torch.Generator(device=DEV).manual_seed(T + E)
    m = TableMoE(TableMoESpec(experts=E, top=1, ff=ff), H, 97, torch.device("cuda"), torch.bfloat16, ops)
    m.w_up, m.w_down, m.table = _rnd(g, E, ff, H, scale=0.05), _rnd(g, E, H, ff, scale=0.05), torch.randint(0, E, (97, 1), device=DEV, generator=g).int()
    h, ids, asked, align = _rnd(g, T, H), torch.randint(0, 97, (T,), device=DEV, generator=g), [], ops.moe_table_align
    monkeypatch.setattr(ops, "moe_table_align", lambda *a: (asked.append(len(a[9])), align(*a)))
    y, ps = m._forward_packed(h, ids, T)
    assert asked == [ordered]
    tile, cus = 128 * gemm.PW_WM, torch.cuda.get_device_properties(0).multi_processor_count
    cap = -(-(T + E * (tile - 1)) // tile) * tile
    slots, te, nt, pair = (torch.empty(n, dtype=torch.int32, device=DEV) for n in (cap, cap // tile, 1, T))
    orders = torch.empty(2, cap // tile, dtype=torch.int32, device=DEV)
    align(m.table, ids, E, tile, slots, te, pair, nt, orders, [cus, cus], [-(-n * gemm.PW_WM // 512) for n in (ff, H)])
    act, want = (torch.empty(cap, n, dtype=torch.bfloat16, device=DEV) for n in (ff, H))
    op.prefill_gemm_packed_grouped(act, h, m.packed[0], ff, 4, te, nt, gemm.PW_WM, gemm.PW_RW, slots, 1, order=orders[0])
    op.prefill_gemm_packed_grouped(want, act, m.packed[1], H, 0, te, nt, gemm.PW_WM, gemm.PW_RW, order=orders[1])
    assert torch.equal(y[ps.long()], want[pair.long()]) and y[ps.long()].isfinite().all()
