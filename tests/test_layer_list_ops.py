"""Kernels of the layer-list decoders alone, at the sizes where their variants meet, against the reference ops."""
import pytest
import torch

from hipserve.ops import NormedRows, get_ops
from hipserve.ops import reference as ref

gpu = pytest.mark.gpu


# ------------------------------------------------------------------ residual update + grouped norm
def norm_case(H, groups, top, parts, dtype, dev, T=3):
    g = torch.Generator().manual_seed(H + 7 * groups + top)

    def rnd(*s):
        return torch.randn(*s, generator=g)

    res, w = rnd(T, H), 1 + 0.1 * rnd(H)
    kw = {}
    if "mix" in parts:
        kw.update(mix=rnd(T, H).to(dtype), ls1=0.5 + 0.1 * rnd(H) if "ls1" in parts else None)
    if "y" in parts:
        kw.update(y=rnd(2 * T * top, H).to(dtype), pair_slot=torch.randperm(2 * T * top, generator=g)[:T * top].int(), top=top,
                  ls2=0.5 + 0.1 * rnd(H))
    if "extra" in parts:
        kw.update(extra=rnd(T, H).to(dtype))
    if "table" in parts:
        kw.update(table=rnd(11, H).to(dtype), ids=torch.tensor([10, 0, 3][:T]))
    return res, w, {k: v.to(dev) if isinstance(v, torch.Tensor) else v for k, v in kw.items()}


@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,groups", [(4, 1), (96, 4), (1020, 5), (1024, 1), (1024, 8), (1026, 1), (1032, 3), (2048, 4), (2056, 1),
                                      (4096, 4), (4104, 1), (8192, 4), (8200, 5), (14000, 2), (1000, 8), (21, 3)])
@pytest.mark.parametrize("parts,top", [((), 0), (("mix",), 0), (("mix", "ls1", "y"), 1), (("mix", "ls1", "y", "extra"), 2),
                                       (("y",), 3), (("table",), 0), (("table", "mix", "ls1"), 0)])
def test_group_norm_variants(H, groups, parts, top, dtype):
    """The register kernel (lengths and groups that are multiples of 4 or 8) and the element loop, every addend."""
    if H % groups:
        pytest.skip("unequal groups")
    res, w, kw = norm_case(H, groups, top, parts, dtype, "cpu")
    want_res, want = res.clone(), torch.empty(res.shape, dtype=dtype)
    ref.scaled_add_group_rmsnorm(want, want_res, w, groups, 1e-6, **kw)
    ops, dev = get_ops("cuda"), "cuda"
    ops.norm_library = "delta"
    got_res, got = res.to(dev), torch.empty(res.shape, dtype=dtype, device=dev)
    ops.scaled_add_group_rmsnorm(got, got_res, w.to(dev), groups, 1e-6,
                                 **{k: v.to(dev) if isinstance(v, torch.Tensor) else v for k, v in kw.items()})
    # at most 6 additions of numbers below 20 in 32 bits; the norm's sums differ in order
    err = 6 * 20 * 2.0 ** -24
    assert (got_res.cpu() - want_res).abs().max() <= err
    tol = 2.0 ** -7 if dtype == torch.bfloat16 else 2e-6   # neighbouring bf16 numbers; the rounding of the norm
    # an element where the addends cancel keeps their absolute error, times 1 / rms (below 2) and w (below 1.5)
    assert ((got.cpu().float() - want.float()).abs() <= tol * want.float().abs() + 3 * err).all()


@gpu
def test_group_norm_unknown_id_and_unaligned_rows():
    """An id outside the table reads nothing and gives NaN; rows that do not start at 16 bytes take the element loop."""
    ops = get_ops("cuda")
    ops.norm_library = "delta"
    H = 64
    table, w = torch.randn(5, H, device="cuda"), torch.ones(H, device="cuda")
    res, out = torch.empty(3, H, device="cuda"), torch.empty(3, H, device="cuda")
    ops.scaled_add_group_rmsnorm(out, res, w, 1, 1e-6, table=table, ids=torch.tensor([5, 2, -1], device="cuda"))
    assert res[[0, 2]].isnan().all() and out[[0, 2]].isnan().all() and torch.equal(res[1], table[2])
    shifted = torch.zeros(3 * H + 1, device="cuda")[1:].view(3, H)   # 4 bytes past a 16-byte boundary
    shifted.copy_(torch.randn(3, H, device="cuda"))
    a, b, ra, rb = torch.empty_like(out), torch.empty_like(out), shifted, shifted.clone()
    ops.scaled_add_group_rmsnorm(a, ra, w, 2, 1e-6)
    ops.scaled_add_group_rmsnorm(b, rb, w, 2, 1e-6)
    assert torch.equal(ra, rb) and torch.allclose(a, b, rtol=2e-6, atol=0)


@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,groups", [(1024, 4), (2048, 1), (2048, 8), (4096, 16), (4096, 2), (1280, 5), (3072, 3)])
@pytest.mark.parametrize("T", [1, 3, 300])
@pytest.mark.parametrize("kind", [0, 1, 2, 3, 4, "table"])
def test_group_norm_of_known_sizes(H, groups, T, kind, dtype):
    """Rows and groups of whole waves, and sizes beside them: ``mix`` as a row, in one to four parts, with two expert rows; ids inside and outside the table."""
    g = torch.Generator().manual_seed(H + T)
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    res, w, kw, mix = rnd(T, H), 1 + 0.1 * rnd(H), {}, None
    if kind == "table":
        ids = torch.randint(0, 7, (T,), generator=g)
        ids[T // 2] = 7 if T > 1 else 6
        kw = dict(table=rnd(7, H).to(dtype), ids=ids)
    else:
        mix = rnd(T, H).to(dtype) if kind == 0 else rnd(kind, T, H)
        kw = dict(ls1=0.5 + 0.1 * rnd(H), y=rnd(2 * T + 3, H).to(dtype), pair_slot=torch.randperm(2 * T + 3, generator=g)[:2 * T].int(), top=2, ls2=0.5 + 0.1 * rnd(H))
    if kind == "table":
        x = torch.where((ids < 7)[:, None], kw["table"][ids.clamp(max=6)].double(), float("nan"))
    else:
        x = res.double() + (mix.double() if kind == 0 else mix.double().sum(0)) * kw["ls1"].double()
        x += kw["y"][kw["pair_slot"].long().view(T, 2)].double().sum(1) / 2 * kw["ls2"].double()
    want = (x.view(T, groups, -1) * torch.rsqrt(x.view(T, groups, -1).square().mean(-1, keepdim=True) + 1e-6)).view(T, H) * w.double()
    dev = lambda v: v.cuda() if isinstance(v, torch.Tensor) else v  # noqa: E731
    got_res, got = res.cuda(), torch.empty(T, H, dtype=dtype, device="cuda")
    ops = get_ops("cuda")
    ops.norm_library = "delta"
    ops.scaled_add_group_rmsnorm(got, got_res, w.cuda(), groups, 1e-6, dev(mix), **{k: dev(v) for k, v in kw.items()})
    ok = ~x.isnan()
    assert torch.equal(got_res.cpu().isnan(), ~ok) and torch.equal(got.cpu().isnan(), ~ok)
    err = 8 * 16 * 2.0 ** -24   # eight additions of numbers below 16 in 32 bits
    assert (got_res.cpu().double() - x)[ok].abs().max() <= err
    # a neighbouring bf16 number; the norm's 32-bit sum and root; where the addends cancel, their error times 1 / rms (below 2) and w (below 1.5)
    tol = 2.0 ** -8 if dtype == torch.bfloat16 else 2e-6
    assert ((got.cpu().double() - want).abs()[ok] <= tol * want.abs()[ok] + 3 * err).all()


@gpu
@pytest.mark.parametrize("T", [2000, 2001])
@pytest.mark.parametrize("groups", [1, 16])
def test_embedding_rows_of_long_prompts(T, groups):
    """Wide rows from a table, at both sides of the change of kernels; ids outside the table give NaN."""
    g = torch.Generator().manual_seed(T)
    H, table, w, ids = 4096, torch.randn(50, 4096, generator=g).bfloat16(), 1 + 0.1 * torch.randn(4096, generator=g), torch.randint(0, 50, (T,), generator=g)
    ids[[0, T - 1]] = torch.tensor([50, -1])
    x = table[ids.clamp(0, 49)].double()
    want = (x.view(T, groups, -1) * torch.rsqrt(x.view(T, groups, -1).square().mean(-1, keepdim=True) + 1e-6)).view(T, H) * w.double()
    ops, res, out = get_ops("cuda"), torch.empty(T, H, device="cuda"), torch.empty(T, H, dtype=torch.bfloat16, device="cuda")
    ops.norm_library = "delta"
    ops.scaled_add_group_rmsnorm(out, res, w.cuda(), groups, 1e-6, table=table.cuda(), ids=ids.cuda())
    res, out, known = res.cpu().double(), out.cpu().double(), slice(1, T - 1)
    assert torch.equal(res[known], x[known]) and ((out - want).abs()[known] <= 2.0 ** -8 * want.abs()[known]).all()   # a neighbouring bf16 number
    assert all(v[i].isnan().all() for v in (res, out) for i in (0, T - 1))


# ------------------------------------------------------------------ soft cap
@pytest.mark.parametrize("dev", ["cpu", pytest.param("cuda", marks=gpu)])
@pytest.mark.parametrize("shape", [(1, 5), (3, 2048), (2, 32001)])
def test_softcap(shape, dev):
    x = torch.randn(shape, generator=torch.Generator().manual_seed(1)) * 40
    x.view(-1)[0], x.view(-1)[-1] = float("inf"), -float("inf")
    want = torch.tanh(x.double() / 25.0) * 25.0
    y = x.to(dev)
    get_ops(dev).activation(y, y, "softcap", 25.0)
    # division, tanh and product: a few units in the last place of numbers up to 25
    assert (y.cpu().double() - want).abs().max() <= 25 * 4 * 2.0 ** -23


# ------------------------------------------------------------------ dense layers of a few rows
def dense_case(B, M, N, K, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(B, M, K, generator=g).bfloat16(), (torch.randn(B, N, K, generator=g) / K ** 0.5).bfloat16()


def act64(z, act, c0, c1):
    """The activations in 64 bits."""
    if act in ("silu_mul", "clamped_glu"):
        g, u = z.chunk(2, -1)
        if act == "silu_mul":
            return g * torch.sigmoid(g) * u
        g, u = g.clamp(max=c0), u.clamp(-c0, c0)
        return g * torch.sigmoid(1.702 * g) * (u + 1)
    return {None: lambda: z, "tanh": z.tanh, "relu2": lambda: z.relu() ** 2, "softcap": lambda: torch.tanh(z / c0) * c0,
            "xielu": lambda: torch.where(z > 0, c0 * z * z + z / 2, c1 * (torch.expm1(z.clamp(max=0)) - z) + z / 2)}[act]()


def close_to(got, want, x, w, scale=1.0):
    """A bf16 rounding of the result, and 32-bit sums of K products taken in any order (times the activation's slope)."""
    K = x.shape[-1]
    err = scale * K * 2.0 ** -24 * torch.matmul(x.double().abs(), w.double().abs().transpose(-1, -2)).max()
    tol = 2.0 ** -8 if got.dtype == torch.bfloat16 else 2.0 ** -21
    assert ((got.double().cpu() - want).abs() <= tol * want.abs() + err + 1e-6).all()


@gpu
@pytest.mark.parametrize("M", [1, 3, 5, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("N,K", [(1, 8), (16, 64), (40, 72), (17, 512), (96, 520), (33, 1024), (48, 1032), (130, 2048), (16, 6152)])
def test_skinny_linear(M, N, K):
    """Row tiles, columns and k that fill the tiles of 16 rows, 16 columns and 64 k partly; bias, 32-bit results, row strides."""
    (x,), (w,) = dense_case(1, M, N, K, M + N + K)
    ops = get_ops("cuda")
    want = x.double() @ w.double().T
    wide = torch.zeros(M, K + 24, dtype=torch.bfloat16, device="cuda")
    wide[:, 8:8 + K] = x.cuda()
    out = torch.full((M, N + 5), 7.0, device="cuda")
    bias = torch.randn(N, generator=torch.Generator().manual_seed(N)).bfloat16()
    ops._moe_lib.skinny_linear(out[:, :N], wide[:, 8:8 + K], w.cuda(), None, -1, 0.0, 0.0)
    close_to(out[:, :N], want, x, w)
    assert (out[:, N:] == 7.0).all()
    half = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    ops._moe_lib.skinny_linear(half, x.cuda(), w.cuda(), bias.cuda(), -1, 0.0, 0.0)
    close_to(half, want + bias.double(), x, w)


def test_rules_of_a_few_rows_are_asked_once_per_size():
    """Every product of every step asks; a step that is not captured waits for the answers."""
    from types import SimpleNamespace

    from hipserve.ops import KernelOps
    ops, asked = KernelOps(), []
    ops._lib_ops = {"seq": SimpleNamespace(skinny_linear=lambda *a: None, skinny_linear_parts=lambda *a: None, skinny_linear_update=lambda *a: None,
                                           skinny_time=lambda *a: asked.append(a) or 3.0)}
    x, w, residual = torch.zeros(7, 1048), torch.zeros(1088, 1048), torch.zeros(7, 1088)
    for _ in range(2):
        seen = len(asked)
        ops.linear(x, w)
        ops.linear_parts(x, w)
        ops.linear_update(x, w, None, residual, torch.ones(1088), 1e-6)
    assert seen > 0 and len(asked) == seen


@pytest.mark.parametrize("dtype,kv,dim,n,keys,normed,one", [
    (torch.float32, 8, 128, 32, 70, True, True), (torch.float32, 8, 128, 33, 70, False, False), (torch.float32, 8, 128, 4, 900, False, True),
    (torch.float32, 8, 128, 5, 900, False, False), (torch.float32, 8, 128, 33, 900, True, False), (torch.float32, 8, 128, 64, 900, False, False),
    (torch.float32, 8, 128, 65, 900, True, True), (torch.float32, 4, 128, 128, 900, True, True), (torch.float32, 4, 128, 128, 128, True, False),
    (torch.float32, 4, 128, 128, 129, True, True), (torch.float32, 8, 64, 64, 900, True, True), (torch.bfloat16, 8, 128, 64, 70, True, True),
    (torch.bfloat16, 8, 128, 64, 900, True, True)])
def test_window_step_in_one_launch_by_its_workgroups(dtype, kv, dim, n, keys, normed, one):
    """A decode step's preparation is a launch of its own where a compute unit would take several workgroups with it in turn."""
    from types import SimpleNamespace

    from hipserve.ops import KernelOps
    ops, ran = KernelOps(), []
    ops._lib_ops = {"delta": SimpleNamespace(window_attention_decode_ok=lambda *a: True, window_attention_step=lambda *a: ran.append(a))}
    sp = SimpleNamespace(maps=1, dim=dim, vdim=dim, heads=4 * kv, kv_heads=kv, window=1024, reach=1024, scale=1.0, sink=False, keep_first=0, softcap=0.0,
                         channel_gate=False, chunk=0, kv_from=None, qk_norm=normed, head_norm=False, unit_qk=False, v_norm=False, scaling=None, temp_coef=0.0,
                         temp_every=0)
    meta = SimpleNamespace(max_q=1, num_prefill_tokens=0, num_decode=n, seq_ctx=torch.zeros(n), seq_cu=None, seq_bt=None, positions=None, slot_mapping=None, max_ctx=keys)
    proj, norm_w = torch.zeros(n, 8, dtype=dtype), torch.zeros(4) if normed else None
    assert ops.window_step(torch.zeros_like(proj), proj, proj, meta, torch.zeros(dim // 2), sp, *(2 * [norm_w]), 1e-6, -1) == one and len(ran) == one


@pytest.mark.parametrize("dtype,rank,most", [(torch.bfloat16, 64, 64), (torch.bfloat16, 128, 32), (torch.float32, 64, 32), (torch.float32, 128, 8)])
def test_bottleneck_in_the_rules_launch_by_its_workgroups(dtype, rank, most):
    """Up to ``most`` rows of 64 heads; a product of its own where its rows would be read too often."""
    from types import SimpleNamespace

    from hipserve.ops import KernelOps
    ops, ran = KernelOps(), []
    ops._lib_ops = {"delta": SimpleNamespace(delta_rule_step_ok=lambda *a: True, delta_rule_step=lambda *a: ran.append(a))}
    sp, w2 = SimpleNamespace(heads=64, dim=64), torch.zeros(4096, rank, dtype=dtype)
    for n in (1, most, most + 1):
        meta, proj = SimpleNamespace(max_q=1, seq_cu=None, seq_ctx=None, seq_state=None), torch.zeros(n, 8, dtype=dtype)
        ran.clear()
        assert ops.delta_rule_low(None, [torch.zeros(4)], proj, w2, None, None, None, sp, 1e-6, meta) == (n <= most) == bool(ran)


@pytest.mark.parametrize("dev", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("M", [1, 17, 70])
@pytest.mark.parametrize("first", [1, 16, 39])
def test_linear_activation_of_last_columns(dev, M, first):
    (x,), (w,) = dense_case(1, M, 40, 64, M + first)
    w = w * 4
    got = get_ops(dev).linear(x.to(dev), w.to(dev), act="tanh", act_from=first)
    want = x.double() @ w.double().T
    want[:, first:] = torch.tanh(want[:, first:])
    # past 64 rows the product is rounded before the activation
    assert ((got.double().cpu() - want).abs() <= 2.0 ** -7 * want.abs() + 1e-3).all()


@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N,K,parts", [(1, 16, 128, 2), (3, 40, 1032, 8), (17, 2064, 1024, 3), (48, 1032, 3080, 6), (64, 16, 64, 1), (5, 5001, 1544, 4)])
def test_product_in_parts(M, N, K, parts, dtype):
    """Parts of k that end inside a wave's share, of a piece each, with a last piece cut off; the bias once; the residual update that
    adds them up (its general kernel for rows that are no multiple of 4)."""
    g = torch.Generator().manual_seed(M + N + K)
    x, w, bias = torch.randn(M, K, generator=g).to(dtype), (torch.randn(N, K, generator=g) / K ** 0.5).to(dtype), torch.randn(N, generator=g).to(dtype)
    ops = get_ops("cuda")
    out = torch.full((parts, M, N), 7.0, device="cuda")
    ops._moe_lib.skinny_linear_parts(out, x.cuda(), w.cuda(), bias.cuda())
    want = x.double() @ w.double().T + bias.double()
    close_to(out.double().sum(0), want, x, w)
    res, norm, ls = torch.randn(M, N, generator=g), torch.randn(N, generator=g), torch.randn(N, generator=g)
    h, r = torch.empty(M, N, dtype=dtype, device="cuda"), res.cuda()
    ops.scaled_add_group_rmsnorm(h, r, norm.cuda(), 1, 1e-6, out, ls.cuda())
    sums = res.double() + want * ls.double()
    # the product's sums (close_to), times ls1, added in 32 bits
    assert ((r.double().cpu() - sums).abs() <= 2.0 ** -20 * (res.double().abs() + 4 * ls.double().abs() * (1 + want.abs())) + 1e-5).all()
    n = sums * torch.rsqrt(sums.square().mean(-1, keepdim=True) + 1e-6) * norm.double()
    assert ((h.double().cpu() - n).abs() <= (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -17) * n.abs() + 2e-5).all()


@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,H,K,N,act", [(1, 64, 96, 40, None), (3, 1024, 520, 96, "xielu"), (9, 2112, 1024, 130, "silu_mul"), (16, 4096, 128, 4128, "tanh"),
                                         (17, 128, 64, 16, None), (32, 1024, 3080, 5008, None)])
def test_norm_inside_the_products(M, H, K, N, act, dtype):
    """The residual update in one product and the norm's factor in the next: blocks of squares that fill a row's lanes partly, one and two
    tiles per workgroup, a bias in both, every row group."""
    g = torch.Generator().manual_seed(M + H)
    x, w, b = torch.randn(M, K, generator=g).to(dtype), (torch.randn(H, K, generator=g) / K ** 0.5).to(dtype), torch.randn(H, generator=g).to(dtype)
    res, norm = torch.randn(M, H, generator=g) * 3, 1 + 0.1 * torch.randn(H, generator=g)
    w2, b2 = (torch.randn(N, H, generator=g) / H ** 0.5).to(dtype), torch.randn(N, generator=g).to(dtype)
    ops, r = get_ops("cuda"), res.cuda()
    rows = torch.empty(M, H, dtype=dtype, device="cuda")
    squares = torch.full((M, H // 16), float("nan"), device="cuda")
    ops._moe_lib.skinny_linear_update(rows, squares, r, norm.cuda(), x.cuda(), w.cuda(), b.cuda())
    want = res.double() + x.double() @ w.double().T + b.double()
    close_to(r, want, x, w)
    close_to(rows, want * norm.double(), x, w, scale=2.0)
    assert torch.allclose(squares.double().cpu().sum(1), want.square().sum(1), rtol=1e-5)
    h = NormedRows(rows, squares, 1e-6)
    for first in (0, 8) if act == "tanh" else (0,):
        got = ops.linear(h, w2.cuda(), b2.cuda(), act=act, c0=0.7, c1=0.9, act_from=first)
        # of the rows as they are; the factor's and the product's 32-bit sums
        n = rows.double().cpu() * torch.rsqrt(squares.double().cpu().sum(1, keepdim=True) / H + 1e-6)
        z = n @ w2.double().T + b2.double()
        y = act64(z, act, 0.7, 0.9)
        close_to(got, torch.cat([z[:, :first], y[:, first:]], 1) if first else y, n, w2, scale=12.0)
    assert torch.allclose(h.normed().double().cpu(), n, rtol=2.0 ** -7 if dtype == torch.bfloat16 else 1e-5, atol=1e-6)


@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 25, 33, 49])
@pytest.mark.parametrize("N,K", [(1, 1032), (9, 2056), (1660, 1096), (2048, 4104)])
def test_products_in_half_tiles(M, N, K, dtype):
    """Workgroups of 8 columns: the same bits as those of 16, which the same columns among more of them take; a last workgroup that is partly
    filled, k past a whole piece, two and three pieces ahead, a bias, an activation."""
    g = torch.Generator().manual_seed(M + N)
    x, b = torch.randn(M, K, generator=g).to(dtype).cuda(), torch.randn(N + 2064, generator=g).to(dtype).cuda()
    w = torch.randn(N + 2064, K, generator=g).to(dtype).cuda()
    lib = get_ops("cuda")._moe_lib
    f32 = dtype == torch.float32
    assert not lib.skinny_half(M, N + 2064, K, f32) and lib.skinny_half(M, N, K, f32) == (M > 8 or N > 1024 or K * (1 + f32) > 4096)
    for act in (-1, 0):
        got, want = torch.empty(M, N, dtype=dtype, device="cuda"), torch.empty(M, N + 2064, dtype=dtype, device="cuda")
        lib.skinny_linear(got, x, w[:N], b[:N], act, 0.0, 0.0)
        lib.skinny_linear(want, x, w, b, act, 0.0, 0.0)
        assert torch.equal(got, want[:, :N])


@gpu
@pytest.mark.parametrize("M,N,K,dtype", [
    (9, 4097, 2048, "bf16"), (16, 6144, 2056, "bf16"), (17, 6133, 1024, "bf16"), (48, 4104, 1032, "bf16"),    # 24 columns
    (16, 8193, 3072, "bf16"), (25, 10239, 1096, "bf16"), (33, 8705, 2048, "bf16"),                           # 40
    (24, 12288, 1024, "bf16"), (41, 10241, 2056, "bf16"), (15, 11264, 3080, "bf16"),                          # 48
    (10, 12289, 3072, "bf16"), (32, 14329, 3080, "bf16"),                                                     # 56
    (18, 20473, 1032, "bf16"), (48, 28665, 3072, "bf16"),                                                     # two rounds, of 40 and 56
    (1, 5648, 2048, "bf16"), (4, 8191, 2048, "bf16"),                                                         # up to 4 rows: half tiles
    (5, 6145, 2048, "bf16"), (8, 8193, 2568, "bf16"), (3, 8200, 4096, "bf16"), (1, 8193, 1032, "f32"), (7, 6160, 1024, "f32")])   # three pieces ahead
def test_products_of_many_columns(M, N, K, dtype):
    """Forms for more workgroups than compute units: the first and last columns have the bits that a product of them alone has, from rows as they are and from
    rows without their norm's factor; a last workgroup that is partly filled, a bias, an activation from some column on."""
    dt = torch.bfloat16 if dtype == "bf16" else torch.float32
    g = torch.Generator("cuda").manual_seed(M + N)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g).to(dt)  # noqa: E731
    x, w, b, ops = rand(M, K), rand(N, K) / 32, rand(N), get_ops("cuda")
    rows = [x] if K % 64 or M > 32 else [x, NormedRows(x, torch.rand(M, K // 16, device="cuda", generator=g) * 16, 1e-6)]
    n = 200   # columns that are looked at, at either end
    for h in rows:
        if h is x:
            got, first, last = (torch.empty(M, c, dtype=dt, device="cuda") for c in (N, n, n))
            for out, a, z, start in ((got, w, b, 50), (first, w[:n], b[:n], 50), (last, w[-n:], b[-n:], 0)):
                ops._moe_lib.skinny_linear(out, x, a, z, 0, 0.0, 0.0, start)
        else:
            got, first, last = (ops.linear(h, a, z, act="tanh", act_from=start) for a, z, start in ((w, b, 50), (w[:n], b[:n], 50), (w[-n:], b[-n:], 0)))
        assert torch.equal(got[:, :n], first) and torch.equal(got[:, -n:], last)
        whole = h.normed() if h is not x else x
        want = torch.mm(whole.float(), w.t().float()) + b.float()
        want = torch.cat([want[:, :50], torch.tanh(want[:, 50:])], 1)
        err = (got.float() - want).abs() / (1 + want.abs())
        assert err.max() < (0.02 if dt == torch.bfloat16 else 1e-4)   # what lies between them: no column left out (a result rounded to 2^-9, of rows rounded to 2^-9; 32-bit sums)


@gpu
@pytest.mark.parametrize("normed", [False, True])
@pytest.mark.parametrize("M,N,K", [(1, 5648, 8192), (4, 6137, 8192), (3, 5640, 16384)])
def test_half_tiles_of_wide_products_are_exact(M, N, K, normed):
    """Three pieces ahead: the bits of the columns' products alone at either end, and in between what 64 bits give."""
    g = torch.Generator("cuda").manual_seed(M + N)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g).bfloat16()  # noqa: E731
    x, w, b, ops, n = rand(M, K), rand(N, K) / 64, rand(N), get_ops("cuda"), 200
    assert ops._moe_lib.skinny_wide(M, N, K, False, normed) == ([0, False] if normed and N <= 6144 else [3, not normed])
    out, first, last = (torch.empty(M, c, dtype=x.dtype, device="cuda") for c in (N, n, n))
    for o, a, z in ((out, w, b), (first, w[:n], b[:n]), (last, w[-n:], b[-n:])):
        if normed:
            ops._moe_lib.skinny_linear_normed(o, x, torch.full((M, 256), K / 256, device="cuda"), 1e-6, a, z, -1, 0.0, 0.0, 0)
        else:
            ops._moe_lib.skinny_linear(o, x, a, z, -1, 0.0, 0.0)
    assert torch.equal(out[:, :n], first) and torch.equal(out[:, -n:], last)
    want = x.double() @ w.double().t() * (1 / (1 + 1e-6) ** 0.5 if normed else 1) + b.double()
    assert ((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + K * 2.0 ** -23 * (x.double().abs() @ w.double().abs().t())).all()


@pytest.mark.parametrize("rows,cols,k,cut", [
    (8192, 6176, 1024, 6144), (8192, 26688, 4096, 26624), (7900, 4128, 2048, 4096), (2048, 8200, 1024, 8192), (1024, 16512, 64, 16384), (1100, 13072, 64, 13056),
    (8192, 2656, 4096, 2048), (8192, 6288, 2048, 6144), (2048, 10304, 2048, 8192), (4073, 13376, 4096, 12288),   # some columns more
    (8192, 6144, 2048, 0), (8192, 13376, 2048, 0), (8192, 6148, 2048, 0), (8192, 6288, 1024, 0), (1000, 16400, 2048, 0), (3133, 15120, 2048, 0), (6144, 13584, 2048, 0),
    (8192, 200, 2048, 0), (0, 6176, 2048, 0), (5142, 0, 4096, 0), (8448, 2656, 4096, 0)])
def test_columns_that_would_start_a_round(rows, cols, k, cut):
    from hipserve.ops.gemm import round_columns

    assert round_columns(rows, cols, k) == cut


@pytest.mark.parametrize("rows,cols,k,cut", [
    (7195, 4456, 8192, 0), (3312, 10072, 4096, 0), (1628, 18768, 4096, 0),              # 29 x 17, 13 x 39, 7 x 73 tiles
    (4298, 7768, 4096, 7680), (1100, 13072, 4096, 13056), (7900, 4128, 4096, 4096)])    # 17 x 30, 5 x 51, 31 x 16
def test_columns_of_tiles_odd_both_ways(rows, cols, k, cut):
    """Tiles in the second round, in an odd number both ways, are slower apart by up to two thirds."""
    from hipserve.ops.gemm import round_columns

    assert round_columns(rows, cols, k) == cut


@pytest.mark.parametrize("rows,cols,k,cut", [
    (5142, 4096, 14336, 4096), (4097, 4096, 2048, 4096), (2713, 24576, 4096, 2048), (6500, 28672, 4096, 4096), (7310, 16384, 2048, 7168),
    (4096, 4096, 14336, 0), (5700, 4096, 12288, 0), (7000, 12288, 2048, 0), (3510, 24576, 1024, 0), (1040, 16384, 8192, 0), (5142, 4104, 14336, 0), (9000, 4096, 4096, 0),
    (5142, 6144, 4096, 0), (0, 4096, 4096, 0), (5142, 0, 4096, 0)])
def test_rows_that_would_start_a_round(rows, cols, k, cut):
    from hipserve.ops.gemm import round_rows

    assert round_rows(rows, cols, k) == cut


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("rows,cols,K,grad", [(1024, 16400, 72, False), (1100, 13072, 40, True), (2049, 8192, 2048, False), (4100, 4096, 2056, False), (2050, 9736, 2048, False)])
def test_products_in_whole_rounds(rows, cols, K, grad, device):
    """A long prompt's product in two: rows and weights at strides of their own, and one product where a gradient is asked for."""
    from hipserve.ops import KernelOps

    g = torch.Generator().manual_seed(rows)
    x = torch.randn(rows, K + 8, generator=g).bfloat16().to(device)[:, 8:]
    w = torch.randn(2 * cols, K, generator=g).bfloat16().to(device)[::2].requires_grad_(grad)
    with torch.set_grad_enabled(grad):
        y = KernelOps()._vendor_linear(x, w, None)
    assert y.requires_grad == grad and y.is_contiguous()
    want = x.float() @ w.detach().float().t()
    # rounded to 2^-9, and sums of K products in 32 bits
    assert ((y.detach().float() - want).abs() <= 2.0 ** -8 * want.abs() + K * 2.0 ** -23 * (x.float().abs() @ w.detach().float().abs().t())).all()


@pytest.mark.parametrize("rows,cols,K", [(1024, 16400, 16), (2049, 8192, 2048)])   # cut by columns, by rows
@pytest.mark.parametrize("way", ["dual", "jvp", "vmap", "vmap of weights", "trace", "fx", "subclass"])
def test_products_in_whole_rounds_are_one_where_calls_are_transformed(way, rows, cols, K):
    """Forward mode, vmap, traces and tensor classes without gradients recorded: what one product does."""
    import torch.autograd.forward_ad as fw
    from torch.fx.experimental.proxy_tensor import make_fx

    from hipserve.ops import KernelOps

    class Rows(torch.Tensor):
        pass

    g = torch.Generator().manual_seed(rows)
    x, t, w = (torch.randn(*s, generator=g).bfloat16() for s in ((rows, K), (rows, K), (cols, K)))
    few, linear = x[:3], KernelOps()._vendor_linear

    def run(f):
        if way == "dual":
            with fw.dual_level():
                return fw.unpack_dual(f(fw.make_dual(x, t), w, None)).tangent
        if way == "jvp":
            return torch.func.jvp(lambda a: f(a, w, None), (x,), (t,))[1]
        if way == "vmap":
            return torch.vmap(lambda a: f(a, w, None))(x[None])
        if way == "vmap of weights":
            return torch.vmap(lambda a: f(x, a, None))(w[None])
        if way == "trace":   # of many rows, used for few
            return torch.jit.trace(lambda a: f(a, w, None), x, check_trace=False)(few)
        if way == "fx":
            return make_fx(lambda a: f(a, w, None))(x)(few)
        y = f(x.as_subclass(Rows), w, None)
        assert type(y) is Rows
        return y.as_subclass(torch.Tensor)

    with torch.no_grad():
        assert torch.equal(run(linear), run(torch.nn.functional.linear))


def test_halves_projected_apart():
    """A parallel mixer whose left half has biases and whose right half ends with an activation: two products give what parts of one do."""
    from types import SimpleNamespace

    from hipserve.models.mixers import ParallelMixer

    def linear(x, w, bias=None, act=None, act_from=0):
        y = torch.nn.functional.linear(x, w, bias)
        return y if act is None else torch.cat([y[:, :act_from], torch.tanh(y[:, act_from:])], 1)

    g = torch.Generator().manual_seed(3)
    x, outs = torch.randn(5, 16, generator=g, dtype=torch.float64), []
    for apart in (False, True):
        m = ParallelMixer.__new__(ParallelMixer)
        m.w_in, m.b_in = (torch.randn(*s, generator=torch.Generator().manual_seed(4), dtype=torch.float64) for s in ((40, 16), (40,)))
        m.split, m.left_biased, m.in_act = 24, True, dict(act="tanh", act_from=36)
        m.b_in[24:] = 0
        m.ops = SimpleNamespace(linear=linear, in_rounds=lambda x, before, cols: apart and (before, cols) == (24, 16))
        outs.append(m._project(x))
    for a, b in zip(*outs):
        assert a.shape == b.shape and torch.allclose(a, b, rtol=1e-12)


@pytest.mark.parametrize("rows,left,right,k,biased,dtype,apart", [
    (4073, 3840, 7712, 3072, True, torch.bfloat16, True), (4096, 4608, 10272, 2048, True, torch.bfloat16, False), (128, 16384, 20512, 4096, True, torch.bfloat16, False),
    (3200, 2560, 5184, 1024, True, torch.bfloat16, True), (6000, 1280, 10272, 2048, False, torch.bfloat16, True), (1500, 3072, 5152, 1024, True, torch.bfloat16, False),
    (2048, 2048, 8256, 4096, True, torch.bfloat16, True), (2048, 2048, 8256, 4096, False, torch.bfloat16, False),   # the one without biases is cut
    (33, 10240, 10336, 4096, True, torch.bfloat16, True), (8, 10240, 10336, 4096, True, torch.bfloat16, False), (16, 2048, 5184, 1024, True, torch.bfloat16, False),
    (40, 3328, 15392, 3072, True, torch.float32, True), (16, 2048, 5184, 1024, True, torch.float32, False), (789, 640, 1296, 512, False, torch.float32, False),
    (900, 1536, 5184, 1024, True, torch.float32, True), (0, 2048, 5184, 1024, True, torch.bfloat16, False), (4073, 3840, 7712, 504, True, torch.bfloat16, False),
    (4073, 3840, 7712, 3072, True, torch.float16, False)])
def test_halves_projected_apart_where_faster(rows, left, right, k, biased, dtype, apart):
    """Either side of the rules on one projection or two, at sizes that were measured, and what they leave alone."""
    from hipserve.ops import KernelOps, NormedRows

    x, ops = torch.empty(rows, k, dtype=dtype, device="meta"), KernelOps()
    assert ops.in_rounds(x, left, right, biased=biased) == apart
    if rows <= 32:
        assert ops.in_rounds(NormedRows(x, None, 1e-5), left, right, biased=biased) == apart


@gpu
@pytest.mark.parametrize("rows,rank,apart", [(1024, 96, True), (1000, 96, False), (1024, 90, True)])
def test_halves_projected_apart_in_rounds(rows, rank, apart):
    """Sizes at which the right half's product goes in whole rounds: what its rule says, and the columns of either product against 64 bits."""
    from hipserve.config import DeltaRuleSpec, ParallelMixerSpec, WindowAttentionSpec
    from hipserve.models.mixers import ParallelMixer

    ops, dev, H, N = get_ops("cuda"), torch.device("cuda"), 64, 51 * 64
    spec = ParallelMixerSpec(WindowAttentionSpec(heads=64, kv_heads=32, dim=128, vdim=128, scale=0.1, window=8, rot_dims=32, bias=True), DeltaRuleSpec(51, 64, rank))
    m = ParallelMixer(spec, H, 1e-5, dev, torch.bfloat16, ops)
    t = m.init_random(torch.Generator().manual_seed(5), 0.05)
    m.load(lambda n: t[n], "")
    h = torch.randn(rows, H, generator=torch.Generator().manual_seed(6)).to(dev, torch.bfloat16)
    assert ops.in_rounds(h, m.split, m.w_in.shape[0] - m.split) == apart
    left, right = m._project(h)
    assert (left.untyped_storage().data_ptr() != right.untyped_storage().data_ptr()) == apart
    assert left.shape == (rows, 16384) and right.shape == (rows, 5 * N + rank)
    w, b = m.w_in.double(), m.b_in.double()
    for got, at, act in ((left, 0, right.shape[1]), (right, m.split, 5 * N)):
        want = h.double() @ w[at:at + got.shape[1]].t() + b[at:at + got.shape[1]]
        want[:, act:] = torch.tanh(want[:, act:])
        assert ((got.double() - want).abs() <= 2.0 ** -7 * (want.abs() + 0.1 * want.abs().max())).all()   # as above


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rank", [3, 20, 24])
@pytest.mark.parametrize("biased", [False, True])
@pytest.mark.parametrize("rows", [1, 70])
def test_one_projection_of_both_halves_keeps_rows_aligned(rows, biased, rank, dtype, device):
    """A parallel mixer's projection whose right half ends with a bottleneck of any rank: the left half's rows stay where the wide kernels take them, and each half has the
    columns of its own product."""
    from hipserve.config import DeltaRuleSpec, ParallelMixerSpec, WindowAttentionSpec
    from hipserve.models.mixers import DeltaRule, ParallelMixer, WindowAttention
    from hipserve.ops import ReferenceOps

    ops = get_ops("cuda") if device == "cuda" else ReferenceOps()
    spec = ParallelMixerSpec(WindowAttentionSpec(heads=2, kv_heads=1, dim=64, vdim=64, scale=0.125, window=8, rot_dims=32, bias=biased), DeltaRuleSpec(2, 64, rank), 0.5, 2.0)
    dev = torch.device(device)
    m = ParallelMixer(spec, 128, 1e-5, dev, dtype, ops)
    t = m.init_random(torch.Generator().manual_seed(rank), 0.1)
    m.load(lambda n: t[n], "")
    assert m.w_in is not None
    h = torch.randn(rows, 128, generator=torch.Generator().manual_seed(rows)).to(dev, dtype)
    left, right = m._project(h)
    assert left.stride(0) * left.element_size() % 16 == 0 and left.data_ptr() % 16 == 0 and right.data_ptr() % 16 == 0
    halves = [(left, WindowAttention(spec.left, 128, 1e-5, dev, dtype, ops), "left."), (right, DeltaRule(spec.right, 128, 1e-5, dev, dtype, ops), "right.")]
    for got, half, name in halves:
        half.load(lambda n: t[n], name)
        want = h.double() @ half.w_in.double().t()
        if getattr(half, "b_in", None) is not None:
            want += half.b_in.double()
        if name == "right.":
            assert got.shape == want.shape
            want[:, 5 * 128:] = torch.tanh(want[:, 5 * 128:])
        # rounded once, and before the activation; sums of 128 products in 32 bits
        tol = 2.0 ** -7 if dtype == torch.bfloat16 else 1e-4
        assert ((got[:, :want.shape[1]].double() - want).abs() <= tol * (want.abs() + 0.1 * want.abs().max())).all()
    if device == "cuda" and rows == 1:
        cache = torch.zeros(2, 16, spec.left.cache_dim, dtype=dtype, device=dev)
        assert ops._window_lib.window_attention_decode_ok(left, cache, 64, 64)


@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,H,K", [(1, 64, 2056), (8, 2048, 4104), (9, 192, 1032), (16, 1024, 3072), (17, 2048, 520), (32, 832, 2048)])
def test_updates_in_half_tiles(M, H, K, dtype):
    """A residual update of 8 columns per workgroup: its sums, rows and squares, and the norm's factor from twice as many of them."""
    g = torch.Generator().manual_seed(M + H)
    x, w, b = torch.randn(M, K, generator=g).to(dtype), (torch.randn(H, K, generator=g) / K ** 0.5).to(dtype), torch.randn(H, generator=g).to(dtype)
    res, norm, w2 = torch.randn(M, H, generator=g) * 3, 1 + 0.1 * torch.randn(H, generator=g), (torch.randn(80, H, generator=g) / H ** 0.5).to(dtype)
    ops, out = get_ops("cuda"), []
    for cols in (8, 16):
        r, rows = res.cuda(), torch.empty(M, H, dtype=dtype, device="cuda")
        squares = torch.full((M, H // cols), float("nan"), device="cuda")
        ops._moe_lib.skinny_linear_update(rows, squares, r, norm.cuda(), x.cuda(), w.cuda(), b.cuda())
        out.append((r, rows, squares, ops.linear(NormedRows(rows, squares, 1e-6), w2.cuda())))
    (r8, rows8, s8, y8), (r16, rows16, s16, y16) = out
    assert torch.equal(r8, r16) and torch.equal(rows8, rows16)
    assert torch.allclose(s8.double().cpu().sum(1), r16.double().cpu().square().sum(1), rtol=1e-5)
    # the factors from the same squares in another order: 2^-22 of a result, which may round the other way
    assert ((y8.double() - y16.double()).abs() <= (2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -20) * y16.double().abs()).all()


@gpu
@pytest.mark.parametrize("M", [8, 9, 24, 25, 40, 41, 64])
@pytest.mark.parametrize("N", [4113, 5001, 12301])
def test_skinny_linear_wide(M, N):
    """More columns than one workgroup of 16 per compute unit: two (5001) or four (12301) tiles per workgroup, the last ones past N."""
    K = 520
    (x,), (w,) = dense_case(1, M, N, K, M + N)
    got = torch.full((M, N), 7.0, dtype=torch.bfloat16, device="cuda")
    get_ops("cuda")._moe_lib.skinny_linear(got, x.cuda(), w.cuda(), None, -1, 0.0, 0.0)
    close_to(got, x.double() @ w.double().T, x, w)


@gpu
@pytest.mark.parametrize("M,N,K", [(1, 1, 4), (3, 40, 36), (16, 16, 256), (17, 96, 260), (33, 33, 1024), (64, 48, 3076)])
def test_skinny_linear_f32(M, N, K):
    """32-bit operands: k that fills a step of 16, a wave's steps and all waves partly; bias, row strides, an activation."""
    g = torch.Generator().manual_seed(M + N + K)
    x, w, bias = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g), torch.randn(N, generator=g)
    wide = torch.zeros(M, K + 12, device="cuda")
    wide[:, 4:4 + K] = x.cuda()
    out = torch.full((M, N + 5), 7.0, device="cuda")
    get_ops("cuda")._moe_lib.skinny_linear(out[:, :N], wide[:, 4:4 + K], w.cuda(), bias.cuda(), 2, 0.0, 0.0)
    z = x.double() @ w.double().T + bias.double()
    # every one of K sums and products rounds to 2^-24 of at most the sum of magnitudes; the square doubles it
    err = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T + bias.double().abs())
    assert ((out[:, :N].double().cpu() - z.clamp_min(0) ** 2).abs() <= 2 * z.abs() * err + err ** 2 + 2.0 ** -22 * z ** 2 + 1e-9).all()
    assert (out[:, N:] == 7.0).all()


@gpu
@pytest.mark.parametrize("M", [1, 16, 31, 50])
@pytest.mark.parametrize("act,c0,c1", [("tanh", 0, 0), ("xielu", 0.8, 0.7), ("relu2", 0, 0), ("silu_mul", 0, 0), ("clamped_glu", 1.0, 0),
                                       ("softcap", 2.0, 0)])
def test_linear_with_activation(M, act, c0, c1):
    """``ops.linear`` with an activation in the kernel's epilogue, and beside it (rows past the kernel's)."""
    ops = get_ops("cuda")
    ops.norm_library = "delta"
    for rows in (M, 70):
        (x,), (w,) = dense_case(1, rows, 96, 520, M)
        z = x.double() @ w.double().T
        got = ops.linear(x.cuda(), w.cuda(), act=act, c0=c0, c1=c1)
        want = act64(z, act, c0, c1)
        if rows == M:
            assert ops.skinny_pays(M, 96, 520, act in ops.GLU_ACTS)
            close_to(got, want, x, w, scale=12.0)
        else:   # the product is rounded to bf16 before the activation, whose slope is below 12 for numbers up to 5
            assert ((got.double().cpu() - want).abs() <= 12 * 2.0 ** -8 * z.abs().max()).all()


@pytest.mark.parametrize("dev", ["cpu", pytest.param("cuda", marks=gpu)])
@pytest.mark.parametrize("M", [5, 70])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_linear_bias_of_32_bit_results(M, dtype, dev):
    """The bias is added whichever product runs."""
    (x,), (w,) = dense_case(1, M, 32, 64, M)
    x, w = x.to(dtype), w.to(dtype)
    bias = torch.randn(32, generator=torch.Generator().manual_seed(1)).to(dtype)
    got = get_ops(dev).linear(x.to(dev), w.to(dev), bias.to(dev), out_f32=True)
    assert got.dtype == torch.float32
    close_to(got, x.double() @ w.double().T + bias.double(), x, w)


@pytest.mark.parametrize("dev", ["cpu", pytest.param("cuda", marks=gpu)])
@pytest.mark.parametrize("M", [5, 70])
@pytest.mark.parametrize("form", ["one number", "every other number"])
def test_linear_bias_forms(M, form, dev):
    """A bias that is broadcast or strided is added by either product."""
    (x,), (w,) = dense_case(1, M, 32, 64, M)
    bias = torch.randn(64, generator=torch.Generator().manual_seed(2)).bfloat16().to(dev)
    bias = bias[:1] if form == "one number" else bias[::2]
    close_to(get_ops(dev).linear(x.to(dev), w.to(dev), bias), x.double() @ w.double().T + bias.cpu().double(), x, w)


@gpu
@pytest.mark.parametrize("M", [5, 70])
def test_arguments_on_another_device(M):
    """Weights, biases, tables and ids in host memory are refused, as the products and lookups of torch refuse them."""
    ops = get_ops("cuda")
    (x,), (w,) = dense_case(1, M, 32, 64, M)
    for args in ((w,), (w.cuda(), torch.zeros(32, dtype=torch.bfloat16))):
        with pytest.raises(RuntimeError):
            ops.linear(x.cuda(), *args)
    ids, table = torch.zeros(M, dtype=torch.long), torch.zeros(7, 64, dtype=torch.bfloat16)
    out, res, norm = torch.empty(M, 64, dtype=torch.bfloat16, device="cuda"), torch.empty(M, 64, device="cuda"), torch.ones(64, device="cuda")
    for lib in ("delta", "seq"):
        ops.norm_library = lib
        for t, i in ((table, ids.cuda()), (table.cuda(), ids)):
            with pytest.raises(RuntimeError):
                ops.scaled_add_group_rmsnorm(out, res, norm, 1, 1e-6, table=t, ids=i)
        slots, tiles, pairs = (torch.empty(n, dtype=torch.int32, device="cuda") for n in (256, 8, M))
        with pytest.raises(RuntimeError):
            ops.moe_table_align(torch.zeros(7, 1, dtype=torch.int32, device="cuda"), ids, 4, 32, slots, tiles, pairs)
    ops.norm_library = "delta"


@gpu
@pytest.mark.parametrize("B,M,N,K", [(3, 1, 40, 16), (16, 17, 512, 128), (5, 64, 24, 520), (2, 33, 128, 512)])
def test_skinny_heads(B, M, N, K):
    """Batches with a stride of their own: heads side by side per row, in and out."""
    x, w = dense_case(B, M, N, K, B + M)
    rows = x.transpose(0, 1).contiguous().cuda()          # [M, B, K]
    out = torch.empty(M, B, N, dtype=torch.bfloat16, device="cuda")
    assert get_ops("cuda").linear_heads(out.transpose(0, 1), rows.transpose(0, 1), w.cuda())
    close_to(out.transpose(0, 1), x.double() @ w.double().transpose(1, 2), x, w)


def test_linear_reference():
    (x,), (w,) = dense_case(1, 5, 32, 64, 0)
    ops = get_ops("cpu")
    z = x.double() @ w.double().T
    assert ops.linear(x, w, out_f32=True).dtype == torch.float32
    for act, c0 in ((None, 0), ("silu_mul", 0), ("softcap", 2.0)):
        assert (ops.linear(x.float(), w.float(), act=act, c0=c0) - act64(z, act, c0, 0)).abs().max() < 1e-5


# ------------------------------------------------------------------ experts
@gpu
@pytest.mark.parametrize("tokens,E,top", [(1, 16, 2), (2, 3, 1), (48, 16, 2), (40, 2, 2), (300, 4, 2)])
@pytest.mark.parametrize("N,K", [(64, 40), (1024, 2048), (48, 512)])
@pytest.mark.parametrize("act", [0, 1, 2, 3])
def test_expert_gemm_tiles_of_few_rows(tokens, E, top, N, K, act):
    """The weight-streaming kernel (few live slots per tile, unused tiles) and the tile kernel, gathered and not."""
    g = torch.Generator().manual_seed(tokens + N)
    x = torch.randn(tokens, K, generator=g).bfloat16()
    w = (torch.randn(E, N, K, generator=g) / K ** 0.5).bfloat16()
    ids = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(tokens)]).int()
    scale = torch.rand(tokens * top, generator=g) if act >= 2 else None
    ops, P, tile = get_ops("cuda"), tokens * top, 32
    cap = -(-(P + E * (tile - 1)) // tile) * tile
    slots, tiles, pair = (torch.empty(n, dtype=torch.int32, device="cuda") for n in (cap, cap // tile, P))
    ops.moe_align(ids.view(-1).cuda(), E, tile, slots, tiles, pair)
    out = torch.empty(cap, N // 2 if act >= 2 else N, dtype=torch.bfloat16, device="cuda")
    ops.expert_gemm(out, x.cuda(), w.cuda(), slots, tiles, tile, top, act, scale.cuda() if scale is not None else None, 1.0, P)
    xp, wp = x.repeat_interleave(top, 0), w[ids.view(-1).long()]
    z = torch.einsum("pk,pnk->pn", xp.double(), wp.double()) * (scale.double()[:, None] if scale is not None else 1.0)
    want = act64(z, {0: None, 1: "relu2", 2: "silu_mul", 3: "clamped_glu"}[act], 1.0, 0.0)
    close_to(out[pair.long()], want, x, w.view(-1, K), scale=12.0)


# ------------------------------------------------------------------ latent attention
def latent_case(lens, ctxs, heads, dim, kv, rot, block, dtype, dev, seed=0, nd=None):
    """Rows of sequences with ``lens`` rows in this step and ``ctxs`` tokens after it: random queries, a random paged cache whose
    pages lie in no order, and a meta of prompt portions first (lens > 1), ``nd`` sequences of decode rows last (the single rows)."""
    from hipserve.models.llama import AttnMeta

    g = torch.Generator().manual_seed(seed)
    T, width = sum(lens), max(-(-c // block) for c in ctxs)
    bt = torch.randperm(len(lens) * width, generator=g).int().view(len(lens), width)
    cache = torch.randn(len(lens) * width, block, kv + rot, generator=g).to(dtype)
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32)
    pos = torch.cat([torch.arange(c - n, c) for n, c in zip(lens, ctxs)])
    q_abs = torch.randn(heads, T, kv + rot, generator=g).to(dtype) * 0.3
    q = torch.randn(T, heads * (dim + rot), generator=g).to(dtype)
    proj = torch.randn(T, heads + 3, generator=g).to(dtype)
    nd = sum(n == 1 for n in lens) if nd is None else nd
    meta = AttnMeta(num_prefill_tokens=int(cu[len(lens) - nd]), num_decode=nd, positions=pos.to(dev), slot_mapping=pos.to(dev), seq_cu=cu.to(dev),
                    seq_ctx=torch.tensor(ctxs, dtype=torch.int32, device=dev), seq_bt=bt.to(dev), max_q=max(lens), max_ctx=max(ctxs))
    return cache, cu, pos, bt, q_abs, q, proj, meta


@gpu
@pytest.mark.parametrize("kv", [128, 256, 512])
@pytest.mark.parametrize("heads,window", [(16, 0), (5, 100), (70, 33)])
@pytest.mark.parametrize("lens,ctxs,nd", [([1], [1], 1), ([1, 1, 1], [64, 65, 700], 3), ([37], [37], 0), ([33, 5, 1], [33, 400, 129], 1), ([2, 190], [31, 255], 0),
                                          ([2, 0], [31, 5], 0), ([1, 0, 1], [64, 9, 700], 0), ([2, 0, 1], [31, 5, 300], 1), ([2, 0], [300, 5], 2),
                                          ([1] * 65 + [40] + [2] * 70, [5] * 65 + [60] + [3] * 70, 0), ([2] + [0] * 64 + [1], [9] * 66, 0)])
def test_latent_attention_dma(kv, heads, window, lens, ctxs, nd):
    """Tiles of 32 and 64 keys filled partly, windows that start inside a tile, rows that leave a workgroup's tiles unused, runs of
    keys of a decode row (some empty), as many rows as sequences, not one each (with runs too), more sequences than lanes, the rotary
    part formed in the kernel, in 64 bits."""
    rot, dim, block, gate, scale = 64, 24, 16, 2, 0.11
    cache, cu, pos, bt, q_abs, q, proj, meta = latent_case(lens, ctxs, heads, dim, kv, rot, block, torch.bfloat16, "cuda", kv + heads, nd)
    inv = torch.pow(torch.tensor(1e4), -2.0 * torch.arange(rot // 2) / rot)
    T = sum(lens)
    qr = q.double().view(T, heads, dim + rot)[..., dim:]
    ang = pos.double()[:, None] * inv.double()
    c, s = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    qr = torch.cat([qr[..., :32] * c - qr[..., 32:] * s, qr[..., 32:] * c + qr[..., :32] * s], -1).bfloat16().double()
    want = torch.empty(heads, T, kv, dtype=torch.float64)
    for i, (n, ctx) in enumerate(zip(lens, ctxs)):
        j = torch.arange(ctx)
        keys = cache[bt[i, j // block].long(), j % block].double()
        rows = slice(int(cu[i]), int(cu[i]) + n)
        sc = (q_abs[:, rows, :kv].double() @ keys[:, :kv].T + qr[rows].transpose(0, 1) @ keys[:, kv:].T) * scale
        back = pos[rows, None] - j
        sc = sc.masked_fill((back < 0) | (back >= window if window else back < 0), -float("inf"))
        want[:, rows] = (torch.softmax(sc, -1) @ keys[:, :kv]) * torch.sigmoid(proj[rows, gate:gate + heads].double().T)[..., None]
    ops = get_ops("cuda")
    assert ops._latent_lib.latent_attention_dma_ok(kv, rot)
    out = torch.full((heads, T, kv), float("nan"), dtype=torch.bfloat16, device="cuda")
    ops.latent_attention(out, q_abs.cuda(), q.cuda(), proj.cuda(), cache.cuda(), meta, inv.cuda(), heads, dim, rot, kv, gate, scale, window)
    # weights and outputs are rounded to bf16; a score is a sum of kv + rot products, exact to 2^-16 or so, before the exponential
    assert ((out.double().cpu() - want).abs() <= 2.0 ** -7 * want.abs() + 2.0 ** -8 * cache.double().abs().max() * 0.5).all()


# us of latent attention's decode rows by keys per run: (rows, heads, span), then by context. The first length is what the rule took before it knew the contexts
RUN_TIMES = {
    (48, 16, 1024): {150: {64: 13.2, 128: 13.8, 256: 15.4, 512: 15.4, 1024: 13.1}, 300: {64: 16.0, 128: 14.6, 256: 17.8, 512: 19.7, 1024: 17.4},
                     700: {64: 28.5, 128: 21.1, 256: 22.8, 512: 32.6, 1024: 38.4}, 1024: {64: 30.7, 128: 24.9, 256: 25.6, 512: 33.5, 1024: 52.4}},
    (16, 32, 8192): {700: {256: 20.3, 128: 20.3, 512: 26.5, 1024: 32.1}, 2000: {256: 27.0, 128: 30.2, 512: 34.2, 1024: 54.1},
                     4096: {256: 34.0, 128: 45.3, 512: 35.6, 1024: 53.0}, 8192: {256: 59.0, 128: 77.3, 512: 47.9, 1024: 59.9}},
    (16, 64, 4096): {700: {256: 22.2, 128: 24.5, 512: 26.5, 1024: 32.1}, 2000: {256: 32.3, 128: 41.4, 512: 34.9, 1024: 54.1}, 4096: {256: 51.5, 128: 71.9, 512: 42.1, 1024: 53.9}},
    (64, 64, 1024): {60: {256: 16.9, 128: 23.2, 512: 13.8, 1024: 9.1}, 300: {256: 28.7, 128: 39.8, 512: 26.6, 1024: 20.5}, 1024: {256: 54.0, 128: 76.0, 512: 43.6, 1024: 50.7}},
    (1, 16, 1024): {60: {64: 9.9, 128: 9.7, 256: 9.6, 512: 9.6, 1024: 7.6}, 300: {64: 10.1, 128: 11.6, 256: 15.7, 512: 18.7, 1024: 16.2},
                    1024: {64: 10.1, 128: 11.8, 256: 16.4, 512: 25.0, 1024: 39.1}}}


@pytest.mark.parametrize("size", sorted(RUN_TIMES))
def test_latent_runs_of_contexts_below_the_span(size):
    """A captured step's span is a bound: the run length is not one that contexts far below it pay for."""
    from hipserve.ops import KernelOps

    part, gain = KernelOps._latent_run(*size), 1.0
    for us in RUN_TIMES[size].values():
        before = next(iter(us.values()))
        assert us[part] <= 1.1 * before, (part, us)
        gain *= us[part] / before
    assert gain <= 1.0


@pytest.mark.parametrize("rows,heads,span", [(0, 16, 0), (1, 1, 1), (1, 16, 128), (64, 128, 1 << 17)])
def test_latent_runs_of_any_size(rows, heads, span):
    from hipserve.ops import KernelOps

    assert KernelOps._latent_run(rows, heads, span) in (64, 128, 256, 512)


@gpu
@pytest.mark.parametrize("part", [64, 128, 192, 256, 512])
def test_latent_decode_runs(part):
    """Contexts that end one key before, at and behind the runs' ends, and a span that leaves runs empty, in 64 bits; a length that is no power of two."""
    kv, heads, rot, dim, block, scale, span = 512, 20, 64, 24, 16, 0.11, 2048
    ctxs = [1, part - 1, part, part + 1, 2 * part, 2 * part + 1, 3 * part + 33]
    lens = [1] * len(ctxs)
    cache, cu, pos, bt, q_abs, q, proj, meta = latent_case(lens, ctxs, heads, dim, kv, rot, block, torch.bfloat16, "cuda", part)
    meta.max_ctx = span
    inv = torch.zeros(rot // 2)   # no rotation
    want = torch.empty(heads, len(ctxs), kv, dtype=torch.float64)
    for i, ctx in enumerate(ctxs):
        j = torch.arange(ctx)
        keys = cache[bt[i, j // block].long(), j % block].double()
        sc = (q_abs[:, i, :kv].double() @ keys[:, :kv].T + q[i].double().view(heads, dim + rot)[:, dim:] @ keys[:, kv:].T) * scale
        want[:, i] = torch.softmax(sc, -1) @ keys[:, :kv]
    ops = type(get_ops("cuda"))()
    ops.latent_run = lambda rows, heads, span: part
    out = torch.full((heads, len(ctxs), kv), float("nan"), dtype=torch.bfloat16, device="cuda")
    ops.latent_attention(out, q_abs.cuda(), q.cuda(), proj.cuda(), cache.cuda(), meta, inv.cuda(), heads, dim, rot, kv, -1, scale, 0)
    # as in test_latent_attention_dma
    assert ((out.double().cpu() - want).abs() <= 2.0 ** -7 * want.abs() + 2.0 ** -8 * cache.double().abs().max() * 0.5).all()


@gpu
@pytest.mark.parametrize("heads,gate,window,lens,ctxs", [
    (3, "head", 0, [130], [130]), (4, "head", 50, [70, 1, 33, 200], [70, 9, 64, 331]), (2, "channel", 33, [31, 128, 129], [31, 128, 400]),
    (2, "none", 0, [3] * 70, [5] * 70), (16, "head", 64, [2000, 0, 2097], [2000, 0, 2100]), (1, "head", 1, [65, 64], [65, 80])])
def test_latent_prompt_attention(heads, gate, window, lens, ctxs):
    """Cache rows side by side (all that a window shows, sequences without rows, more sequences than lanes), and attention to formed
    keys and values: tiles filled partly, waves that leave tiles out, both row counts per wave, in 64 bits."""
    D, rot, kv, block, scale = 128, 64, 32, 16, 0.07
    dim = kv + rot
    cache, cu, pos, bt, _, _, _, meta = latent_case(lens, ctxs, heads, D, kv, rot, block, torch.bfloat16, "cuda", heads + window)
    lib, g, T = get_ops("cuda")._latent_lib, torch.Generator().manual_seed(window), sum(lens)
    seen = [ctx - max(0, ctx - n - window + 1 if window else 0) if n else 0 for n, ctx in zip(lens, ctxs)]
    rows = sum(seen) + 5
    lat = torch.zeros(rows, dim, dtype=torch.bfloat16, device="cuda")
    off = torch.empty(len(lens) + 1, dtype=torch.int32, device="cuda")
    lib.latent_gather(lat, off, cache.cuda(), meta.seq_cu, meta.seq_ctx, meta.seq_bt, window)
    assert off.tolist() == [sum(seen[:i]) for i in range(len(lens) + 1)]
    q, kvs = torch.randn(T, heads * (D + rot), generator=g).bfloat16(), torch.randn(rows, 2 * heads * D, generator=g).bfloat16()
    proj = torch.randn(T, 8 + heads * D, generator=g).bfloat16()
    inv = torch.pow(torch.tensor(1e4), -2.0 * torch.arange(rot // 2) / rot)
    out = torch.full((T, heads * D), float("nan"), dtype=torch.bfloat16, device="cuda")
    lib.latent_prompt_attention(out, q.cuda(), kvs.cuda(), lat, off, meta.seq_cu, meta.seq_ctx, pos.cuda(), inv.cuda(), proj.cuda(), heads,
                                -1 if gate == "none" else 8, gate == "channel", scale, window)
    qh = q.double().view(T, heads, D + rot)
    ang = pos.double()[:, None] * inv.double()
    c, s, r = torch.cos(ang)[:, None], torch.sin(ang)[:, None], qh[..., D:]
    qr = torch.cat([r[..., :32] * c - r[..., 32:] * s, r[..., 32:] * c + r[..., :32] * s], -1).bfloat16().double()
    qh, lat = torch.cat([qh[..., :D], qr], -1), lat.cpu()
    want = torch.empty(T, heads, D, dtype=torch.float64)
    for i, (n, ctx) in enumerate(zip(lens, ctxs)):
        j, at = torch.arange(ctx - seen[i], ctx), slice(sum(seen[:i]), sum(seen[:i + 1]))
        assert torch.equal(lat[at], cache[bt[i, j // block].long(), j % block])
        k, v = kvs[at].double().view(-1, 2, heads, D).unbind(1)
        k = torch.cat([k, lat[at, None, kv:].double().expand(-1, heads, -1)], -1)
        mine = slice(int(cu[i]), int(cu[i]) + n)
        back = pos[mine, None] - j
        for h in range(heads):
            sc = (qh[mine, h] @ k[:, h].T * scale).masked_fill((back < 0) | (back >= window if window else back < 0), -float("inf"))
            want[mine, h] = torch.softmax(sc, -1) @ v[:, h]
    if gate != "none":
        gates = torch.sigmoid(proj[:, 8:8 + heads * (D if gate == "channel" else 1)].double()).view(T, heads, -1)
        want *= gates
    # weights and outputs are rounded to bf16; a score is a sum of 192 products, exact to 2^-16 or so, before the exponential
    assert ((out.double().cpu().view(T, heads, D) - want).abs() <= 2.0 ** -7 * want.abs() + 2.0 ** -8 * kvs.double().abs().max() * 0.5).all()


def test_latent_weights_are_laid_out_at_load():
    from types import SimpleNamespace

    from hipserve.config import LatentAttentionSpec
    from hipserve.models.mixers import LatentAttention
    spec = LatentAttentionSpec(heads=2, dim=8, rot_dim=4, vdim=8, q_rank=8, kv_rank=16, scale=0.1)
    for in_place in (True, False):
        m = LatentAttention(spec, 32, 1e-6, "cpu", torch.bfloat16, SimpleNamespace(latent_query_in_place=lambda *a: in_place))
        m.init_random(torch.Generator().manual_seed(0), 0.02)
        assert (m.w_uk_t is not None) == (m.w_uk_wide is not None) == in_place
        if in_place:
            assert torch.equal(m.w_uk_t.transpose(1, 2), m.w_uk) and torch.equal(m.w_uk_wide[..., :16], m.w_uk) and not m.w_uk_wide[..., 16:].any()


def test_latent_weights_of_other_sizes_are_refused():
    """W_uk and W_uv lie side by side in one allocation: rows that one has too many must not become the other's."""
    from types import SimpleNamespace

    from hipserve.config import LatentAttentionSpec
    from hipserve.models.mixers import LatentAttention
    spec = LatentAttentionSpec(heads=2, dim=8, rot_dim=4, vdim=12, q_rank=8, kv_rank=16, scale=0.1)
    m = LatentAttention(spec, 32, 1e-6, "cpu", torch.float32, SimpleNamespace(latent_query_in_place=lambda *a: False))
    t = m.init_random(torch.Generator().manual_seed(0), 0.02)
    m.load(t.__getitem__, "")
    assert torch.equal(m.w_uk.flatten(0, 1), t["uk"].view(-1, 16)) and torch.equal(m.w_uv.flatten(0, 1), t["uv"].view(-1, 16))
    both = torch.cat([t["uk"].view(-1, 16), t["uv"].view(-1, 16)])
    for rows in (24, 17):   # the two exchanged, a row of one with the other
        wrong = dict(t, uk=both[:rows], uv=both[rows:])
        with pytest.raises(RuntimeError):
            m.load(wrong.__getitem__, "")


@gpu
@pytest.mark.parametrize("kv", [128, 512])
@pytest.mark.parametrize("n,ctx,window", [(3, 100, 40), (4, 64, 33), (2, 200, 64)])
def test_latent_attention_hidden_keys(kv, n, ctx, window):
    """Keys before the first row's window, which no row sees, may hold anything."""
    heads, dim, rot = 8, 24, 64
    cache, cu, pos, bt, q_abs, q, proj, meta = latent_case([n], [ctx], heads, dim, kv, rot, 16, torch.bfloat16, "cuda", ctx, 0)
    j = torch.arange(ctx - n - window + 1)
    outs = []
    for value in (0.0, float("nan"), float("inf")):
        cache[bt[0, j // 16].long(), j % 16] = value
        outs.append(torch.empty(heads, n, kv, dtype=torch.bfloat16, device="cuda"))
        get_ops("cuda").latent_attention(outs[-1], q_abs.cuda(), q.cuda(), proj.cuda(), cache.cuda(), meta, torch.zeros(rot // 2, device="cuda"), heads, dim,
                                         rot, kv, -1, 0.1, window)
    assert outs[0].isfinite().all() and torch.equal(outs[1], outs[0]) and torch.equal(outs[2], outs[0])


def tiled_softmax(sc, v, sink=False, tile=32):
    """softmax(sc) . v as the matrix-core kernels do it, in 64 bits but for bf16 weights relative to the maximum so far."""
    m = torch.full((sc.shape[0], 1), 0.0 if sink else -float("inf"), dtype=torch.float64)
    l, acc = torch.full_like(m, float(sink)), torch.zeros(sc.shape[0], v.shape[1], dtype=torch.float64)
    for j in range(0, sc.shape[1], tile):
        s = sc[:, j:j + tile]
        mn = torch.maximum(m, s.amax(1, keepdim=True))
        al = torch.where(mn > -float("inf"), torch.exp(m - mn), 1.0)
        p = torch.exp(s - torch.where(mn > -float("inf"), mn, 0.0)).bfloat16().double()
        m, l, acc = mn, l * al + p.sum(1, keepdim=True), acc * al + p @ v[j:j + tile]
    return acc / l


def no_further(got, rounded, want):
    """The kernel's bf16 outputs are as far from 64 bits as weights relative to the row's maximum make them."""
    ours, theirs = ((x.double().cpu() - want).norm() / want.norm() for x in (got, rounded.bfloat16()))
    assert ours <= 1.02 * theirs, (ours, theirs)   # sums in other orders, exponentials: a few of the roundings fall otherwise


@gpu
@pytest.mark.parametrize("kv,size", [(512, 2.0), (128, 1.0), (256, 3.0)])
def test_latent_attention_prompt_error(kv, size):
    rot, dim, heads, n, scale = 64, 24, 8, 300, (kv + 64) ** -0.5
    cache, cu, pos, bt, q_abs, q, proj, meta = latent_case([n], [n], heads, dim, kv, rot, 16, torch.bfloat16, "cuda", kv)
    q_abs, q = (q_abs.float() * size / 0.3).bfloat16(), (q.float() * size).bfloat16()
    out = torch.empty(heads, n, kv, dtype=torch.bfloat16, device="cuda")
    get_ops("cuda").latent_attention(out, q_abs.cuda(), q.cuda(), proj.cuda(), cache.cuda(), meta, torch.zeros(rot // 2, device="cuda"), heads, dim, rot,
                                     kv, -1, scale, 0)
    j = torch.arange(n)
    keys = cache[bt[0, j // 16].long(), j % 16].double()
    qr = q.double().view(n, heads, dim + rot)[..., dim:]
    want, rounded = torch.empty(2, heads, n, kv, dtype=torch.float64)
    for h in range(heads):
        sc = (q_abs[h, :, :kv].double() @ keys[:, :kv].T + qr[:, h] @ keys[:, kv:].T) * scale
        sc = sc.masked_fill(j > j[:, None], -float("inf"))
        want[h], rounded[h] = torch.softmax(sc, -1) @ keys[:, :kv], tiled_softmax(sc, keys[:, :kv])
    no_further(out, rounded, want)


@gpu
@pytest.mark.parametrize("dim,size,sink", [(128, 1.5, True), (128, 1.0, False), (64, 1.5, True)])
def test_window_attention_prompt_error(dim, size, sink):
    from types import SimpleNamespace
    g = torch.Generator().manual_seed(dim)
    heads, kv, n, bs = 8, 2, 300, 16
    sp = SimpleNamespace(maps=1, dim=dim, vdim=dim, heads=heads, kv_heads=kv, window=0, reach=0, scale=dim ** -0.5, sink=sink, keep_first=0,
                         softcap=0.0, channel_gate=False, chunk=0, diff=0.0)
    pages = -(-n // bs)
    cache, proj = torch.randn(pages, bs, 2 * kv * dim, generator=g), (torch.randn(n, heads * dim, generator=g) * size).bfloat16()
    cache[..., :kv * dim] *= size
    cache = cache.bfloat16()
    meta = SimpleNamespace(seq_cu=torch.tensor([0, n]).int().cuda(), seq_ctx=torch.tensor([n]).int().cuda(), seq_bt=torch.arange(pages).int().view(1, -1).cuda(),
                           num_decode=0, num_prefill_tokens=n, max_ctx=n)
    out = torch.empty(n, heads * dim, dtype=torch.bfloat16, device="cuda")
    get_ops("cuda").window_attention(out, proj.cuda(), cache.cuda(), meta, sp, -1)
    rows, j = cache.double().view(-1, 2 * kv, dim)[:n], torch.arange(n)
    want, rounded = torch.empty(2, n, heads, dim, dtype=torch.float64)
    for h in range(heads):
        k, v = rows[:, h // (heads // kv)], rows[:, kv + h // (heads // kv)]
        sc = (proj[:, h * dim:(h + 1) * dim].double() @ k.T * sp.scale).masked_fill(j > j[:, None], -float("inf"))
        full = torch.cat([sc, torch.zeros(n, 1, dtype=torch.float64)], 1) if sink else sc
        want[:, h], rounded[:, h] = torch.softmax(full, -1)[:, :n] @ v, tiled_softmax(sc, v, sink)
    no_further(out, rounded.view(n, -1), want.view(n, -1))


# ------------------------------------------------------------------ minGRU
@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,width,K,gaps", [(1, 16, 64, ()), (3, 40, 520, (0, 2)), (16, 260, 1024, ()), (17, 1028, 136, (5,)), (41, 64, 2048, (41,)), (64, 30, 256, ())])
def test_mingru_product(M, width, K, gaps, dtype):
    """The decode step in its product's epilogue: every row group, channels that fill no tile, sequences without a row, fresh states."""
    g = torch.Generator().manual_seed(M + width)
    lens = [1] * M
    for i in gaps:
        lens.insert(i, 0)
    n = len(lens)
    wide = torch.randn(M, K + 16, generator=g).to(dtype)
    x, w = wide[:, 8:8 + K], (torch.randn(3 * width, K, generator=g) / K ** 0.5).to(dtype)
    state, bz, bx = torch.randn(n + 2, width, generator=g), torch.randn(width, generator=g), torch.randn(width, generator=g)
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32)
    ctx = torch.tensor([m + (7 if i % 2 else 0) for i, m in enumerate(lens)], dtype=torch.int32)
    slots = torch.randperm(n + 2, generator=g)[:n].int()
    want_s, want = state.clone(), torch.empty(M, width)
    ref.mingru_scan(want, want_s, (x.double() @ w.double().T).float(), bz, bx, cu, ctx, slots)
    got_s, got = state.cuda(), torch.empty(M, width, dtype=dtype, device="cuda")
    get_ops("cuda")._seq.mingru_product(got, got_s, wide.cuda()[:, 8:8 + K], w.cuda(), bz.cuda(), bx.cuda(), cu.cuda(), ctx.cuda(), slots.cuda())
    # 32-bit sums of K products, and slopes of at most a few
    err = 16 * K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T).max() + 64 * 2.0 ** -24 * 6
    assert (got_s.cpu() - want_s).abs().max() < err
    assert ((got.cpu().float() - want).abs() <= (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -18) * want.abs() + 8 * err).all()


@gpu
@pytest.mark.parametrize("M,width,K", [(1, 2048, 1024), (3, 4101, 2056), (4, 4096, 2048), (8, 1030, 1032), (9, 2041, 2048), (16, 1999, 1096)])
def test_mingru_product_of_8_channels(M, width, K):
    """Workgroups of 8 channels for up to 16 rows: the bits that the same rows have among more of them, which take 16; a last workgroup that is partly filled, k
    past a whole piece, a sequence without a row."""
    g = torch.Generator("cuda").manual_seed(M + width)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    x, w, state, bz, bx = rand(20, K).bfloat16(), (rand(3 * width, K) / K ** 0.5).bfloat16(), rand(24, width), rand(width), rand(width)
    seq = torch.randperm(24, device="cuda", generator=g)[:21].int()
    cu = torch.tensor([0, 0, *range(1, 21)], dtype=torch.int32, device="cuda")   # the first sequence has no row
    ctx = torch.arange(21, dtype=torch.int32, device="cuda") % 3 + 1
    outs = []
    for n in (M, 20):
        y, s = torch.full((n, width), float("nan"), dtype=torch.bfloat16, device="cuda"), state.clone()
        get_ops("cuda")._seq.mingru_product(y, s, x[:n], w, bz, bx, cu[:n + 2], ctx[:n + 1], seq[:n + 1])
        outs.append((y[:M], s[seq[1:M + 1].long()], s[seq[:1].long()]))
    assert all(torch.equal(a, b) for a, b in zip(*outs))


@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("width", [4, 260, 1028, 6])
@pytest.mark.parametrize("lens", [[1], [1, 1, 1], [17], [16, 1, 256], [1, 300, 63]])
def test_mingru_blocks(lens, width, dtype):
    """Single rows, waves of 16 rows and blocks of 256 (full, partly filled, several), fresh and carried states, beside the reference scan."""
    g = torch.Generator().manual_seed(sum(lens) + width)
    T, n = sum(lens), len(lens)
    proj = torch.randn(T, 3 * width, generator=g).to(dtype)
    state, bz, bx = torch.randn(n + 2, width, generator=g), torch.randn(width, generator=g), torch.randn(width, generator=g)
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32)
    ctx = torch.tensor([m + (7 if i % 2 else 0) for i, m in enumerate(lens)], dtype=torch.int32)
    slots = torch.randperm(n + 2, generator=g)[:n].int()
    want_s, want = state.clone(), torch.empty(T, width, dtype=dtype)
    ref.mingru_scan(want, want_s, proj, bz, bx, cu, ctx, slots)
    got_s, got = state.cuda(), torch.empty(T, width, dtype=dtype, device="cuda")
    get_ops("cuda")._seq.mingru_scan(got, got_s, proj.cuda(), bz.cuda(), bx.cuda(), cu.cuda(), ctx.cuda(), slots.cuda(), max(lens))
    # every row averages the state with a bounded candidate: errors do not grow with the rows
    assert (got_s.cpu() - want_s).abs().max() < 64 * 2.0 ** -24 * 6
    tol = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -18
    assert ((got.cpu().float() - want.float()).abs() <= tol * want.float().abs() + 1e-5).all()


@gpu
@pytest.mark.parametrize("rows", [9, 77, 600])
def test_mingru_state_error(rows):
    """The state is as far from 64 bits as a recurrence that rounds z, z c and S once per row."""
    g = torch.Generator().manual_seed(rows)
    width = 8192
    proj, S0 = torch.randn(rows, 3 * width, generator=g), torch.randn(1, width, generator=g)
    bz, bx = torch.randn(width, generator=g), torch.randn(width, generator=g)
    z = torch.sigmoid((proj[:, :width] + bz).double())
    u = (proj[:, width:2 * width] + bx).double()
    c = torch.where(u >= 0, u + 0.5, torch.sigmoid(u))
    z32 = z.float()
    zc32 = (z32 * c.float())
    want, rounded = S0[0].double(), S0[0].double()
    for t in range(rows):
        want = want + z[t] * (c[t] - want)
        rounded = ((1 - z32[t]).double() * rounded + zc32[t].double()).float().double()
    got, y = S0.cuda(), torch.empty(rows, width, device="cuda")
    get_ops("cuda")._seq.mingru_scan(y, got, proj.cuda(), bz.cuda(), bx.cuda(), torch.tensor([0, rows]).int().cuda(), torch.tensor([rows + 1]).int().cuda(),
                                     torch.zeros(1).int().cuda(), rows)
    ours, theirs = (got[0].cpu().double() - want).norm(), (rounded - want).norm()
    assert ours <= 1.1 * theirs, (ours, theirs)   # the kernel's own sigmoids make it 1.04, another rounding of S 1.16


# ------------------------------------------------------------------ experts by token
@gpu
@pytest.mark.parametrize("tokens,top", [(1, 2), (48, 3), (3000, 2)])
def test_moe_table_align(tokens, top):
    g = torch.Generator().manual_seed(tokens)
    E, tile, V = 9, 32, 40
    table = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(V)]).int()
    ids = torch.randint(0, V, (tokens,), generator=g)
    P = tokens * top
    cap = -(-(P + E * (tile - 1)) // tile) * tile
    ops = get_ops("cuda")
    slots, tiles, pair = (torch.empty(n, dtype=torch.int32, device="cuda") for n in (cap, cap // tile, P))
    ops.moe_table_align(table.cuda(), ids.cuda(), E, tile, slots, tiles, pair)
    experts = table[ids].view(-1)
    assert torch.equal(tiles.cpu()[pair.cpu().long() // tile], experts)          # a pair's slot lies in a tile of its expert
    assert torch.equal(slots.cpu()[pair.cpu().long()], torch.arange(P).int())    # and the slot names the pair
    assert int((slots >= 0).sum()) == P


@gpu
@pytest.mark.parametrize("P", [1024, 1025, 4096, 4097, 16383, 65536, 65537])
@pytest.mark.parametrize("E,tile", [(5, 128), (128, 16)])
def test_moe_align_sizes(P, E, tile):
    """One pair per thread and more, many workgroups of 1024 and 4096 pairs: the pairs of an expert in its tiles, the experts' tiles in order, nothing
    else; looked up in a table as well, its tiles counted, and several tables by a workgroup each."""
    g = torch.Generator().manual_seed(P + E)
    table, tokens = torch.randint(0, E, (50, 1), generator=g).int(), torch.randint(0, 50, (P,), generator=g)
    experts, ops = table[tokens].view(-1), get_ops("cuda")
    counts = torch.bincount(experts.long(), minlength=E)
    labels = torch.repeat_interleave(torch.arange(E), (counts + tile - 1) // tile).int()
    cap = -(-(P + E * (tile - 1)) // tile) * tile

    def check(slots, tiles, pair):
        slots, tiles, pair = slots.cpu(), tiles.cpu(), pair.cpu().long()
        assert torch.equal(slots[pair], torch.arange(P).int()) and int((slots == -1).sum()) == cap - P
        assert torch.equal(tiles[:len(labels)], labels) and bool((tiles[len(labels):] == -1).all()) and torch.equal(tiles[pair // tile], experts)
    made = lambda *n: [torch.full((*n, k), 7, dtype=torch.int32, device="cuda") for k in (cap, cap // tile, P)]  # noqa: E731
    out = made()
    ops.moe_align(experts.cuda(), E, tile, *out)
    check(*out)
    if P <= 16384:
        out, count = made(), torch.empty(1, dtype=torch.int32, device="cuda")
        ops.moe_table_align(table.cuda(), tokens.cuda(), E, tile, *out, count)
        check(*out)
        assert int(count) == len(labels)
        out = made(2)
        ops.moe_table_align(torch.stack([table] * 2).cuda(), tokens.cuda(), E, tile, *out)
        for i in range(2):
            check(*(x[i] for x in out))


@gpu
@pytest.mark.parametrize("tokens,top", [(1, 2), (48, 3), (1500, 2)])
def test_moe_table_align_of_layers(tokens, top):
    """Every table's tiles in one launch, as one by one."""
    g = torch.Generator().manual_seed(tokens)
    L, E, tile, V = 3, 9, 32, 40
    tables = torch.stack([torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(V)]) for _ in range(L)]).int()
    ids = torch.randint(0, V, (tokens,), generator=g)
    P = tokens * top
    cap = -(-(P + E * (tile - 1)) // tile) * tile
    ops = get_ops("cuda")
    assert ops.moe_tables_align_ok(tables, ids, E)
    slots, tiles, pair = (torch.empty(L, n, dtype=torch.int32, device="cuda") for n in (cap, cap // tile, P))
    ops.moe_table_align(tables.cuda(), ids.cuda(), E, tile, slots, tiles, pair)
    for i in range(L):
        experts = tables[i][ids].view(-1)
        assert torch.equal(tiles[i].cpu()[pair[i].cpu().long() // tile], experts)
        assert torch.equal(slots[i].cpu()[pair[i].cpu().long()], torch.arange(P).int())
        assert int((slots[i] >= 0).sum()) == P


def test_moe_tables_of_layers_after_a_reload():
    """A layer that loads another table after the tables were stacked is not aligned by what it had before."""
    from types import SimpleNamespace

    from hipserve.config import TableMoESpec
    from hipserve.models.mixers import TableMoE
    calls = []
    ops = SimpleNamespace(name="stub", moe_tables_align_ok=lambda *a: True, moe_table_align=lambda tables, *a: calls.append(tables.clone()))
    layers = [TableMoE(TableMoESpec(experts=4, top=2, ff=8), 16, 40, "cpu", torch.float32, ops) for _ in range(3)]
    g = torch.Generator().manual_seed(0)
    for m in layers:
        m.init_random(g, 0.02)
    tables = TableMoE.stack(layers)
    h, ids = torch.zeros(5, 16), torch.arange(5)
    assert len(TableMoE.align(layers, tables, h, ids)) == 3 and torch.equal(calls[0], torch.stack([m.table for m in layers]))
    for i in range(3):
        TableMoE.stack(layers)   # of its own: `tables` is no longer what the layers hold
        assert TableMoE.align(layers, tables, h, ids) is None
        tables = TableMoE.stack(layers)
        assert TableMoE.align(layers, tables, h, ids) is not None
        layers[i].init_random(g, 0.02)
        assert TableMoE.align(layers, tables, h, ids) is None
    assert len(calls) == 4


# ------------------------------------------------------------------ queries, keys and values of window attention
@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads,kv,maps,dim,vdim,nfreq", [
    (1, 1, 1, 16, 16, 8), (4, 2, 1, 64, 128, 16), (3, 1, 2, 128, 32, 64), (32, 8, 1, 128, 128, 32), (64, 4, 1, 128, 128, 64),
    (2, 1, 1, 1024, 256, 0), (5, 1, 1, 32, 512, 16), (2, 1, 1, 48, 64, 8), (2, 2, 1, 64, 64, 12), (130, 2, 1, 128, 128, 8)])
@pytest.mark.parametrize("mode,v_norm,own", [(0, False, True), (1, True, True), (2, False, True), (3, True, True), (2, False, False)])
def test_attn_prepare(heads, kv, maps, dim, vdim, nfreq, mode, v_norm, own, dtype):
    """One item of 16 dims to two per thread, heads whose values do not start at a multiple of their size, each norm, rows
    without a slot, and sizes of the general kernel."""
    from types import SimpleNamespace
    g = torch.Generator().manual_seed(heads * dim + mode)
    T, nq, nk, nv = 5, heads * maps * dim, kv * maps * dim, kv * vdim
    proj = torch.randn(T, nq + (nk + nv if own else 0) + 16, generator=g).to(dtype)
    cache = torch.zeros(2, 16, nk + nv, dtype=dtype)
    inv = 1e4 ** (-torch.arange(nfreq).float() / max(nfreq, 1))
    positions, slots = torch.tensor([0, 1, 77, 4000, 16000]), torch.tensor([3, -1, 31, 0, 7])
    n = {1: (nq, nk), 2: (dim, dim)}.get(mode)
    w = [torch.rand(m, generator=g) + 0.5 for m in n] if n else [None, None]
    amp, eps = 1.25, 1e-5
    sp = SimpleNamespace(q_size=nq, k_size=nk, v_size=nv, heads=heads, kv_heads=kv, maps=maps, dim=dim, vdim=vdim, kv_from=None if own else 0,
                         qk_norm=mode == 1, head_norm=mode == 2, unit_qk=mode == 3, v_norm=v_norm, temp_coef=0.1, temp_every=64,
                         scaling=SimpleNamespace(amplitude=amp))
    meta = SimpleNamespace(positions=positions.cuda(), slot_mapping=slots.cuda())
    p, c = proj.cuda(), cache.cuda()
    get_ops("cuda").attn_prepare(p, c, meta, inv.cuda(), sp, *[v if v is None else v.cuda() for v in w], eps)
    ref.attn_prepare(proj, cache, positions, slots, inv, sp, w[0], w[1], eps)
    # 32-bit: sums of squares and a product or two; an angle of up to 16000 rounds to 2^-10.
    tol = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -18
    for got, want in ((p.cpu().float(), proj.float()), (c.cpu().float(), cache.float())):
        assert ((got - want).abs() <= tol * want.abs() + (2.0 ** -9 if nfreq else 2.0 ** -20) * want.abs().max()).all()


@gpu
def test_attn_prepare_norm_error():
    """How far the heads' norms are from 64 bits: their mean relative error over a head, in which its elements' own roundings cancel."""
    from types import SimpleNamespace
    heads, kv, dim, T = 16, 4, 128, 2000
    proj = torch.randn(T, (heads + 2 * kv) * dim, generator=torch.Generator().manual_seed(3))
    sp = SimpleNamespace(q_size=heads * dim, k_size=kv * dim, v_size=kv * dim, heads=heads, kv_heads=kv, maps=1, dim=dim, vdim=dim, kv_from=None,
                         qk_norm=False, head_norm=True, unit_qk=False, v_norm=True, temp_coef=0.0, temp_every=0, scaling=None)
    meta = SimpleNamespace(positions=torch.zeros(T, dtype=torch.long, device="cuda"), slot_mapping=torch.arange(T, device="cuda"))
    p, cache, one = proj.cuda(), torch.zeros(T, 1, 2 * kv * dim, device="cuda"), torch.ones(dim, device="cuda")
    get_ops("cuda").attn_prepare(p, cache, meta, torch.empty(0, device="cuda"), sp, one, one, 1e-6)
    got = torch.cat([p[:, :heads * dim].cpu(), cache.view(T, -1).cpu()], 1).double().view(T, -1, dim)
    want = proj.double().view(T, -1, dim)
    want = want * torch.rsqrt(want.square().mean(-1, keepdim=True) + 1e-6)
    off = (got * want).sum(-1) / want.square().sum(-1) - 1
    # 4.56e-8 over 48000 heads, nearly all of it from the root and the quotient; a single chain of 16 squares per thread makes it 4.63e-8
    assert off.square().mean().sqrt() <= 4.6e-8


# ------------------------------------------------------------------ window attention of decode rows
@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads,kv,dim,ctxs,opts", [
    (1, 1, 64, [1], {}), (4, 1, 128, [1, 31, 32, 33, 700], {"window": 0}), (8, 2, 128, [16, 17, 300, 257], {"window": 256, "sink": True, "gate": True}),
    (40, 2, 64, [5, 129, 400], {"window": 100, "keep_first": 7, "softcap": 3.0, "channel_gate": True}),
    (32, 2, 128, [64, 65, 1500], {"chunk": 64, "sink_w": True}), (16, 1, 256, [3, 290], {"window": 0}), (16, 1, 128, [300], {"window": 0})])
def test_window_attention_decode(heads, kv, dim, ctxs, opts, dtype):
    """One key, runs that end inside a tile, several runs, more than 16 heads per key / value head, and every mask and gate."""
    from types import SimpleNamespace
    g = torch.Generator().manual_seed(heads * dim)
    n, bs, gate = len(ctxs), 8, opts.get("gate", False) or opts.get("channel_gate", False)
    sp = SimpleNamespace(maps=1, dim=dim, vdim=dim, heads=heads, kv_heads=kv, window=opts.get("window", 0), scale=dim ** -0.5, sink=opts.get("sink", "sink_w" in opts),
                         keep_first=opts.get("keep_first", 0), softcap=opts.get("softcap", 0.0), channel_gate=opts.get("channel_gate", False),
                         chunk=opts.get("chunk", 0), diff=0.0, q_size=heads * dim, k_size=kv * dim, v_size=kv * dim, kv_from=None)
    sp.reach = sp.window + sp.keep_first if sp.window > 0 else sp.chunk
    width = -(-max(ctxs) // bs)
    bt = torch.randperm(n * width, generator=g).int().view(n, width)
    cache = torch.randn(n * width, bs, 2 * kv * dim, generator=g).to(dtype)
    gate_off = heads * dim
    proj = torch.randn(n, heads * dim + heads * dim, generator=g).to(dtype)
    sink_w = torch.randn(heads, generator=g) if opts.get("sink_w") else None
    cu, ctx = torch.arange(n + 1).int(), torch.tensor(ctxs, dtype=torch.int32)
    want = torch.empty(n, heads * dim, dtype=torch.float64)
    rows = cache.double().view(-1, 2 * kv, dim)
    for s in range(n):
        p = ctxs[s] - 1
        lo = p - p % sp.chunk if sp.chunk else max(0, p - sp.window + 1) if sp.window else 0
        js = sorted(set(range(lo, p + 1)) | (set(range(min(sp.keep_first, p + 1))) if sp.window else set()))
        kv_rows = rows[[int(bt[s, j // bs]) * bs + j % bs for j in js]]
        for h in range(heads):
            k, v = kv_rows[:, h // (heads // kv)], kv_rows[:, kv + h // (heads // kv)]
            x = k @ proj[s, h * dim:(h + 1) * dim].double() * sp.scale
            if sp.softcap:
                x = sp.softcap * torch.tanh(x / sp.softcap)
            extra = torch.tensor([float(sink_w[h]) if sink_w is not None else 0.0]).double() if sp.sink else torch.empty(0).double()
            w = torch.softmax(torch.cat([x, extra]), 0)[:len(js)]
            want[s, h * dim:(h + 1) * dim] = w @ v
    if gate:
        gates = torch.sigmoid(proj[:, gate_off:gate_off + (heads * dim if sp.channel_gate else heads)].double())
        want *= gates if sp.channel_gate else gates.repeat_interleave(dim, 1)
    ops = get_ops("cuda")
    meta = SimpleNamespace(seq_ctx=ctx.cuda(), seq_cu=cu.cuda(), seq_bt=bt.cuda(), num_decode=n, num_prefill_tokens=0, max_ctx=max(ctxs))
    p, c, out = proj.cuda(), cache.cuda(), torch.empty(n, heads * dim, dtype=dtype, device="cuda")
    taken = ops._window_decode(out, p, c, meta, sp, gate_off if gate else -1, 1.0, None if sink_w is None else sink_w.cuda())
    assert taken == (dim < 256 or dtype == torch.bfloat16)
    if taken:
        # bf16: weights and outputs rounded to 2^-9, the largest value about 4.5; fp32: sums of up to 1500 products
        tol, least = (2.0 ** -7, 2.0 ** -8) if dtype == torch.bfloat16 else (2.0 ** -18, 2.0 ** -19)
        assert ((out.double().cpu() - want).abs() <= tol * want.abs() + least * rows.abs().max() * 0.5).all()


@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("ctx", [40, 700])   # one run of keys, several
def test_window_attention_decode_rows_of_one_sequence(ctx, dtype):
    """Row counts (2, 0, 1): every row sees what it would see as its sequence's last one, in the same bits."""
    from types import SimpleNamespace
    g = torch.Generator().manual_seed(ctx)
    heads, kv, dim, bs = 4, 2, 64, 16
    sp = SimpleNamespace(maps=1, dim=dim, vdim=dim, heads=heads, kv_heads=kv, window=0, reach=0, scale=dim ** -0.5, sink=False,
                         keep_first=0, softcap=0.0, channel_gate=False, chunk=0)
    width = -(-ctx // bs)
    bt = torch.randperm(3 * width, generator=g).int().view(3, width).cuda()
    cache, proj = torch.randn(3 * width, bs, 2 * kv * dim, generator=g).to(dtype).cuda(), torch.randn(3, heads * dim, generator=g).to(dtype).cuda()

    def run(cu, ctxs, tables):
        meta = SimpleNamespace(seq_ctx=torch.tensor(ctxs).int().cuda(), seq_cu=torch.tensor(cu).int().cuda(), seq_bt=tables.contiguous(),
                               num_decode=3, num_prefill_tokens=0, max_ctx=ctx)
        out = torch.full((3, heads * dim), float("nan"), dtype=dtype, device="cuda")
        assert get_ops("cuda")._window_decode(out, proj, cache, meta, sp, -1, 1.0, None)
        return out
    want = run([0, 1, 2, 3], [ctx - 1, ctx, ctx - 5], bt[[0, 0, 2]])
    assert torch.equal(run([0, 2, 2, 3], [ctx, 9, ctx - 5], bt), want) and want.isfinite().all()


@gpu
@pytest.mark.parametrize("dim,lens,ctx", [(64, [1] * 16, 1024), (128, [1] * 6, 500)])
def test_window_attention_fp32_error(dim, lens, ctx, monkeypatch):
    """fp32 decode rows on the matrix cores beside the kernel without them, both against 64 bits."""
    from types import SimpleNamespace
    g = torch.Generator().manual_seed(dim)
    heads, kv, bs, n, T = 8, 2, 16, len(lens), sum(lens)
    sp = SimpleNamespace(maps=1, dim=dim, vdim=dim, heads=heads, kv_heads=kv, window=0, reach=0, scale=dim ** -0.5, sink=False,
                         keep_first=0, softcap=0.0, channel_gate=False, chunk=0, diff=0.0)
    width = -(-ctx // bs)
    cache, proj = torch.randn(n * width, bs, 2 * kv * dim, generator=g) * 1.2, torch.randn(T, heads * dim, generator=g) * 1.3
    cu, nd = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist()).int(), n if T == n else 0
    meta = SimpleNamespace(seq_ctx=torch.full((n,), ctx).int().cuda(), seq_cu=cu.cuda(), seq_bt=torch.arange(n * width).int().view(n, width).cuda(),
                           num_decode=nd, num_prefill_tokens=0 if nd else T, max_ctx=ctx)
    rows, want = cache.double().view(n, -1, 2 * kv, dim), torch.empty(T, heads, dim, dtype=torch.float64)
    for s in range(n):
        mine = slice(int(cu[s]), int(cu[s + 1]))
        hidden = torch.arange(ctx) > torch.arange(ctx - lens[s], ctx)[:, None]
        for h in range(heads):
            k, v = rows[s, :ctx, h // (heads // kv)], rows[s, :ctx, kv + h // (heads // kv)]
            sc = proj[mine, h * dim:(h + 1) * dim].double() @ k.T * sp.scale
            want[mine, h] = torch.softmax(sc.masked_fill(hidden, -float("inf")), -1) @ v
    ops, errs = get_ops("cuda"), []
    for on in (True, False):
        monkeypatch.setattr(type(ops), "WINDOW_MFMA", on)
        out = torch.empty(T, heads * dim, device="cuda")
        ops.window_attention(out, proj.cuda(), cache.cuda(), meta, sp, -1)
        errs.append(((out.double().cpu().view(T, heads, dim) - want).norm() / want.norm()).item())
    assert errs[0] <= 0.8 * errs[1], errs   # measured 0.57 - 0.71; scores summed in a single chain make it 0.96 - 1.02


# ------------------------------------------------------------------ generalized delta rule in chunks
@gpu
@pytest.mark.parametrize("lens", [[32], [33, 1, 16], [40, 15, 100], [33] + [1] * 70 + [50] + [2] * 65])
def test_delta_rule_chunks(lens):
    """Whole and partly filled chunks, more sequences than lanes, carried and fresh states, beside the reference; a row that is not finite poisons itself
    and what follows, not the rows before it."""
    from types import SimpleNamespace
    g = torch.Generator().manual_seed(sum(lens))
    H, d, T, n = 3, 64, sum(lens), len(lens)
    N, eps = H * d, 1e-5
    proj = torch.randn(T, 5 * N + 64, generator=g).bfloat16()
    wl, S = torch.randn(T, N, generator=g) * 2, torch.randn(n + 1, H, d, d, generator=g)
    a_b, w0, nw = torch.randn(N, generator=g), torch.randn(N, generator=g), torch.rand(N, generator=g) + 0.5
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32)
    ctx = torch.tensor([m + (9 if i % 2 == 0 else 0) for i, m in enumerate(lens)], dtype=torch.int32)
    slots = torch.randperm(n + 1, generator=g)[:n].int()
    sp = SimpleNamespace(heads=H, dim=d, size=N)
    meta = SimpleNamespace(seq_cu=cu.cuda(), seq_ctx=ctx.cuda(), seq_state=slots.cuda(), max_q=max(lens))
    ops = get_ops("cuda")
    assert ops._delta.delta_rule_chunk_floats(proj.cuda(), n, H, d) > 0

    def run(p):
        out, state = torch.empty(T, N, dtype=torch.bfloat16, device="cuda"), S.cuda()
        ops.delta_rule(out, [state], p.cuda(), wl.cuda(), a_b.cuda(), w0.cuda(), nw.cuda(), sp, eps, meta)
        return out.cpu(), state.cpu()
    want_s, want = S.clone(), torch.empty(T, N, dtype=torch.bfloat16)
    ref.delta_rule(want, want_s, proj, wl, a_b, w0, nw, sp, eps, cu, ctx, slots, 1.0)
    got, got_s = run(proj)
    # states are sums of about 64 products of either order, 2^-24 each, that a decay of at least 0.545 per row forgets
    assert ((got_s - want_s).abs() <= 2.0 ** -15 * want_s.abs().max()).all()
    assert ((got.float() - want.float()).abs() <= 2.0 ** -7 * want.float().abs() + 2.0 ** -13 * want.float().abs().max()).all()
    for col, last in ((2 * N + 5, lens[0]), (3, 21)):   # a value: the rest of the sequence; r: the row alone
        bad = proj.clone()
        bad[20, col] = float("nan")
        hit = torch.zeros(T, N, dtype=torch.bool)
        hit[20:last, :d] = True
        out, _ = run(bad)
        assert torch.equal(out.isnan(), hit) and torch.equal(out[~hit], got[~hit])


@gpu
@pytest.mark.parametrize("T,decay,carried", [(32, 0.6, False), (100, 0.6, True), (400, 2.0, False), (300, 0.2, True)])
def test_delta_rule_chunks_are_as_precise(T, decay, carried):
    """The chunks' states and outputs are no further from 64 bits than the token by token ones."""
    g = torch.Generator().manual_seed(T)
    H, d = 16, 64
    N = H * d
    proj, wl = torch.randn(T, 5 * N, generator=g).bfloat16().cuda(), (torch.randn(T, N, generator=g) * decay).cuda()
    a_b, w0, nw = (torch.randn(N, generator=g).cuda() for _ in range(3))
    S0 = (torch.randn(1, H, d, d, generator=g) * carried).cuda()
    r, k, v, a = (proj[:, i * N:(i + 1) * N].double().view(T, H, d) for i in range(4))
    w = torch.exp(-0.6065306597126334 * torch.sigmoid(wl.double() + w0.double())).view(T, H, d)
    u = k * torch.rsqrt(k.square().sum(-1, keepdim=True) + 1e-6)
    au = torch.sigmoid(a + a_b.double().view(H, d)) * u
    S, o = S0[0].double(), torch.empty(T, H, d, dtype=torch.float64, device="cuda")
    for t in range(T):
        S = S * w[t][..., None] - au[t][..., None] * (u[t][..., None] * S).sum(1, keepdim=True) + k[t][..., None] * v[t][:, None]
        o[t] = (r[t][..., None] * S).sum(1)
    delta = get_ops("cuda")._delta
    cu, ctx, slot = torch.tensor([0, T]).int().cuda(), torch.tensor([T + carried]).int().cuda(), torch.zeros(1).int().cuda()
    errs = []
    for floats in (0, delta.delta_rule_chunk_floats(proj, 1, H, d)):
        out, state, scratch = torch.empty(T, N, dtype=torch.bfloat16, device="cuda"), S0.clone(), torch.empty(7 * T * N + 64, device="cuda")
        delta.delta_rule(out, state, proj, wl, a_b, w0, nw, cu, ctx, slot, scratch, H, d, 1e-6, 1.0, torch.empty(floats, device="cuda") if floats else None)
        raw = (scratch[:T * N] if floats else scratch[6 * T * N:7 * T * N]).view(T, H, d)   # the outputs before their norm
        errs.append([((x.double() - y).norm() / y.norm()).item() for x, y in ((state[0], S), (raw, o))])
    assert errs[1][0] <= errs[0][0] and errs[1][1] <= errs[0][1], errs


@gpu
@pytest.mark.parametrize("what,value", [("a", "inf"), ("a", "-inf"), ("w", "inf"), ("w", "-inf"), ("a", "nan"), ("w", "nan"), ("k", "nan"), ("k", "inf"),
                                        ("r", "nan"), ("r", "-inf"), ("v", "nan"), ("v", "inf")])
@pytest.mark.parametrize("row", [16, 21, 38])   # a chunk's first row, one inside, one in the last chunk (the next row spreads a NaN over the state's rows)
def test_delta_rule_chunks_not_finite(row, what, value):
    """What one input that is not finite does to outputs and states is what it does token by token: pre-activations saturate, a
    value reaches its column alone."""
    from types import SimpleNamespace
    g = torch.Generator().manual_seed(row)
    H, d, lens = 2, 64, [40, 7]
    N, T, eps = H * d, sum(lens), 1e-5
    proj, wl, S = torch.randn(T, 5 * N, generator=g).bfloat16(), torch.randn(T, N, generator=g), torch.randn(2, H, d, d, generator=g)
    a_b, w0, nw = torch.randn(N, generator=g), torch.randn(N, generator=g), torch.rand(N, generator=g) + 0.5
    into, col = (wl, 5) if what == "w" else (proj, {"r": 0, "k": N, "v": 2 * N, "a": 3 * N}[what] + 5)
    into[row, col] = float(value)
    sp = SimpleNamespace(heads=H, dim=d, size=N)
    meta = SimpleNamespace(seq_cu=torch.tensor([0, 40, 47]).int().cuda(), seq_ctx=torch.tensor([60, 7]).int().cuda(),
                           seq_state=torch.tensor([1, 0]).int().cuda(), max_q=40)
    res = []
    for chunks in (False, True):
        ops = get_ops("cuda")
        ops.DELTA_CHUNK = chunks
        out, state = torch.empty(T, N, dtype=torch.bfloat16, device="cuda"), S.cuda()
        ops.delta_rule(out, [state], proj.cuda(), wl.cuda(), a_b.cuda(), w0.cuda(), nw.cuda(), sp, eps, meta)
        res.append((out.float(), state))
    for (want, got), tol, least in zip(zip(*res), (2.0 ** -7, 2.0 ** -15), (2.0 ** -13, 2.0 ** -15)):
        assert torch.equal(got.isfinite(), want.isfinite())
        want, got = want.nan_to_num(0.0, 0.0, 0.0), got.nan_to_num(0.0, 0.0, 0.0)
        assert ((got - want).abs() <= tol * want.abs() + least * want.abs().max()).all()
    assert bool(res[0][1].isfinite().all()) == (what == "r" or (what in "aw" and value != "nan"))


@gpu
@pytest.mark.parametrize("n", [6, 12, 37])
def test_gated_delta_rows_of_a_run(n):
    """What enters the rule, prepared in runs of 4, 8 and 16 rows (by the size of the step) and, a sequence by itself, of 2: the same bits."""
    g = torch.Generator().manual_seed(n)
    H, dim, one = 32, 32, 100
    N = H * dim
    cols, T = 3 * N, n * one
    delta = get_ops("cuda")._delta
    proj = torch.randn(T, cols + 2 * H + N, generator=g).bfloat16().cuda()
    conv, kept = torch.randn(cols, 4, generator=g).cuda(), torch.randn(n, 3, cols, generator=g).cuda()
    a, b, nw = (torch.randn(H, generator=g).cuda() for _ in range(3))

    def run(rows, kept):
        t, m = rows.shape[0], kept.shape[0]
        scratch = torch.empty(t * (4 * N + 2 * H) + 64, device="cuda")
        delta.gated_delta(torch.empty(t, N, dtype=torch.bfloat16, device="cuda"), torch.zeros(m, H, dim, dim, device="cuda"), kept.clone(), rows, conv, a, b,
                          nw, None, None, (torch.arange(m + 1) * one).int().cuda(), torch.full((m,), one + 1).int().cuda(), torch.arange(m).int().cuda(), scratch, H,
                          H, dim, dim, 4, 1e-6, cols + H, cols + 2 * H, cols, False, True, torch.empty(delta.delta_chunk_floats(t, m, H, dim, dim), device="cuda"))
        return [x.view(t, -1) for x in scratch[:-64].split([t * 2 * N, t * H, t * N, t * H, t * N])[:4]]
    whole = run(proj, kept)
    for i in (0, 1, n - 1):
        rows = slice(i * one, (i + 1) * one)
        assert all(torch.equal(x, y[rows]) for x, y in zip(run(proj[rows], kept[i:i + 1]), whole)), i


@gpu
@pytest.mark.parametrize("rule,heads,vdim", [("gated", 16, 128), ("gated", 13, 100), ("generalized", 32, 64)])
def test_delta_chunks_of_one_and_two_tiles(rule, heads, vdim):
    """Eight sequences in one step (two tiles of value channels per workgroup) and each by itself (one): the same bits; the last rows of a
    sequence's last chunk, and columns past a tile's end, belong to others."""
    g = torch.Generator().manual_seed(heads)
    lens, dim = [33, 1, 16, 50, 64, 17, 5, 100], 128 if rule == "gated" else 64
    T, n, N, nq = sum(lens), len(lens), heads * vdim, heads * dim
    cols = 2 * nq + N
    delta = get_ops("cuda")._delta
    proj = torch.randn(T, cols + 2 * heads + N if rule == "gated" else 5 * N, generator=g).bfloat16().cuda()
    wl, conv, S0 = torch.randn(T, N, generator=g).cuda(), torch.randn(cols, 4, generator=g).cuda(), torch.randn(n, heads, dim, vdim, generator=g).cuda()
    a, b, nw = (torch.randn(max(heads, N), generator=g).cuda() for _ in range(3))
    start = [0] + torch.tensor(lens).cumsum(0).tolist()

    def run(first, last):
        rows, m = slice(start[first], start[last]), last - first
        t, state, out = start[last] - start[first], S0[first:last].clone(), torch.empty(start[last] - start[first], N, dtype=torch.bfloat16, device="cuda")
        cu = torch.tensor([c - start[first] for c in start[first:last + 1]]).int().cuda()
        ctx, slots = torch.tensor([k + (i % 2) for i, k in enumerate(lens)][first:last]).int().cuda(), torch.arange(m).int().cuda()
        if rule == "gated":
            scratch, chunks = torch.empty(t * (2 * nq + 2 * N + 2 * heads) + 64, device="cuda"), torch.empty(delta.delta_chunk_floats(t, m, heads, dim, vdim), device="cuda")
            delta.gated_delta(out, state, torch.zeros(m, 3, cols, device="cuda"), proj[rows], conv, a[:heads], b[:heads], nw[:vdim], None, None, cu, ctx, slots,
                              scratch, heads, heads, dim, vdim, 4, 1e-6, cols + heads, cols + 2 * heads, cols, False, True, chunks)
        else:
            scratch, chunks = torch.empty(t * N + 64, device="cuda"), torch.empty(delta.delta_rule_chunk_floats(proj[rows], m, heads, dim), device="cuda")
            delta.delta_rule(out, state, proj[rows], wl[rows], a, b, nw, cu, ctx, slots, scratch, heads, dim, 1e-6, 1.0, chunks)
        return out, state
    out, state = run(0, n)
    for i in range(n):
        alone, its = run(i, i + 1)
        assert torch.equal(alone, out[start[i]:start[i + 1]]) and torch.equal(its, state[i:i + 1]), i
    assert out.isfinite().all()


@gpu
@pytest.mark.parametrize("lens,dim,vdim,a,carried", [([40, 33], 128, 128, 0.0, False), ([300], 128, 128, -2.0, True), ([200], 64, 48, -1.0, True), ([100, 64], 32, 64, 0.0, False)])
def test_gated_delta_chunks_precision(lens, dim, vdim, a, carried):
    """States and outputs of the chunked gated rule beside the scan's, both against 64 bits from the same prepared rows."""
    g = torch.Generator().manual_seed(sum(lens))
    H, G, T, n = 8, 4, sum(lens), len(lens)
    N, nq = H * vdim, G * dim
    cols = 2 * nq + N
    proj = torch.randn(T, cols + 2 * H + N, generator=g).bfloat16().cuda()
    conv, a_log, dt_bias, nw = (v.cuda() for v in (torch.randn(cols, 4, generator=g), torch.randn(H, generator=g) * 0.5 + a,
                                                   torch.randn(H, generator=g) * 0.5, torch.rand(vdim, generator=g) + 0.5))
    S0 = (torch.randn(n, H, dim, vdim, generator=g) * 0.3 * carried).cuda()
    cu, ctx = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist()).int(), torch.tensor([m + carried for m in lens]).int().cuda()
    delta, errs = get_ops("cuda")._delta, []
    for floats in (0, delta.delta_chunk_floats(T, n, H, dim, vdim)):
        state, conv_state = S0.clone(), torch.zeros(n, 3, cols, device="cuda")
        out, scratch = torch.empty(T, N, dtype=torch.bfloat16, device="cuda"), torch.empty(T * (2 * nq + 2 * N + 2 * H) + 64, device="cuda")
        delta.gated_delta(out, state, conv_state, proj, conv, a_log, dt_bias, nw, None, None, cu.cuda(), ctx, torch.arange(n).int().cuda(), scratch, H, G,
                          dim, vdim, 4, 1e-6, cols + H, cols + 2 * H, cols, False, True, torch.empty(floats, device="cuda") if floats else None)
        # the rows that both prepare: queries and keys, decays, values, rates; then the outputs before their norm
        qk, dec, v, beta, raw = (x.double() for x in scratch[:-64].split([T * 2 * nq, T * H, T * N, T * H, T * N]))
        q, k = qk.view(T, 2, G, dim).repeat_interleave(H // G, 2).unbind(1)
        dec, v, beta, raw = dec.view(T, H, 1, 1), v.view(T, H, vdim), beta.view(T, H, 1), raw.view(T, H, vdim)
        S, o = S0.double(), torch.empty_like(raw)
        for s in range(n):
            for t in range(int(cu[s]), int(cu[s + 1])):
                S[s] *= dec[t]
                S[s] += k[t][..., None] * (beta[t] * (v[t] - (S[s] * k[t][..., None]).sum(1)))[:, None]
                o[t] = (S[s] * q[t][..., None]).sum(1)
        errs.append([((x.double() - y).norm() / y.norm()).item() for x, y in ((state, S), (raw, o))])
    # measured 1.1 - 1.25 and 1.2 - 1.35 times the scan's; sums that start at their largest part make it 1.7 - 2.8
    assert errs[1][0] <= 1.4 * errs[0][0] and errs[1][1] <= 1.5 * errs[0][1], errs


@gpu
@pytest.mark.parametrize("dim,vdim", [(70, 70), (128, 40), (129, 129), (200, 72), (256, 256)])
def test_scans_of_wide_heads(dim, vdim):
    """8 and 16 channels per lane, token by token: whole and partly filled batches of tokens, carried and fresh states, beside the reference; a slot that
    no sequence has stays as it was."""
    from types import SimpleNamespace
    g = torch.Generator().manual_seed(dim)
    lens, H, G = [3, 1, 8, 17, 10], 4, 2
    T, n, N, nq = sum(lens), len(lens), H * vdim, G * dim
    cols = 2 * nq + N
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist()).int()
    ctx, slots = torch.tensor([m + (7 if i % 2 else 0) for i, m in enumerate(lens)]).int(), torch.randperm(n + 1, generator=g)[:n].int()
    S, ops = torch.randn(n + 1, H, dim, vdim, generator=g), get_ops("cuda")
    meta = SimpleNamespace(seq_cu=cu.cuda(), seq_ctx=ctx.cuda(), seq_state=slots.cuda(), max_q=max(lens))

    def same(got, want):   # sums of up to 256 products of either order, 2^-24 each
        for a, b in zip(got, want):
            assert ((a.cpu() - b).abs() <= 2.0 ** -15 * b.abs().max()).all()
    proj = torch.randn(T, cols + 2 * H + N, generator=g)
    conv, dt, nw = torch.randn(cols, 4, generator=g), torch.randn(H, dim, generator=g), torch.rand(vdim, generator=g) + 0.5
    a_log, per, gate = torch.randn(H, generator=g) * 0.5, torch.randn(T, H * dim, generator=g), torch.randn(T, N, generator=g)
    for wide in (False, True):   # a decay per head, from the row; per key channel, given as the gate is
        sp = SimpleNamespace(heads=H, kv_heads=G, dim=dim, vdim=vdim, out_size=N, conv=4, conv_channels=cols, gate_act="silu", channel_decay=wide)
        bias, offs, kept = (dt if wide else dt[:, 0]).flatten(), (cols + H, cols + 2 * H, cols), torch.randn(n + 1, 3, cols, generator=g)
        own = (per, gate) if wide else (None, None)
        y, want, wc = torch.empty(T, N), S.clone(), kept.clone()
        ref.gated_delta(y, want, wc, proj, conv, a_log, bias, nw, *own, offs, sp, 1e-6, cu, ctx, slots)
        out, state = torch.empty(T, N, device="cuda"), [S.cuda(), kept.cuda()]
        ops.gated_delta(out, state, proj.cuda(), conv.cuda(), a_log.cuda(), bias.cuda(), nw.cuda(), *(x if x is None else x.cuda() for x in own), offs, sp,
                        1e-6, meta)
        same((out, *state), (y, want, wc))
    if dim != vdim: return
    proj, wl = torch.randn(T, 5 * N + 64, generator=g), torch.randn(T, N, generator=g) * 2
    a_b, w0, nw = torch.randn(N, generator=g), torch.randn(N, generator=g), torch.rand(N, generator=g) + 0.5
    sp = SimpleNamespace(heads=H, dim=dim, size=N)
    y, want, out, state = torch.empty(T, N), S.clone(), torch.empty(T, N, device="cuda"), S.cuda()
    ref.delta_rule(y, want, proj, wl, a_b, w0, nw, sp, 1e-5, cu, ctx, slots, 1.0)
    ops.delta_rule(out, [state], proj.cuda(), wl.cuda(), a_b.cuda(), w0.cuda(), nw.cuda(), sp, 1e-5, meta)
    same((out, state), (y, want))


# ------------------------------------------------------------------ window attention of prompts
@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads,kv,dim,bs,lens,ctxs,opts", [
    (1, 1, 64, 16, [1, 33], [1, 40], {}), (8, 2, 128, 16, [31, 32, 65], [31, 100, 65], {"window": 40, "sink": True, "gate": True}),
    (5, 1, 64, 64, [130, 7], [300, 7], {"window": 0, "softcap": 3.0, "channel_gate": True}),
    (130, 1, 64, 16, [9], [50], {"window": 20, "sink_w": True}), (4, 4, 128, 128, [200, 3], [210, 203], {"chunk": 64}),
    (16, 4, 128, 16, [700, 300], [700, 450], {"window": 256, "sink": True}), (2, 1, 128, 8, [40], [64], {"window": 16, "keep_first": 5}),
    (4, 2, 64, 16, [1] * 65 + [40] + [2] * 70, [5] * 65 + [60] + [3] * 70, {"window": 30})])
def test_window_attention_prompts(heads, kv, dim, bs, lens, ctxs, opts, dtype):
    """Tokens, heads and keys that do not fill a tile, windows and chunks that start inside one, pages smaller and larger than a
    tile, one and two row tiles per wave, more than 128 heads per key / value head, kept keys, which the other
    kernel takes in bf16, and more sequences than lanes; fp32."""
    from types import SimpleNamespace
    g = torch.Generator().manual_seed(heads * dim + sum(lens))
    n, T, gate = len(lens), sum(lens), opts.get("gate", False) or opts.get("channel_gate", False)
    sp = SimpleNamespace(maps=1, dim=dim, vdim=dim, heads=heads, kv_heads=kv, window=opts.get("window", 0), scale=dim ** -0.5, sink=opts.get("sink", "sink_w" in opts),
                         keep_first=opts.get("keep_first", 0), softcap=opts.get("softcap", 0.0), channel_gate=opts.get("channel_gate", False), chunk=opts.get("chunk", 0), diff=0.0)
    sp.reach = sp.window + sp.keep_first if sp.window else sp.chunk
    width = -(-max(ctxs) // bs)
    bt = torch.randperm(n * width, generator=g).int().view(n, width)
    cache = torch.randn(n * width, bs, 2 * kv * dim, generator=g).to(dtype)
    proj = torch.randn(T, 2 * heads * dim, generator=g).to(dtype)
    sink_w = torch.randn(heads, generator=g) if opts.get("sink_w") else None
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32)
    want = torch.empty(T, heads, dim, dtype=torch.float64)
    rows = cache.double().view(-1, 2 * kv, dim)
    for s in range(n):
        j = torch.arange(ctxs[s])
        kvr = rows[bt[s].long()[j // bs] * bs + j % bs]
        p = torch.arange(ctxs[s] - lens[s], ctxs[s])[:, None]
        lo = p - p % sp.chunk if sp.chunk else p - sp.window + 1 if sp.window else torch.zeros_like(p)
        seen = (j <= p) & ((j >= lo) | (j < sp.keep_first))
        for h in range(heads):
            q = proj[cu[s]:cu[s + 1], h * dim:(h + 1) * dim].double()
            x = q @ kvr[:, h // (heads // kv)].t() * sp.scale
            x = sp.softcap * torch.tanh(x / sp.softcap) if sp.softcap else x
            x = x.masked_fill(~seen, float("-inf"))
            if sp.sink:
                x = torch.cat([x, torch.full((len(p), 1), float(sink_w[h]) if sink_w is not None else 0.0, dtype=torch.float64)], 1)
            want[cu[s]:cu[s + 1], h] = torch.softmax(x, 1)[:, :len(j)] @ kvr[:, kv + h // (heads // kv)]
    want = want.view(T, -1)
    if gate:
        gates = torch.sigmoid(proj[:, heads * dim:heads * dim + (heads * dim if sp.channel_gate else heads)].double())
        want *= gates if sp.channel_gate else gates.repeat_interleave(dim, 1)
    meta = SimpleNamespace(seq_ctx=torch.tensor(ctxs).int().cuda(), seq_cu=cu.cuda(), seq_bt=bt.cuda(), num_decode=0, num_prefill_tokens=T, max_ctx=max(ctxs))
    out = torch.empty(T, heads * dim, dtype=dtype, device="cuda")
    get_ops("cuda").window_attention(out, proj.cuda(), cache.cuda(), meta, sp, heads * dim if gate else -1, 1.0, 0.0, 0.0, None if sink_w is None else sink_w.cuda())
    # bf16: weights and outputs rounded to 2^-9, the largest value about 4.5; fp32: sums of up to 700 products
    tol, least = (2.0 ** -7, 2.0 ** -8) if dtype == torch.bfloat16 else (2.0 ** -18, 2.0 ** -19)
    assert ((out.double().cpu() - want).abs() <= tol * want.abs() + least * rows.abs().max() * 0.5).all()


@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_delta_rule_step(dtype):
    """One row per sequence, fresh and carried states, a sequence without a row, in one launch beside the reference."""
    from types import SimpleNamespace
    g = torch.Generator().manual_seed(5)
    H, d, cu = 3, 64, [0, 1, 2, 2, 3]
    N, T, n, eps = H * d, 3, 4, 1e-5
    proj = torch.randn(T, 5 * N + 4, generator=g).to(dtype)
    wl, S = torch.randn(T, N, generator=g) * 2, torch.randn(n + 1, H, d, d, generator=g)
    a_b, w0, nw = torch.randn(N, generator=g), torch.randn(N, generator=g), torch.rand(N, generator=g) + 0.5
    cu, ctx, slots = torch.tensor(cu).int(), torch.tensor([1, 9, 4, 2]).int(), torch.tensor([4, 0, 3, 1]).int()
    sp, meta = SimpleNamespace(heads=H, dim=d, size=N), SimpleNamespace(seq_cu=cu.cuda(), seq_ctx=ctx.cuda(), seq_state=slots.cuda(), max_q=1)
    want_s, want = S.clone(), torch.empty(T, N, dtype=dtype)
    ref.delta_rule(want, want_s, proj, wl, a_b, w0, nw, sp, eps, cu, ctx, slots, 1.5)
    got_s, got = S.cuda(), torch.empty(T, N, dtype=dtype, device="cuda")
    get_ops("cuda").delta_rule(got, [got_s], proj.cuda(), wl.cuda(), a_b.cuda(), w0.cuda(), nw.cuda(), sp, eps, meta, 1.5)
    assert ((got_s.cpu() - want_s).abs() <= 64 * 2.0 ** -24 * want_s.abs().max()).all()   # a sum of 64 products
    tol, least = (2.0 ** -7, 2.0 ** -13) if dtype == torch.bfloat16 else (2.0 ** -17, 2.0 ** -17)
    assert ((got.cpu().float() - want.float()).abs() <= tol * want.float().abs() + least * want.float().abs().max()).all()


@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rank", [32, 96, 128])
def test_delta_rule_low(rank, dtype):
    """The decay bottleneck's product in the decode step's launch: one load per wave and more."""
    from types import SimpleNamespace
    g = torch.Generator().manual_seed(rank)
    H, d, cu = 3, 64, torch.tensor([0, 1, 2, 2, 3]).int()
    N, T, n, eps = H * d, 3, 4, 1e-5
    proj, w2 = torch.randn(T, 5 * N + rank + 8, generator=g).to(dtype), (torch.randn(N, rank, generator=g) / rank ** 0.5).to(dtype)
    proj[:, 5 * N:] = proj[:, 5 * N:].tanh()
    S = torch.randn(n + 1, H, d, d, generator=g)
    a_b, w0, nw = torch.randn(N, generator=g), torch.randn(N, generator=g), torch.rand(N, generator=g) + 0.5
    ctx, slots = torch.tensor([1, 9, 4, 2]).int(), torch.tensor([4, 0, 3, 1]).int()
    sp, meta = SimpleNamespace(heads=H, dim=d, size=N), SimpleNamespace(seq_cu=cu.cuda(), seq_ctx=ctx.cuda(), seq_state=slots.cuda(), max_q=1)
    want_s, want = S.clone(), torch.empty(T, N, dtype=dtype)
    wl = (proj[:, 5 * N:5 * N + rank].double() @ w2.double().T).float()
    ref.delta_rule(want, want_s, proj, wl, a_b, w0, nw, sp, eps, cu, ctx, slots, 1.5)
    got_s, got = S.cuda(), torch.empty(T, N, dtype=dtype, device="cuda")
    assert get_ops("cuda").delta_rule_low(got, [got_s], proj.cuda(), w2.cuda(), a_b.cuda(), w0.cuda(), nw.cuda(), sp, eps, meta, 1.5)
    # a sum of 64 products, and `rank` of them in a decay, whose slope is at most 0.15
    assert ((got_s.cpu() - want_s).abs() <= (64 + rank) * 2.0 ** -24 * want_s.abs().max()).all()
    # the outputs of test_delta_rule_step, 2^-17 = 64 x 2^-23 for sums of 64 products, with `rank` products more
    tol, least = (2.0 ** -7, 2.0 ** -13) if dtype == torch.bfloat16 else ((64 + rank) * 2.0 ** -23,) * 2
    assert ((got.cpu().float() - want.float()).abs() <= tol * want.float().abs() + least * want.float().abs().max()).all()


@gpu
@pytest.mark.parametrize("rows", [1, 40])
def test_delta_rule_unaligned(rows):
    """States and 32-bit rows that do not start at 16 bytes take the token by token kernels, as other sizes do."""
    from types import SimpleNamespace
    g = torch.Generator().manual_seed(rows)
    H, d, n = 2, 64, 2
    N, T = H * d, n * rows
    proj, wl, S = torch.randn(T, 5 * N, generator=g).bfloat16(), torch.randn(T, N, generator=g), torch.randn(n, H, d, d, generator=g)
    a_b, w0, nw = torch.randn(N, generator=g), torch.randn(N, generator=g), torch.rand(N, generator=g) + 0.5
    cu, ctx, slots = torch.tensor([0, rows, T]).int(), torch.tensor([rows + 4, rows]).int(), torch.tensor([1, 0]).int()
    sp = SimpleNamespace(heads=H, dim=d, size=N)
    meta = SimpleNamespace(seq_cu=cu.cuda(), seq_ctx=ctx.cuda(), seq_state=slots.cuda(), max_q=rows)
    want_s, want = S.clone(), torch.empty(T, N, dtype=torch.bfloat16)
    ref.delta_rule(want, want_s, proj, wl, a_b, w0, nw, sp, 1e-5, cu, ctx, slots, 1.0)

    def shifted(t):
        out = torch.empty(t.numel() + 1, device="cuda")[1:].view(t.shape)
        return out.copy_(t)
    got_s, got = shifted(S), torch.empty(T, N, dtype=torch.bfloat16, device="cuda")
    get_ops("cuda").delta_rule(got, [got_s], proj.cuda(), shifted(wl), shifted(a_b), shifted(w0), nw.cuda(), sp, 1e-5, meta)
    assert ((got_s.cpu() - want_s).abs() <= 2.0 ** -15 * want_s.abs().max()).all()
    assert ((got.cpu().float() - want.float()).abs() <= 2.0 ** -7 * want.float().abs() + 2.0 ** -13 * want.float().abs().max()).all()


# ------------------------------------------------------------------ latent rows
@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("q_rank,kv_rank,rot,nfreq", [(8, 8, 8, 4), (512, 128, 64, 32), (1024, 512, 64, 32), (7680, 512, 72, 20), (1536, 8192, 128, 64),
                                                      (20, 12, 8, 4)])
def test_latent_prepare(q_rank, kv_rank, rot, nfreq, dtype):
    """One item of 8 to two per thread, rotary dims that do not all rotate, rows without a slot; the last two: the general kernel."""
    g = torch.Generator().manual_seed(q_rank)
    T, eps = 4, 1e-5
    proj = torch.randn(T, q_rank + kv_rank + rot + 8, generator=g).to(dtype)
    cache, cq = torch.zeros(2, 16, kv_rank + rot, dtype=dtype), torch.empty(T, q_rank, dtype=dtype)
    pos, slots = torch.tensor([0, 5, 300, 9000]), torch.tensor([31, -1, 0, 2])
    inv = 1e4 ** (-torch.arange(nfreq).float() / nfreq)
    qn, kn = torch.rand(q_rank, generator=g) + 0.5, torch.rand(kv_rank, generator=g) + 0.5
    c, q = cache.cuda(), torch.empty(T, q_rank, dtype=dtype, device="cuda")
    get_ops("cuda").latent_prepare(q, c, proj.cuda(), pos.cuda(), slots.cuda(), qn.cuda(), kn.cuda(), inv.cuda(), q_rank, kv_rank, rot, eps)
    ref.latent_prepare(cq, cache, proj, pos, slots, qn, kn, inv, q_rank, kv_rank, rot, eps)
    # an angle of up to 9000 rounds to 2^-11
    tol = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -18
    assert ((q.cpu().float() - cq.float()).abs() <= tol * cq.float().abs() + 2.0 ** -20).all()
    assert ((c.cpu().float() - cache.float()).abs() <= tol * cache.float().abs() + 2.0 ** -10 * 4.5).all()


@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("dim,n,ctx,window,chunk", [(128, 10, 100, 40, 0), (64, 20, 64, 33, 0), (128, 30, 200, 64, 0), (64, 5, 90, 0, 50)])
def test_window_attention_hidden_keys(dim, n, ctx, window, chunk, dtype):
    """Keys before the first row's window or chunk, which no row sees, may hold anything."""
    from types import SimpleNamespace
    g = torch.Generator().manual_seed(ctx)
    heads, kv, bs = 4, 2, 16
    sp = SimpleNamespace(maps=1, dim=dim, vdim=dim, heads=heads, kv_heads=kv, window=window, reach=window or chunk, scale=dim ** -0.5, sink=True, keep_first=0,
                         softcap=0.0, channel_gate=False, chunk=chunk, diff=0.0)
    pages = -(-ctx // bs)
    cache, proj = torch.randn(pages * bs, 2 * kv * dim, generator=g).to(dtype), torch.randn(n, heads * dim, generator=g).to(dtype).cuda()
    meta = SimpleNamespace(seq_cu=torch.tensor([0, n]).int().cuda(), seq_ctx=torch.tensor([ctx]).int().cuda(), seq_bt=torch.arange(pages).int().view(1, -1).cuda(),
                           num_decode=0, num_prefill_tokens=n, max_ctx=ctx)
    outs = []
    for value in (0.0, float("nan"), -float("inf")):
        cache[:(ctx - n) // chunk * chunk if chunk else ctx - n - window + 1] = value
        outs.append(torch.empty(n, heads * dim, dtype=dtype, device="cuda"))
        get_ops("cuda").window_attention(outs[-1], proj, cache.view(pages, bs, -1).cuda(), meta, sp, -1)
    assert outs[0].isfinite().all() and torch.equal(outs[1], outs[0]) and torch.equal(outs[2], outs[0])


@gpu
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("chunk,at,rows", [(0, 23, slice(0, 8)), (16, 3, slice(8, 16))])
def test_window_attention_fp32_values_of_hidden_tiles(dim, chunk, at, rows):
    """Positions 8 .. 23 share a tile of rows, and two waves their keys 0 .. 15 and 16 .. 23: what a row's wave holds that sees none of its
    keys, those after it or of the chunk before it, stays out of the row whatever their values are."""
    from types import SimpleNamespace
    g = torch.Generator().manual_seed(dim + chunk)
    n, ctx, heads = 16, 24, 2
    sp = SimpleNamespace(maps=1, dim=dim, vdim=dim, heads=heads, kv_heads=heads, window=0, reach=chunk, scale=dim ** -0.5, sink=False, keep_first=0,
                         softcap=0.0, channel_gate=False, chunk=chunk, diff=0.0)
    cache, proj = torch.randn(2, 16, 2 * heads * dim, generator=g), torch.randn(n, heads * dim, generator=g).cuda()
    meta = SimpleNamespace(seq_cu=torch.tensor([0, n]).int().cuda(), seq_ctx=torch.tensor([ctx]).int().cuda(), seq_bt=torch.arange(2).int().view(1, -1).cuda(),
                           num_decode=0, num_prefill_tokens=n, max_ctx=ctx)
    outs = []
    for value in (0.0, float("nan"), -float("inf")):
        cache[at // 16, at % 16, heads * dim:] = value
        outs.append(torch.empty(n, heads * dim, device="cuda"))
        get_ops("cuda").window_attention(outs[-1], proj, cache.cuda(), meta, sp, -1)
    assert outs[0].isfinite().all() and not outs[1][n - 1 if chunk == 0 else 0].isfinite().any()
    assert torch.equal(outs[1][rows], outs[0][rows]) and torch.equal(outs[2][rows], outs[0][rows])


@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads,kv,dim,ctxs,nfreq,mode,own,opts", [
    (1, 1, 64, [1], 0, 0, True, {}), (16, 4, 128, [1, 31, 32, 33, 700], 64, 1, True, {"v_norm": True}),
    (40, 2, 64, [5, 129, 400], 16, 2, True, {"window": 100, "keep_first": 7, "temp_every": 64}), (64, 8, 128, [2, 20], 64, 1, True, {}),
    (32, 2, 128, [64, 65, 1500], 32, 3, True, {"chunk": 64}), (16, 1, 256, [3, 290], 128, 2, True, {}), (8, 2, 128, [16, 300], 64, 1, False, {})])
def test_window_step(heads, kv, dim, ctxs, nfreq, mode, own, opts, dtype):
    """The launch for a decode step beside the two it takes the place of: one key, runs that end before, at and behind a tile's end, several
    runs, more than 16 heads per key / value head, more than one round of items and sums (one wave, 72 heads), each norm, a
    row without a slot, queries alone, and a sequence without a row."""
    from types import SimpleNamespace
    g = torch.Generator().manual_seed(heads * dim + mode)
    n, bs, nq, nk = len(ctxs), 8, heads * dim, kv * dim
    sp = SimpleNamespace(maps=1, dim=dim, vdim=dim, heads=heads, kv_heads=kv, window=opts.get("window", 0), scale=dim ** -0.5, sink=False,
                         keep_first=opts.get("keep_first", 0), softcap=0.0, channel_gate=False, chunk=opts.get("chunk", 0), diff=0.0, q_size=nq,
                         k_size=nk, v_size=nk, kv_from=None if own else 0, qk_norm=mode == 1, head_norm=mode == 2, unit_qk=mode == 3,
                         v_norm=opts.get("v_norm", False), temp_coef=0.1, temp_every=opts.get("temp_every", 0), scaling=SimpleNamespace(amplitude=1.25))
    sp.reach = sp.window + sp.keep_first if sp.window > 0 else sp.chunk
    width = -(-max(ctxs) // bs)
    bt = torch.randperm((n + 1) * width, generator=g).int().view(n + 1, width)
    cache = torch.randn((n + 1) * width, bs, 2 * nk, generator=g).to(dtype).cuda()
    proj = torch.randn(n + 1, nq + (2 * nk if own else 0) + 16, generator=g).to(dtype).cuda()   # a padding row at the end
    w = [torch.rand(m, generator=g).cuda() + 0.5 for m in {1: (nq, nk), 2: (dim, dim)}[mode]] if mode in (1, 2) else [None, None]
    pos = torch.tensor([c - 1 for c in ctxs] + [0])
    slots = torch.tensor([int(bt[s, (c - 1) // bs]) * bs + (c - 1) % bs for s, c in enumerate(ctxs)] + [-1])
    if n > 2:
        slots[1] = -1   # its key and value stay what the cache holds
    cu, ctx = torch.tensor([*range(n + 1), n]).int(), torch.tensor(ctxs + [0]).int()
    meta = SimpleNamespace(seq_ctx=ctx.cuda(), seq_cu=cu.cuda(), seq_bt=bt.cuda(), num_decode=n + 1, num_prefill_tokens=0, max_ctx=max(ctxs), max_q=1,
                           positions=pos.cuda(), slot_mapping=slots.cuda())
    inv = (1e4 ** (-torch.arange(nfreq).float() / max(nfreq, 1))).cuda()
    ops = get_ops("cuda")
    p, c, out, want = proj.clone(), cache.clone(), torch.zeros(n + 1, nq, dtype=dtype, device="cuda"), torch.zeros(n + 1, nq, dtype=dtype, device="cuda")
    taken = ops.window_step(out, p, c, meta, inv, sp, *w, 1e-5, -1)
    assert taken == (dim < 256)
    if not taken:
        return
    assert torch.equal(p, proj)
    ops.attn_prepare(p, cache, meta, inv, sp, *w, 1e-5)
    ops.window_attention(want, p, cache, meta, sp, -1)
    # sums of squares in another order: 2^-22 of a head's factor, so that an element of the cache, and of the queries, may round the other way:
    # 2^-8 in bf16; in fp32 that factor and three more roundings. A score of up to about 60 (queries and keys times 1.25 and weights of up to 1.5, sums
    # of 256 products at 16 standard deviations) moves by 60 x 2^-8 x 3 / sqrt(128) at the most, an output by that share and its own rounding.
    tol = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -20
    assert ((c.float() - cache.float()).abs() <= tol * cache.float().abs() + 2.0 ** -20).all()
    tol = 0.08 if dtype == torch.bfloat16 else 60 * 2.0 ** -20
    out, want = out[:n].float(), want[:n].float()   # the padding row's is nobody's
    assert (out - want).abs().max() <= tol * max(1.0, float(want.abs().max()))


@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads,kv,dim,ctxs,opts", [
    (8, 2, 128, [1, 5, 33], {"sink": True}), (8, 2, 128, [2, 300, 600], {"sink": True}), (8, 2, 128, [1, 31, 200], {"sink_w": True, "gate": True}),
    (8, 2, 128, [129, 500], {"sink_w": True, "softcap": 3.0}), (40, 2, 64, [5, 129, 400], {"window": 100, "keep_first": 7, "channel_gate": True, "scale": 0.5}),
    (4, 4, 64, [40, 257], {"softcap": 2.0, "channel_gate": True, "scale": 1.5}), (16, 2, 64, [64, 65, 300], {"chunk": 64, "gate": True, "scale": 0.25})])
def test_window_step_options(heads, kv, dim, ctxs, opts, dtype):
    """Sinks, gates, the cap and the factor of the launch for a decode step, in one run and in several, against 64 bits. Projections that are neither
    normed nor turned go through unaltered, so that the bound holds the attention's own roundings alone: it sees any one key left out (asserted on
    the 64-bit side), and any sink but one of weight 1 among hundreds of keys in bf16."""
    from types import SimpleNamespace
    g = torch.Generator().manual_seed(heads * dim + sum(ctxs))
    n, bs, nq, nk = len(ctxs), 8, heads * dim, kv * dim
    gated, factor = opts.get("gate", False) or opts.get("channel_gate", False), opts.get("scale", 1.0)
    sp = SimpleNamespace(maps=1, dim=dim, vdim=dim, heads=heads, kv_heads=kv, window=opts.get("window", 0), scale=dim ** -0.5, sink=opts.get("sink", "sink_w" in opts),
                         keep_first=opts.get("keep_first", 0), softcap=opts.get("softcap", 0.0), channel_gate=opts.get("channel_gate", False),
                         chunk=opts.get("chunk", 0), diff=0.0, q_size=nq, k_size=nk, v_size=nk, kv_from=None, qk_norm=False, head_norm=False, unit_qk=False,
                         v_norm=False, temp_coef=0.0, temp_every=0, scaling=None)
    sp.reach = sp.window + sp.keep_first if sp.window > 0 else sp.chunk
    width = -(-max(ctxs) // bs)
    bt = torch.randperm(n * width, generator=g).int().view(n, width)
    cache, proj = torch.randn(n * width * bs, 2 * kv, dim, generator=g), torch.randn(n, nq + 2 * nk + nq, generator=g)
    for s, c in enumerate(ctxs):   # an element of every key's value that tells it from its neighbours
        for j in range(c):
            cache[int(bt[s, j // bs]) * bs + j % bs, kv:, j % dim] += 16
        proj[s, nq + nk:].view(-1, dim)[:kv, (c - 1) % dim] += 16
    cache, proj = cache.view(n * width, bs, 2 * nk).to(dtype), proj.to(dtype)
    slots = torch.tensor([int(bt[s, (c - 1) // bs]) * bs + (c - 1) % bs for s, c in enumerate(ctxs)])
    after = cache.clone()   # with every step's own key and value
    after.view(-1, 2 * nk)[slots] = proj[:, nq:nq + 2 * nk]
    sink_w = torch.randn(heads, generator=g) + 4 if opts.get("sink_w") else None
    rows, gate_off = after.double().view(-1, 2 * kv, dim), nq + 2 * nk
    want, size = torch.empty(n, heads, dim, dtype=torch.float64), torch.empty(n, heads, dim, dtype=torch.float64)   # size: sum of weight x |value|
    unit = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -17   # weights and outputs rounded to 8 bits, 2^-8 each; in fp32 scores of sums of up to 128 products
    for s in range(n):
        p = ctxs[s] - 1
        lo = p - p % sp.chunk if sp.chunk else max(0, p - sp.window + 1) if sp.window else 0
        js = sorted(set(range(lo, p + 1)) | (set(range(min(sp.keep_first, p + 1))) if sp.window else set()))
        kv_rows = rows[[int(bt[s, j // bs]) * bs + j % bs for j in js]].repeat_interleave(heads // kv, 1)
        k, v = kv_rows[:, :heads], kv_rows[:, heads:]
        x = torch.einsum("jhd,hd->hj", k, proj[s, :nq].double().view(heads, dim)) * sp.scale
        x = sp.softcap * torch.tanh(x / sp.softcap) if sp.softcap else x
        extra = torch.zeros(heads, int(sp.sink), dtype=torch.float64) if sink_w is None else sink_w.double()[:, None]
        w = torch.softmax(torch.cat([x, extra], 1), 1)[:, :len(js), None]
        v = v.transpose(0, 1)
        want[s], size[s] = (w * v).sum(1), (w * v.abs()).sum(1)
        if len(js) > 1:   # what any one key left out would change
            change = (w / (1 - w) * (want[s][:, None] - v)).abs() / (unit * size[s])[:, None]
            assert float(change.amax((0, 2)).min()) > 1
    if gated:
        gates = torch.sigmoid(proj[:, gate_off:gate_off + (nq if sp.channel_gate else heads)].double()).view(n, heads, -1)
        want, size = want * gates, size * gates
    ops = get_ops("cuda")
    meta = SimpleNamespace(seq_ctx=torch.tensor(ctxs).int().cuda(), seq_cu=torch.arange(n + 1).int().cuda(), seq_bt=bt.cuda(), num_decode=n, num_prefill_tokens=0,
                           max_ctx=max(ctxs), max_q=1, positions=torch.tensor(ctxs).cuda() - 1, slot_mapping=slots.cuda())
    c, out = cache.cuda(), torch.empty(n, nq, dtype=dtype, device="cuda")
    assert ops.window_step(out, proj.cuda(), c, meta, torch.empty(0, device="cuda"), sp, None, None, 1e-5, gate_off if gated else -1, factor,
                           None if sink_w is None else sink_w.cuda())
    assert torch.equal(c.cpu(), after)
    wrong = (out.double().cpu().view(n, heads, dim) - factor * want).abs() / (unit * factor * size)
    assert wrong.max() < 1, wrong.max()


# ------------------------------------------------------------------ experts whose used tiles are known
@gpu
@pytest.mark.parametrize("E,top,N,K,T", [(16, 2, 1024, 2048, 1), (16, 2, 2048, 1024, 3), (4, 3, 40, 648, 5), (5, 2, 24, 640, 70), (8, 1, 264, 632, 9), (3, 2, 16, 1032, 120)])
@pytest.mark.parametrize("act", [0, 1, 2])
def test_expert_gemm_of_known_tiles(E, top, N, K, T, act):
    """Tiles of one to 32 rows, as many as there are pairs launched at most; k and columns with remainders, choices that are no power of two, rows by slot."""
    g = torch.Generator().manual_seed(E * N + T)
    P, tile = T * top, 32
    x = torch.randn(T, K, generator=g).bfloat16().cuda()
    w = (torch.randn(E, N, K, generator=g) / K ** 0.5).bfloat16().cuda()
    ids = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(T)]).int().cuda()
    ops, cap = get_ops("cuda"), -(-(P + E * (tile - 1)) // tile) * tile
    slots, te, ps = (torch.empty(n, dtype=torch.int32, device="cuda") for n in (cap, cap // tile, P))
    ops.moe_align(ids.view(-1), E, tile, slots, te, ps)
    y = torch.einsum("pk,pnk->pn", x.double().repeat_interleave(top, 0), w.double()[ids.view(-1).long()])
    size = torch.einsum("pk,pnk->pn", x.double().abs().repeat_interleave(top, 0), w.double().abs()[ids.view(-1).long()])   # bounds the sums' rounding
    if act == 1:
        y, size = y.clamp(min=0) ** 2, 2 * y.abs() * size
    if act == 2:
        a, b = y.chunk(2, 1)
        y, size = a * torch.sigmoid(a) * b, (2 * size[:, : N // 2] * b.abs() + size[:, N // 2:] * a.abs())
    rows = torch.zeros(cap, K, dtype=torch.bfloat16, device="cuda")
    rows[ps.long()] = x.repeat_interleave(top, 0)
    for src, k in ((x, top), (rows, 0)):
        for tiles in (0, P):
            out = torch.full((cap, y.shape[1]), float("nan"), dtype=torch.bfloat16, device="cuda")
            ops.expert_gemm(out, src, w, slots, te, tile, k, act, pairs=P, tiles=tiles)
            assert ((out[ps.long()].double() - y).abs() <= 2.0 ** -8 * y.abs() + K * 2.0 ** -23 * size + 1e-30).all()


@gpu
@pytest.mark.parametrize("tile,dtype,E,top,N,K,T", [(64, torch.bfloat16, 5, 2, 264, 640, 70), (32, torch.bfloat16, 70, 1, 2048, 512, 70), (32, torch.bfloat16, 3, 2, 20, 72, 40),
                                                    (32, torch.float32, 4, 2, 40, 652, 9), (64, torch.float32, 3, 1, 72, 100, 150)])
def test_expert_gemm_of_known_tiles_by_the_other_kernels(tile, dtype, E, top, N, K, T):
    """Fewer tiles launched than the capacity has, by the kernels for larger tiles, for thousands of workgroups of few k, for odd columns and for 32 bits:
    the rows of all pairs, the same bits as with all tiles."""
    g = torch.Generator().manual_seed(E + N)
    P = T * top
    x, w = torch.randn(T, K, generator=g).to(dtype).cuda(), (torch.randn(E, N, K, generator=g) / K ** 0.5).to(dtype).cuda()
    ids = torch.arange(P).remainder(E).int().cuda()
    ops, cap = get_ops("cuda"), -(-(P + E * (tile - 1)) // tile) * tile
    slots, te, ps = (torch.empty(n, dtype=torch.int32, device="cuda") for n in (cap, cap // tile, P))
    ops.moe_align(ids, E, tile, slots, te, ps)
    used = int((te >= 0).sum())
    assert used <= P and ops._moe_lib.expert_rows_pay(used, P, N, K) == (K != 512)
    outs = []
    for tiles in (0, used, P):
        out = torch.full((cap, N), float("nan"), dtype=dtype, device="cuda")
        ops.expert_gemm(out, x, w, slots, te, tile, top, 0, pairs=P, tiles=tiles)
        outs.append(out[ps.long()])
    rows, mine = x.double().repeat_interleave(top, 0), w.double()[ids.long()]
    y, size = (torch.matmul(m, r[:, :, None])[..., 0] for m, r in ((mine, rows), (mine.abs(), rows.abs())))
    # a result of its type, and the sums' rounding
    assert ((outs[0].double() - y).abs() <= (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -23) * y.abs() + K * 2.0 ** -23 * size).all()
    assert torch.equal(outs[1], outs[0]) and torch.equal(outs[2], outs[0])


# ------------------------------------------------------------------ experts beside another product
@gpu
@pytest.mark.parametrize("M,N,K,parts", [(1, 8, 64, 1), (1, 3232, 2048, 1), (3, 2048, 4160, 2), (7, 1000, 4800, 1), (9, 2048, 1048, 1), (16, 1032, 520, 4), (24, 4104, 1024, 1),
                                         (33, 2000, 2048, 1), (41, 2048, 4096, 4), (48, 6152, 1096, 1), (64, 40, 8192, 2), (64, 4112, 2048, 1)])
@pytest.mark.parametrize("E,top,eN,eK,gather", [(16, 2, 1024, 2048, True), (3, 3, 40, 648, False)])
def test_experts_beside_a_product(M, N, K, parts, E, top, eN, eK, gather):
    """Every form of the dense product, tiles of one row to 32: the bits of the two launches."""
    g = torch.Generator().manual_seed(M + N + E)
    P, tile, ops = M * top, 32, get_ops("cuda")
    rnd = lambda *s: torch.randn(*s, generator=g).bfloat16().cuda()  # noqa: E731
    ids = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(M)]).int().cuda()
    cap = -(-(P + E * (tile - 1)) // tile) * tile
    slots, te, ps = (torch.empty(n, dtype=torch.int32, device="cuda") for n in (cap, cap // tile, P))
    ops.moe_align(ids.view(-1), E, tile, slots, te, ps)
    x, w, ex, ew = rnd(M, K + 8)[:, :K], rnd(N, K) / K ** 0.5, rnd(M if gather else cap, eK), rnd(E, eN, eK) / eK ** 0.5
    nan = lambda *s, dt=torch.bfloat16: torch.full(s, float("nan"), dtype=dt, device="cuda")  # noqa: E731
    k = top if gather else 0
    want_e, got_e = nan(cap, eN), nan(cap, eN)
    ops.expert_gemm(want_e, ex, ew, slots, te, tile, k, int(gather), pairs=P, tiles=P)
    dt = torch.float32 if parts > 1 else torch.bfloat16
    want, got = (nan(*((parts, M, N) if parts > 1 else (M, N)), dt=dt) for _ in range(2))
    if parts > 1:
        ops._seq.skinny_linear_parts(want, x, w, None)
    else:
        ops._seq.skinny_linear(want, x, w, None, -1, 0.0, 0.0)
    assert ops._seq.skinny_linear_experts(got, x, w, got_e, ex, ew, slots, te, k, int(gather), P, P)
    assert torch.equal(got, want) and torch.equal(got_e[ps.long()], want_e[ps.long()])
    # minGRU's product
    width, n = max(8, N // 4), M
    wide, bz, bx, state = rnd(3 * width, K) / K ** 0.5, *(torch.randn(*s, generator=g).cuda() for s in ((width,), (width,), (n + 2, width)))
    cu, ctx = torch.arange(n + 1, dtype=torch.int32, device="cuda"), torch.arange(n, dtype=torch.int32, device="cuda") % 3 + 1
    seq = torch.randperm(n + 2, generator=g)[:n].int().cuda()
    outs = []
    for beside in (False, True):
        y, s, e = nan(M, width), state.clone(), nan(cap, eN)
        if beside and ops._seq.mingru_product_experts(y, s, x, wide, bz, bx, cu, ctx, seq, e, ex, ew, slots, te, k, int(gather), P, P):
            assert M <= 32
        else:
            assert not beside or M > 32
            ops._seq.mingru_product(y, s, x, wide, bz, bx, cu, ctx, seq)
            e = want_e
        outs.append((y, s, e[ps.long()]))
    assert all(torch.equal(a, b) for a, b in zip(*outs))


@gpu
@pytest.mark.parametrize("M,N,K,E,eN,eK,together", [
    (33, 4096, 1024, 16, 4096, 1024, False), (40, 8192, 2048, 64, 1024, 512, False), (24, 6144, 2048, 32, 2048, 768, False), (48, 4096, 2048, 16, 2048, 1024, False),
    (33, 4096, 1024, 16, 1024, 2048, True), (40, 4096, 2048, 16, 1024, 1024, True), (24, 4096, 1024, 16, 4096, 1024, True), (8, 2048, 1024, 16, 4096, 1024, True), (9, 2048, 1024, 8, 4096, 1024, True), (64, 1024, 1024, 8, 1024, 512, True),
    (33, 6656, 2056, 16, 512, 2560, False), (40, 6640, 2560, 16, 512, 2560, True), (64, 6656, 2048, 8, 1024, 2048, True)])
def test_experts_beside_where_they_are_faster(M, N, K, E, eN, eK, together):
    """Thousands of experts' workgroups of a short k stay in a launch of their own where the dense product's leave room for two per compute unit, and any beside
    many dense ones of 33 rows and a long k; minGRU's product alike."""
    P, tile, ops = 2 * M, 32, get_ops("cuda")
    cap = -(-(P + E * (tile - 1)) // tile) * tile
    slots, te, ps = (torch.empty(n, dtype=torch.int32, device="cuda") for n in (cap, cap // tile, P))
    ops.moe_align((torch.arange(P, device="cuda") % E).int(), E, tile, slots, te, ps)
    zeros = lambda *s, dt=torch.bfloat16: torch.zeros(*s, dtype=dt, device="cuda")  # noqa: E731
    experts = (zeros(cap, eN), zeros(cap, eK), zeros(E, eN, eK), slots, te, 0, 0, P, P)
    assert ops._seq.skinny_linear_experts(zeros(M, N), zeros(M, K), zeros(N, K), *experts) == together
    if M <= 32:
        n, width = M, 2048
        seqs = [torch.arange(c, dtype=torch.int32, device="cuda") for c in (n + 1, n, n)]
        f32 = lambda *s: zeros(*s, dt=torch.float32)  # noqa: E731
        got = ops._seq.mingru_product_experts(zeros(M, width), f32(n, width), zeros(M, K), zeros(3 * width, K), f32(width), f32(width), *seqs, *experts)
        assert got == (eN // 16 * (cap // tile) <= (2200 if M <= 16 else 4000) or eK >= 2048)


class _Recorder:
    """Expert products that are asked for and never launched."""


def test_expert_steps_run_in_order_and_once():
    from hipserve.ops import ExpertSteps

    ran = []
    ops = _Recorder()
    ops.expert_gemm = lambda out, *a, **kw: ran.append(("alone", out))
    h = torch.zeros(1, 8, dtype=torch.bfloat16)
    steps = ExpertSteps(ops, [(i, h, h, h, h, 32, 1, True, 2, 2) for i in "ab"])
    assert not steps.take(lambda *e: False) and steps.take(lambda *e: ran.append(("beside", e[0])) or True)
    steps.finish()
    steps.finish()
    assert ran == [("beside", "a"), ("alone", "b")] and not steps.take(lambda *e: True)
    for other in (dict(tile=64), dict(x=h.float()), dict(pairs=0), dict(tiles=0), dict(act=2)):
        a = dict(out="a", x=h, w=h, slots=h, te=h, tile=32, k=1, act=0, pairs=2, tiles=2, **{})
        a.update(other)
        assert not ExpertSteps(ops, [tuple(a.values())]).take(lambda *e: True)


# ------------------------------------------------------------------ experts of prompts
@gpu
@pytest.mark.parametrize("counts", [[1, 128, 33, 0, 97], [64, 65, 300, 32], [31, 96, 16, 129, 2]])
@pytest.mark.parametrize("N,K,top", [(64, 64, 2), (200, 192, 3), (1024, 128, 2), (72, 640, 1), (2048, 1024, 2)])
@pytest.mark.parametrize("act", [0, 1])
def test_expert_gemm_of_prompt_tiles(counts, N, K, top, act):
    """Tiles of 128 slots: every number of row groups, columns that fill no tile, fewer stages than are in flight, rows by token and by slot."""
    from hipserve.models.mixers import MOE_TILE_PROMPT as tile

    g, E, ops = torch.Generator().manual_seed(sum(counts) + N), len(counts), get_ops("cuda")
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    P = -(-len(ids) // top) * top
    ids = torch.cat([ids, torch.full((P - len(ids),), E - 1)])[torch.randperm(P, generator=g)]
    cap = -(-(P + E * (tile - 1)) // tile) * tile
    slots, te, ps = (torch.empty(n, dtype=torch.int32, device="cuda") for n in (cap, cap // tile, P))
    ops.moe_align(ids.int().cuda(), E, tile, slots, te, ps)
    x, w = torch.randn(P // top, K + 8, generator=g).bfloat16().cuda()[:, :K], (torch.randn(E, N, K, generator=g) / K ** 0.5).bfloat16().cuda()
    rows, at = x.repeat_interleave(top, 0), ps.long()
    by_slot = torch.full((cap, K), float("nan"), dtype=torch.bfloat16, device="cuda")   # what lies in slots of no pair is not used
    by_slot[at] = rows
    y, size = (torch.stack([a[p] @ b[e].T for p, e in enumerate(ids.tolist())]) for a, b in ((rows.double(), w.double()), (rows.double().abs(), w.double().abs())))
    if act:
        y, size = y.clamp(min=0) ** 2, 2 * y.abs() * size
    for src, k in ((x, top), (by_slot, 0)):
        out = torch.full((cap, N), 7.0, dtype=torch.bfloat16, device="cuda")
        ops.expert_gemm(out, src, w, slots, te, tile, k, act, pairs=P, tiles=P)
        assert ((out[at].double() - y).abs() <= 2.0 ** -8 * y.abs() + K * 2.0 ** -23 * size + 1e-30).all()   # the result's type, the sums' rounding
        assert bool((out[slots < 0] == 7.0).all())


@gpu
@pytest.mark.parametrize("live", [[0], [33], [127], [1, 40, 63], [64, 96], [0, 31, 95], [5, 70, 126]])
@pytest.mark.parametrize("tile", [32, 64, 128])
def test_expert_gemm_of_tables_with_gaps(live, tile):
    """Slots without a pair ahead of ones with a pair, as a table of one's own may have them: all of these are computed, by the kernels of every tile."""
    g = torch.Generator().manual_seed(len(live) + tile)
    E, N, K, cap = 3, 72, 128, 256
    x, w = torch.randn(cap, K, generator=g).bfloat16().cuda(), torch.randn(E, N, K, generator=g).bfloat16().cuda() / K ** 0.5
    slots = torch.full((cap,), -1, dtype=torch.int32)
    at = torch.tensor([s + t for t in (0, 128) for s in live])
    slots[at] = torch.randperm(len(at), generator=g).int()
    te = (torch.arange(cap // tile) * tile // 128).int() + 1   # the first 128 slots are expert 1's, the rest expert 2's
    out = torch.full((cap, N), 7.0, dtype=torch.bfloat16, device="cuda")
    get_ops("cuda").expert_gemm(out, x, w, slots.cuda(), te.cuda(), tile, 1, 0)
    want = (x.double()[slots[at].long().cuda()][:, None] * w.double()[1 + at.cuda() // 128]).sum(-1)
    got = out[at.cuda()].double()
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -16 * K ** 0.5).all()   # rounded to bf16; sums of 128 products in 32 bits


def test_expert_plan_of_a_prompt():
    """What the three kernels were measured to take has the choice; sizes that were not looked at stay where they were."""
    from types import SimpleNamespace

    from hipserve.models.mixers import TableMoE
    from hipserve.ops import KernelOps

    rule = KernelOps()._expert_plan
    assert rule(132, 8, 512, 1024, False) == "rows" and rule(600, 8, 512, 1024, False) == "rows" and rule(2000, 8, 512, 1024, False) == "tiles"
    assert rule(400, 16, 1024, 2048, False) == "tiles" and rule(4096, 16, 1024, 2048, True) == "tiles" and rule(8000, 16, 1024, 2048, True) == "packed"
    assert rule(2048, 8, 2048, 4096, True) == "tiles" and rule(4000, 8, 2048, 4096, True) == "packed" and rule(4000, 8, 2048, 4096, False) == "tiles"
    assert rule(500, 64, 768, 1536, False) == "rows"
    ops = SimpleNamespace(name="hip", SKINNY_ROWS=64, expert_plan=lambda *a: "tiles")
    spec = lambda **kw: SimpleNamespace(**{**dict(experts=4, top=2, ff=512), **kw})  # noqa: E731
    planned = lambda dtype=torch.bfloat16, hidden=1024, ops=ops, **kw: TableMoE(spec(**kw), hidden, 9, "cpu", dtype, ops).planned  # noqa: E731
    none = float("inf")
    assert planned() == 128 and planned(torch.float32) == planned(ff=256) == planned(ff=520) == planned(hidden=1000) == planned(ops=None) == none
    tile = lambda P, **kw: TableMoE(spec(**kw), 1024, 9, "cpu", torch.bfloat16, ops)._tables(P, "cpu")[0]  # noqa: E731
    assert tile(128) == 32 and tile(129) == 128 and tile(1024, ff=256) == 64


@pytest.mark.parametrize("pairs,experts,ff,hidden,may_pack,want", [
    (320, 24, 2048, 4096, False, "rows"), (240, 24, 4096, 2560, False, "rows"), (441, 6, 896, 4096, False, "rows"), (525, 6, 1024, 1536, False, "rows"),
    (3088, 12, 4096, 768, True, "packed"), (426, 24, 576, 2048, False, "tiles"), (1524, 4, 640, 640, False, "tiles"), (2496, 8, 1024, 1024, True, "tiles"),
    (4806, 4, 2816, 512, True, "packed"), (3130, 4, 3840, 768, True, "packed"), (4806, 4, 2816, 512, False, "tiles")])
def test_expert_plan_where_a_choice_was_slower(pairs, experts, ff, hidden, may_pack, want):
    """Few pairs each, or little between the two by the model: tiles of 32; few groups of columns with many k: packed weights."""
    from hipserve.ops import KernelOps

    assert KernelOps()._expert_plan(pairs, experts, ff, hidden, may_pack) == want


# ------------------------------------------------------------------ window attention and the generalized delta rule in one launch
@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads,kv,dim,ctxs,mode,dheads,rank", [(1, 1, 64, [1], 0, 1, 32), (16, 4, 128, [1, 31, 33, 700], 1, 5, 64), (8, 2, 128, [16, 40, 290], 2, 32, 128),
                                                               (40, 2, 64, [5, 129, 400, 1], 1, 3, 96), (32, 8, 128, [90] * 20, 0, 64, 64)])
def test_window_and_delta_step_in_one_launch(heads, kv, dim, ctxs, mode, dheads, rank, dtype):
    """Fewer and more waves than the rule's four, several runs, each norm, a sequence without a row: the bits of the two launches."""
    from types import SimpleNamespace
    g = torch.Generator().manual_seed(heads * dim + rank)
    n, bs, nq, nk, N, eps = len(ctxs), 8, heads * dim, kv * dim, 64 * dheads, 1e-5
    sp = SimpleNamespace(maps=1, dim=dim, vdim=dim, heads=heads, kv_heads=kv, window=0, reach=0, scale=dim ** -0.5, sink=True, keep_first=0, softcap=0.0,
                         channel_gate=False, chunk=0, diff=0.0, q_size=nq, k_size=nk, v_size=nk, kv_from=None, qk_norm=mode == 1, head_norm=mode == 2,
                         unit_qk=False, v_norm=True, temp_coef=0.0, temp_every=0, scaling=None)
    width = -(-max(ctxs) // bs)
    bt = torch.randperm((n + 1) * width, generator=g).int().view(n + 1, width)
    cache = torch.randn((n + 1) * width, bs, 2 * nk, generator=g).to(dtype).cuda()
    both = torch.randn(n + 1, nq + 2 * nk + 5 * N + rank + 8, generator=g).to(dtype).cuda()   # the two projections side by side, a padding row
    left, right = both[:, :nq + 2 * nk], both[:, nq + 2 * nk:]
    w = [torch.rand(m, generator=g).cuda() + 0.5 for m in {1: (nq, nk), 2: (dim, dim)}[mode]] if mode else [None, None]
    meta = SimpleNamespace(seq_ctx=torch.tensor(ctxs + [3]).int().cuda(), seq_cu=torch.tensor([*range(n + 1), n]).int().cuda(), seq_bt=bt.cuda(),
                           num_decode=n + 1, num_prefill_tokens=0, max_ctx=max(ctxs), max_q=1, positions=torch.tensor([c - 1 for c in ctxs] + [0]).cuda(),
                           slot_mapping=torch.tensor([int(bt[s, (c - 1) // bs]) * bs + (c - 1) % bs for s, c in enumerate(ctxs)] + [-1]).cuda(),
                           seq_state=torch.randperm(n + 2, generator=g)[:n + 1].int().cuda())
    inv = (1e4 ** (-torch.arange(16).float() / 16)).cuda()
    S = torch.randn(n + 2, dheads, 64, 64, generator=g).cuda()
    w2 = (torch.randn(N, rank, generator=g) / rank ** 0.5).to(dtype).cuda()
    a_b, w0, nw = (torch.randn(N, generator=g).cuda() for _ in range(3))
    dsp, ops, outs = SimpleNamespace(heads=dheads, dim=64, size=N), get_ops("cuda"), []
    for one in (False, True):
        c, s, out = cache.clone(), S.clone(), torch.zeros(n + 1, nq + N, dtype=dtype, device="cuda")
        rule = (out[:, nq:], [s], right, w2, a_b, w0, nw, dsp, eps, meta, 1.25)
        beside = ops.delta_beside(*rule) if one else None
        assert ops.window_step(out[:, :nq], left, c, meta, inv, sp, *w, eps, -1, 0.75, beside=beside)
        assert beside.taken if one else ops.delta_rule_low(*rule)
        outs.append((out[:n], c, s))
    assert all(torch.equal(a, b) for a, b in zip(*outs)) and outs[0][0].isfinite().all()


@pytest.mark.parametrize("dim,ctx,rows,dheads,want", [
    (128, 300, 128, 32, False), (128, 230, 64, 64, False), (128, 230, 64, 32, False),              # up to 15 % slower in one launch
    (128, 230, 63, 32, True), (128, 100, 96, 48, True), (64, 300, 128, 32, True), (128, 230, 16, 32, True)])
def test_delta_step_apart_where_many_workgroups_wait(monkeypatch, dim, ctx, rows, dheads, want):
    """What window attention is offered and takes, by its runs and the rule's workgroups."""
    from types import SimpleNamespace

    from hipserve.ops import DeltaBeside, KernelOps
    ops, apart = KernelOps(), []
    monkeypatch.setattr(KernelOps, "_window_lib", SimpleNamespace(window_attention_decode_ok=lambda *a: True, window_attention_step=lambda *a: apart.append(a)))
    monkeypatch.setattr(KernelOps, "_delta", SimpleNamespace(window_delta_step=lambda *a: True))
    sp = SimpleNamespace(maps=1, dim=dim, vdim=dim, heads=16, kv_heads=4, reach=0, scale=1.0, window=0, sink=True, keep_first=0, softcap=0.0,
                         channel_gate=False, chunk=0)
    meta = SimpleNamespace(num_decode=rows, max_ctx=ctx, seq_cu=None, seq_ctx=None, seq_bt=None)
    beside = DeltaBeside((), rows * dheads)
    assert ops._window_decode(None, torch.empty(1, dtype=torch.bfloat16), None, meta, sp, -1, 1.0, None, (), beside)
    assert beside.taken == want and len(apart) == (not want)


@pytest.mark.parametrize("T,N,K,dtype,want", [(16, 2048, 4096, torch.float32, True), (17, 2048, 2048, torch.float32, False), (17, 2048, 2044, torch.float32, True),
                                              (32, 2112, 4096, torch.float32, True), (17, 2048, 4096, torch.bfloat16, True)])
def test_update_and_conv_apart_where_faster(monkeypatch, T, N, K, dtype, want):
    """The launch of a residual update takes the convolution's at the measured side of its bounds alone, and the update runs either way."""
    from types import SimpleNamespace
    from hipserve.ops import ConvBeside, KernelOps
    ops, ran = KernelOps(), []
    monkeypatch.setattr(KernelOps, "_delta", SimpleNamespace(skinny_update_conv=lambda *a: ran.append("both") or True))
    monkeypatch.setattr(KernelOps, "_moe_lib", SimpleNamespace(skinny_linear_update=lambda *a: ran.append("update")))
    ops.update_pays = lambda *a: True
    conv = ConvBeside(ops)
    conv.left = ()
    x, w, r = torch.empty(T, K, dtype=dtype), torch.empty(N, K, dtype=dtype), torch.empty(T, N)
    assert ops.linear_update(x, w, None, r, torch.empty(N), 1e-6, conv=conv) is not None
    assert ran == ["both" if want else "update"] and (conv.left is None) == want


@gpu
@pytest.mark.parametrize("T,N,K,C,dtype", [(1, 64, 512, 1, torch.bfloat16), (8, 1024, 6144, 513, torch.bfloat16), (9, 1024, 2048, 512, torch.float32),
                                           (16, 4096, 512, 96, torch.bfloat16), (17, 4096, 512, 96, torch.float32), (32, 1024, 3072, 1025, torch.bfloat16),
                                           (20, 2048, 256, 2048, torch.float32)])
def test_update_and_conv_in_one_launch(T, N, K, C, dtype):
    """A workgroup's channels and one more, a first step, sequences without a row, every size of a product's workgroups: the bits of the two launches."""
    from hipserve.ops import ConvBeside
    g = torch.Generator().manual_seed(T + N + C)
    ops, nseq = get_ops("cuda"), T + 2
    x, w, proj = (torch.randn(*s, generator=g).to(dtype).cuda() for s in ((T, K), (N, K), (T, C + 24)))
    norm, kept = torch.rand(N, generator=g).cuda(), torch.randn(nseq + 1, 3, C, generator=g).cuda()
    seqs = (torch.tensor([0, *range(T + 1), T]).int().cuda(), torch.randint(1, 3, (nseq,), generator=g).int().cuda(),
            torch.randperm(nseq + 1, generator=g)[:nseq].int().cuda())   # the first and the last have no row
    ops.update_pays = lambda *a: True
    outs = []
    for one in (False, True):
        conv, c, r = ConvBeside(ops), kept.clone(), torch.ones(T, N).cuda()
        conv.left = (c, proj, *seqs, 4)
        got = ops.linear_update(x, w, None, r, norm, 1e-6, conv=conv if one else None)
        assert (conv.left is None) == one
        conv.finish()
        outs.append((got.rows, got.squares, r, c))
    assert all(torch.equal(a, b) for a, b in zip(*outs)) and outs[0][0].isfinite().all()
    want = kept.clone()
    for s in range(1, T + 1):
        old = kept[seqs[2][s], 1:] * float(seqs[1][s] > 1)
        want[seqs[2][s]] = torch.cat([old, proj[s - 1:s, :C].float()])
    assert torch.equal(outs[0][3], want)
    conv.left = (kept[:, :2].contiguous(), proj, *seqs, 3)   # other taps are a launch of their own
    ops.linear_update(x, w, None, r, norm, 1e-6, conv=conv)
    assert conv.left is not None
