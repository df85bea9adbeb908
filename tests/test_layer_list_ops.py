"""Kernels of the layer-list decoders alone, at the sizes where their variants meet, against the reference ops."""
import pytest
import torch

from hipserve.ops import get_ops
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
