"""Activations in the epilogues of bfloat16 products (gate and up rows that stand one behind the other; the square of relu): the same
bits as the product in 32 bits and the activation's own kernel, and close to 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def operands(rows, n, k, seed):
    gen = torch.Generator().manual_seed(seed)
    return (torch.randn((rows, k), generator=gen).to(torch.bfloat16).to(DEV),
            (torch.randn((n, k), generator=gen) * k ** -0.5).to(torch.bfloat16).to(DEV))


def gated(g, u, act, limit):
    if act:
        return g / (1 + torch.exp(-g)) * u
    g, u = g.clamp(max=limit), u.clamp(-limit, limit)
    return g / (1 + torch.exp(-1.702 * g)) * (u + 1)


# widths that end inside a run of 32 and inside a tile, that are no multiple of eight; one k tile and several; groups of no, one and many rows
@pytest.mark.parametrize("counts,f,k", [([5, 0, 1, 300], 96, 64), ([257, 40, 128], 100, 192), ([64, 700], 517, 128), ([2048], 1024, 256)])
@pytest.mark.parametrize("variant", [2, 12, 13])
@pytest.mark.parametrize("act,limit", [(1, 0.0), (0, 0.7)])
def test_groups(counts, f, k, variant, act, limit):
    from minfer_amd.kernels import ops
    rows = sum(counts)
    x, w = operands(rows, 2 * f * len(counts), k, rows + f)
    w = w.view(len(counts), 2 * f, k)
    groups = torch.tensor(ops.row_groups(counts, variant), dtype=torch.int32, device=DEV)
    sums = torch.empty((rows, 2 * f), device=DEV)
    ops.linear_grouped(x, w, groups, variant, sums)
    want = torch.empty((rows, f), dtype=torch.bfloat16, device=DEV)
    ops.moe_act(sums, torch.ones((rows, 1), device=DEV), want, limit, act)
    out = torch.full((rows, f), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.linear_grouped_gated(x, w, groups, variant, out, limit, act)
    assert torch.equal(out, want)
    first = 0
    for e, c in enumerate(counts):
        z = x[first:first + c].double() @ w[e].double().t()
        ref = gated(z[:, :f], z[:, f:], act, limit)
        assert ((out[first:first + c].double() - ref).abs() <= ref.abs() * 2.0 ** -8 + 1e-5).all()
        first += c


@pytest.mark.parametrize("m,f,k", [(65, 4096, 128), (300, 8200, 64), (2048, 1000, 192), (2048, 4096, 64), (1000, 16385, 64)])
@pytest.mark.parametrize("z_rows", [0, 1, 16])
def test_one_product(m, f, k, z_rows):
    from minfer_amd.kernels import ops
    x, w = operands(m, 2 * f + z_rows, k, m + f)
    assert ops.linear_gated_takes(m, f, k)
    sums = torch.empty((m, 2 * f + max(1, z_rows)), device=DEV)
    plain = torch.empty((m, 2 * f), device=DEV)
    ops.linear(x, w[:2 * f], None, plain)
    sums[:, :2 * f] = plain
    z = None
    if z_rows:
        z = torch.empty((m, z_rows), device=DEV)
        ops.linear(x, w[2 * f:], None, z)
        sums[:, 2 * f:] = z
    else:
        sums[:, 2 * f:] = 1e30                                           # sigmoid 1
    want = torch.empty((m, f), dtype=torch.bfloat16, device=DEV)
    ops.gated_expert_act(sums, want)
    out = torch.full((m, f), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.linear_gated(x, w[:2 * f], out, act=1, gate_logits=z)
    assert torch.equal(out, want)


# the kernels by rows: register-resident, rolling, guarded; K split and staged, ring, 64 x 64 tiles, panels; tiles of every size, of
# operands that are not aligned, with K cut
@pytest.mark.parametrize("m,n,k", [(1, 4096, 1024), (8, 8192, 2048), (16, 300, 320), (3, 500, 100), (20, 4096, 2048), (33, 300, 200), (40, 1000, 512),
                                   (64, 40960, 64), (65, 40000, 64), (100, 500, 100), (300, 1000, 1024), (2048, 8192, 256), (2048, 896, 4864),
                                   (128, 1024, 8192)])
def test_square_of_relu(m, n, k):
    from minfer_amd.kernels import ops
    x, w = operands(m, n, k, m + n + k)
    for tiled in (None, ops.tile_weight(w)) if k % 32 == 0 and m <= 64 else (None,):
        half, out = (torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(2))
        b = torch.randn(n, device=DEV)
        ops.linear(x, w, b, out, tiled=tiled, relu2=True)
        z = x.double() @ w.double().t() + b.double()
        ref = z.clamp(min=0) ** 2
        tol = 4 * 2.0 ** -20 * k ** 0.5                                  # of z: 32-bit sums of exact products of size one and below
        assert ((out.double() - ref).abs() <= ref * 2.0 ** -8 + 2 * tol * ref.sqrt() + tol ** 2).all()
        if m <= 64 or ops.tile_plan(m, n, k, ops.EPI_RELU2) == ops.tile_plan(m, n, k, ops.EPI_F32):   # K cut alike: the very bits
            sums, want = torch.empty((m, n), device=DEV), torch.empty_like(out)
            ops.linear(x, w, b, sums, tiled=tiled)
            ops.relu2(sums, want)
            assert torch.equal(out, want)
        ops.linear(x, w, b, half, tiled=tiled)                           # (whose epilogue is the plain one)
        assert ((half.double() - z).abs() <= z.abs() * 2.0 ** -8 + tol).all()


def test_activations_that_are_none():
    """What `moe_act` refuses these refuse, and one product's clamped form without a limit, before anything is launched."""
    from minfer_amd.kernels import ops
    x, w = operands(128, 256, 64, 1)
    groups = torch.tensor(ops.row_groups([128], 2), dtype=torch.int32, device=DEV)
    out = torch.full((128, 128), 7.0, dtype=torch.bfloat16, device=DEV)
    for act, limit in ((2, 1.0), (-1, 1.0), (0, 0.0), (0, -1.0), (0, float("nan"))):
        with pytest.raises(ops.KernelError):
            ops.linear_gated(x, w, out, limit=limit, act=act)
    for act in (2, -1):
        with pytest.raises(ops.KernelError):
            ops.moe_act(torch.zeros((128, 256), device=DEV), torch.ones((128, 1), device=DEV), out, 1.0, act)
        with pytest.raises(ops.KernelError):
            ops.linear_grouped_gated(x, w.view(1, 256, 64), groups, 2, out, 1.0, act)
    assert (out == 7.0).all()


@pytest.mark.parametrize("offset", [0, 1])
def test_shared_expert(offset):
    """The expert every token takes, by the joined kernel and, for rows that stand off 16 bytes, by product and kernel."""
    from types import SimpleNamespace

    from minfer_amd.kernels import ops
    from minfer_amd.parts.moe import SharedExpert
    m, f, k = 1024, 2048, 64
    assert ops.linear_gated_takes(m, f, k) and ops.linear_gated_pays(m, f, 2 * f + 16, k)
    flat, w = operands(m * k + 8, 1, 1, 5)[0].view(-1), operands(1, 2 * f + 1, k, 6)[1]
    x = flat[offset:offset + m * k].view(m, k)
    down = operands(1, k, f, 7)[1]
    expert = SharedExpert(dict(stem="e", weight="z", intermediate_size=f), k, SimpleNamespace(dtype=torch.bfloat16))
    expert.load({"e.gate": w[:f], "e.up": w[f:2 * f], "z": w[2 * f:], "e.down": down}.__getitem__)
    h = torch.zeros((m, k), device=DEV)
    expert.forward(x, h, True)
    z = x.double() @ w.double().t()
    y = gated(z[:, :f], z[:, f:2 * f], 1, 0.0) / (1 + torch.exp(-z[:, 2 * f:]))
    want, bound = y @ down.double().t(), y.abs() @ down.double().abs().t() * 2.0 ** -8          # each y rounded to bfloat16
    assert ((h.double() - want).abs() <= bound + 1e-4).all()
