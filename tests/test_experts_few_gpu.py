"""The experts' kernels of steps with few rows against the ones for any step: the same bits, since the same sums are taken in the
same order (csrc/experts_few.hip, route and arrangement in one block, the gated norm with its row in registers)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("counts, N, K, form", [
    ([1, 16, 0, 17, 33], 48, 64, "relu2"), ([64, 65, 3], 40, 72, "plain"), ([1], 16, 8, "plain"), ([2, 0, 1, 31], 33, 456, "gated"),
    ([5, 40, 64], 17, 2048, "gated"), ([15, 32, 1], 100, 1032, "relu2"), ([3, 7], 200, 392, "scatter")])
def test_streamed_matrices_against_tiles(monkeypatch, counts, N, K, form):
    """Tiles with one row, whole and broken sixteens, several tiles an expert, experts without rows; columns and inner sizes off
    the kernel's units; operands by place and by row, results by place and by pair."""
    from runtime.kernels import ops
    rng = np.random.default_rng(N + K)
    experts, pairs = len(counts), sum(counts)
    order = rng.permutation(pairs)
    tiles = ops.expert_tiles(pairs, 1, experts)
    pair_of_pos, tile_expert, at, first = np.full(tiles * 64, -1, np.int32), np.full(tiles, -1, np.int32), 0, 0
    for e, n in enumerate(counts):
        pair_of_pos[at:at + n] = order[first:first + n]
        tile_expert[at // 64:at // 64 - (-n // 64)] = e
        at, first = at + -(-n // 64) * 64, first + n
    pp, te = torch.from_numpy(pair_of_pos).to(DEV), torch.from_numpy(tile_expert).to(DEV)
    gated, scatter = form == "gated", form == "scatter"
    w = torch.randn(experts, N * (2 if gated else 1), K, device=DEV, dtype=torch.bfloat16)
    a = torch.randn(tiles * 64 if scatter else -(-pairs // 2), K, device=DEV, dtype=torch.bfloat16)
    if scatter:
        a[pp < 0] = float("nan")                                  # (rows of padding are never read)
    outs = []
    for few in (10 ** 9, 0):
        monkeypatch.setattr(ops, "EXPERT_FEW_PAIRS", few)
        assert ops.experts_few_ok(a, w, tiles) == bool(few)
        out = torch.full((pairs if scatter else tiles * 64, N), 3.0, device=DEV, dtype=torch.float32 if form in ("plain", "scatter") else torch.bfloat16)
        if gated:
            ops.experts_gemm_gated(a, w, pp, te, out, (7.0, 1.702, 1.0), top=2)
        else:
            ops.experts_gemm(a, w, pp, te, out, top=0 if scatter else 2, scatter=scatter, act=form == "relu2")
        outs.append(out)
    assert torch.equal(*outs) and (not scatter) == bool((outs[0][pp < 0] == 3.0).all() if not scatter else False)
    place = int(np.flatnonzero(pair_of_pos >= 0)[-1])              # one place against 64 bits
    pair, e = pair_of_pos[place], tile_expert[place // 64]
    want = w[e].double() @ a[place if scatter else pair // 2].double()
    if form == "relu2":
        want = want.clamp(min=0) ** 2
    if not gated:
        got = outs[0][pair if scatter else place].double()
        assert ((got - want).abs().max() / want.abs().max()).item() < (1e-5 if form != "relu2" else 5e-3)


@pytest.mark.parametrize("rows, experts, top, bias", [(1, 1, 1, False), (24, 16, 2, True), (300, 16, 4, True), (33, 200, 16, False), (8192, 1, 1, False), (600, 16, 2, True)])
def test_route_and_arrangement_in_one_block(rows, experts, top, bias):
    from runtime.kernels import ops
    logits = torch.randn(rows, experts + 3, device=DEV)[:, 1:1 + experts]
    logits[rows // 2] = 0.5                                        # (a tie of everything)
    b = torch.randn(experts, device=DEV) if bias else None
    tiles = ops.expert_tiles(rows, top, experts)
    new = lambda *shape, dtype=torch.int32: torch.full(shape, 77, device=DEV, dtype=dtype)
    alone, together = [(new(rows, top), new(rows, top, dtype=torch.float32)) for _ in range(2)]
    places, tile_expert = new(tiles * 64), new(tiles)
    ops.experts_route(logits, b, top, *alone)
    ops.experts_route(logits, b, top, *together, places, tile_expert)
    assert all(torch.equal(x, y) for x, y in zip(alone, together))
    chosen, pp, te = together[0].cpu().numpy().reshape(-1), places.cpu().numpy(), tile_expert.cpu().numpy()
    assert sorted(pp[pp >= 0].tolist()) == list(range(rows * top))
    for tile, e in enumerate(te):
        run = pp[tile * 64:tile * 64 + 64]
        n = int((run >= 0).sum())
        assert (run[:n] >= 0).all() and (run[n:] == -1).all() and (n > 0) == (e >= 0) and (chosen[run[:n]] == e).all()


@pytest.mark.parametrize("dim", [1, 255, 1024, 1030, 2048, 2049, 4096])
def test_gated_norm_with_its_row_in_registers(dim):
    """Two choices take the form with the row in registers; a third of weight zero the general one: the same sums."""
    from runtime.kernels import ops
    rows = 5
    x, w, gb = torch.randn(rows, dim, device=DEV), torch.randn(dim, device=DEV), torch.randn(dim, device=DEV)
    y, g = torch.randn(rows, 3, dim, device=DEV), torch.randn(rows, dim + 2, device=DEV)[:, 1:1 + dim]
    share = torch.rand(rows, 3, device=DEV)
    share[:, 2] = 0.0
    got = []
    for top in (2, 3):
        xd, cast = x.clone(), torch.empty(rows, dim, device=DEV, dtype=torch.bfloat16)
        ops.gate_post_norm(xd, ops.WeightedRows(y[:, :top].reshape(rows * top, dim).contiguous(), share[:, :top].contiguous(), top), w, 1e-5, 2.0,
                           gate=g, gate_bias=gb, cast=cast)
        got.append((xd, cast))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    v = (share[:, :2, None].double() * y[:, :2].double()).sum(1) * torch.sigmoid(g.double() + gb.double()) + 2.0 * x.double()
    want = v * torch.rsqrt(v.square().mean(1, keepdim=True) + 1e-5) * w.double()
    assert ((got[0][0] - want).abs().max() / want.abs().max()).item() < 1e-5


def test_operands_on_the_host_are_refused():
    from runtime.kernels import ops
    w = torch.zeros(16, 16, 64, device=DEV, dtype=torch.bfloat16)
    tiles = ops.expert_tiles(2, 1, 16)
    pp, te = torch.full((tiles * 64,), -1, dtype=torch.int32, device=DEV), torch.full((tiles,), -1, dtype=torch.int32, device=DEV)
    a, out = torch.zeros(2, 64, dtype=torch.bfloat16), torch.zeros(tiles * 64, 16, device=DEV, dtype=torch.bfloat16)
    assert ops.experts_few_ok(a, w, tiles)
    with pytest.raises(ops.KernelError):
        ops.experts_gemm(a, w, pp, te, out, top=1)
    with pytest.raises(ops.KernelError):
        ops.experts_gemm_gated(a, w, pp, te, out[:, :8].contiguous(), (7.0, 1.0, 0.0), top=1)
