"""The ring products (bf16 products of many rows, csrc/gemm_ring.inc) against products in 64 bits: every tile at the edges of its
rows, columns and inner size, every epilogue, slices of the inner size and what adds them, and the rule that picks them."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
TILES = [64032, 64064, 64128, 128064, 96128, 128128, 160128, 192128, 224128, 256128, 64256, 96256, 128256, 160256, 192256, 224256, 256256, 288256]


@pytest.fixture(scope="module")
def ops():
    from runtime.kernels import ops
    return ops


def operands(M, N, K, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(M, K, generator=g, device=DEV).bfloat16(), torch.randn(N, K, generator=g, device=DEV).bfloat16(),
            torch.randn(M, N, generator=g, device=DEV))


def close(got, want, K, half=False):
    """Float accumulation of K products of standard normals: at most K roundings of half an ulp of a sum below 8 sqrt(K); a bf16
    result is rounded once more."""
    bound = K * 2.0 ** -24 * 8 * K ** 0.5 + 1e-6
    return ((got.double() - want).abs() <= bound + (2.0 ** -8 * want.abs() if half else 0.0)).all().item()


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("K", [64, 128, 320, 576])
def test_every_tile_at_its_edges(ops, tile, K):
    """Rows and columns that no tile divides (and fewer than a tile has), inner sizes of one step, of as many as the ring holds, and
    of more; the rows and columns that no tile owns stay."""
    rows, cols = tile // 1000, tile % 1000
    for M, N in ((2 * rows + 5, 2 * cols + 12), (7, 20)):
        a, w, r = operands(M, N, K, seed=K + M)
        want = a.double() @ w.double().T
        held = torch.full((M + 1, N + 8), 7.0, device=DEV)
        out = held[:M, :N]
        out.copy_(r)
        ops.gemm_ring(a, w, out, residual=out, tile=tile)
        assert close(out, want + r.double(), K) and (held[M:] == 7.0).all() and (held[:, N:] == 7.0).all()
        half = torch.full((M + 1, N + 8), 7.0, dtype=torch.bfloat16, device=DEV)
        ops.gemm_ring(a, w, half[:M, :N], tile=tile)
        assert close(half[:M, :N], want, K, half=True) and (half[M:] == 7.0).all() and (half[:, N:] == 7.0).all()
        ops.gemm_ring(a, w, half[:M, :N], act=3, tile=tile)                      # relu(z)^2 of the rounded product
        z = want.float().bfloat16().double().clamp(min=0.0)
        # z may round to the neighbouring bf16 (2^-7 of it, twice that of its square), the square is rounded (2^-8)
        assert (((half[:M, :N].double() - z * z).abs() <= 6 * 2.0 ** -8 * z * z + 1e-3).all()).item()
        inter = N // 2 // 4 * 4
        act = torch.full((M + 1, inter + 8), 7.0, dtype=torch.bfloat16, device=DEV)
        wg = torch.cat([w[:inter], w[-inter:]]).contiguous()
        gate, up = (x.float().bfloat16().double() for x in (a.double() @ wg[:inter].double().T, a.double() @ wg[inter:].double().T))
        for law in (None, (7.0, 1.702, 1.0)):
            ops.gemm_ring_gated(a, wg, act[:M, :inter], law, tile=tile)
            if law is None:
                ref = gate / (1 + torch.exp(-gate)) * up
            else:
                g, u = gate.clamp(max=7.0), up.clamp(-7.0, 7.0)
                ref = g / (1 + torch.exp(-1.702 * g)) * (u + 1.0)
            # gate and up may round to the neighbouring bf16 (2^-8 of each), and the result is rounded
            assert ((act[:M, :inter].double() - ref).abs() <= 2.0 ** -5 * ref.abs() + 2.0 ** -6 * (gate.abs() + up.abs()) + 1e-3).all()
            assert (act[M:] == 7.0).all() and (act[:, inter:] == 7.0).all()


@pytest.mark.parametrize("tile", [64064, 128128, 128256, 288256])
@pytest.mark.parametrize("slices", [1, 2, 3, 9])
def test_slices_and_the_norm_that_adds_them(ops, tile, slices):
    """Partial sums add up to the product; the norm of many rows equals, bit for bit, the sum made alone and the norm of it."""
    M, N, K = 131, 260, 576
    a, w, r = operands(M, N, K, seed=slices)
    parts = torch.full((slices * M * N + 8,), 7.0, device=DEV)
    ops.gemm_ring_partials(a, w, parts, slices, tile=tile)
    assert close(parts[:slices * M * N].view(slices, M, N).double().sum(0), a.double() @ w.double().T, K) and (parts[slices * M * N:] == 7.0).all()
    left = (ops.RingSums(parts, slices, M, N), 0)
    weight = 1 + 0.1 * torch.randn(N, device=DEV)
    for dtype in (torch.bfloat16, torch.float32):
        alone = ops.add_partials(r.clone(), left)
        want = ops.rmsnorm(alone, weight, torch.empty(M, N, dtype=dtype, device=DEV), 1e-5)
        x = r.clone()
        got = ops.rmsnorm_partials(x, left, weight, torch.empty(M, N, dtype=dtype, device=DEV), 1e-5)
        assert torch.equal(x, alone) and torch.equal(got, want)
        x = r.clone()
        centred = ops.layernorm_partials(x, left, weight, torch.empty(M, N, dtype=dtype, device=DEV), 1e-5)
        assert torch.equal(x, alone)
        ref = torch.nn.functional.layer_norm(alone.double(), (N,), weight.double(), eps=1e-5)
        assert (centred.double() - ref).abs().max().item() <= (2.0 ** -7 * ref.abs().max().item() if dtype == torch.bfloat16 else 1e-5)
    with pytest.raises(ops.KernelError):
        ops.add_partials(torch.zeros(M, N + 4, device=DEV), left)


def test_sums_of_calls_without_a_pool_lie_apart(ops, monkeypatch):
    """Two products that are cut, neither of them added yet, as callers on two streams have them that name no pool: each holds its own
    partial sums, and none lie in the buffers that such calls share."""
    M, N, K = 2000, 448, 8192
    a, w, r = operands(M, N, K)
    b = a.flip(0).contiguous()
    monkeypatch.setattr(ops, "DEFAULT_SCRATCH", ops.ScratchPool())
    left = [ops.gemm_unfinished(x, w, r) for x in (a, b)]
    x = r.clone()
    ops.gemm(a, w, x, residual=x)
    assert not any(kind == "wide" for kind, _, _ in ops.DEFAULT_SCRATCH.buffers)
    assert all(isinstance(sums, ops.RingSums) and sums.slices > 1 for sums, _ in left)
    got = [ops.add_partials(torch.zeros_like(r), part) for part in left]
    for rows, out in zip((a, b), got):
        assert close(out, rows.double() @ w.double().T, K)
    assert torch.equal(x, ops.add_partials(r.clone(), left[0]))


@pytest.mark.parametrize("dim", [4, 576, 1028, 8192])
def test_norm_of_sums_over_the_widths(ops, dim):
    M, slices = 5, 4
    parts, r, weight = torch.randn(slices, M, dim, device=DEV), torch.randn(M, dim, device=DEV), torch.randn(dim, device=DEV)
    left, x = (ops.RingSums(parts.view(-1), slices, M, dim), 0), r.clone()
    got = ops.rmsnorm_partials(x, left, weight, torch.empty(M, dim, device=DEV), 1e-5)
    want = parts[0] + parts[1] + parts[2] + parts[3] + r
    assert torch.equal(x, want) and torch.equal(got, ops.rmsnorm(want, weight, torch.empty(M, dim, device=DEV), 1e-5))


def test_norm_of_sums_with_weights_between_words(ops):
    """Norm weights that are views into one buffer, as a program may bind them: the sum and the norm, as two kernels."""
    M, N, K = 300, 260, 8192
    a, w, r = operands(M, N, K)
    held = torch.randn(2 * N + 2, device=DEV)
    weight, bias = held[1:1 + N], held[1 + N:1 + 2 * N]
    parts = torch.empty(2 * M * N, device=DEV)
    ops.gemm_ring_partials(a, w, parts, 2)
    product = (a.float() @ w.float().T).bfloat16()
    for left in ((ops.RingSums(parts, 2, M, N), 0), (parts, 2), (product, 0)):
        alone = ops.add_partials(r.clone(), left)
        for norm, alone_norm in ((lambda x, out: ops.rmsnorm_partials(x, left, weight, out, 1e-5), lambda x, out: ops.rmsnorm(x, weight, out, 1e-5)),
                                 (lambda x, out: ops.layernorm_partials(x, left, weight, out, 1e-5, bias=bias),
                                  lambda x, out: ops.layernorm(x, weight, out, 1e-5, bias=bias))):
            x = r.clone()
            got = norm(x, torch.empty(M, N, dtype=torch.bfloat16, device=DEV))
            assert torch.equal(x, alone) and torch.equal(got, alone_norm(alone, torch.empty_like(got)))


def test_what_is_not_taken(ops):
    a, w, r = operands(70, 64, 128)
    for bad in ((a[:, :96], w[:, :96], r), (a, w[:62], r[:, :62]), (a[:, 1:65], w[:, :64], r), (a.float(), w.float(), r),
                (a, w, torch.empty(64, 70, device=DEV).t())):
        with pytest.raises(ops.KernelError):
            ops.gemm_ring(*bad)
    with pytest.raises(ops.KernelError):
        ops.gemm_ring(a, w, r, tile=32064)
    with pytest.raises(ops.KernelError):
        ops.gemm_ring(a, w, torch.empty(70, 64, dtype=torch.bfloat16, device=DEV), residual=r)
    with pytest.raises(ops.KernelError):
        ops.gemm_ring_partials(a, w, torch.empty(70 * 64 * 2, device=DEV), 3)
    assert not ops.ring_fits(a[:, :96], w[:, :96], r) and ops.ring_fits(a, w, r)


@pytest.mark.parametrize("M, N, K", [(17, 16384, 2048), (33, 2048, 8192), (64, 2048, 8192), (65, 2048, 2048), (65, 4096, 2048), (700, 1024, 1024), (700, 960, 576), (1061, 576, 1536), (400, 2048, 1024)])
def test_calls_that_came_to_these_kernels_against_the_others(ops, M, N, K, monkeypatch):
    """The same calls with the ring products off: rows with a stride, results in views, the residual apart from the output."""
    a, w, r = operands(M, N, K, seed=M)
    wide = torch.randn(M, K + 64, device=DEV).bfloat16()
    wide[:, 64:] = a
    held = torch.zeros(M, N + 16, device=DEV)
    gu = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    assert ops.ring_ahead(M, w, fused=True, cut=True) and ops.ring_ahead(M, w, gated=True)

    def calls():
        x = r.clone()
        yield ops.gemm(wide[:, 64:], w, x, residual=x)
        yield ops.gemm(a, w, held[:, 16:], residual=r).clone()
        yield ops.gemm(a, w, torch.empty(M, N, device=DEV))
        yield ops.gemm(a, w, torch.empty(M, N, dtype=torch.bfloat16, device=DEV))
        yield ops.gemm_swiglu(a, w, torch.empty(M, N // 2, dtype=torch.bfloat16, device=DEV), gate_up=gu)
        yield ops.gemm_swiglu(a, w, torch.empty(M, N // 2, dtype=torch.bfloat16, device=DEV), gate_up=gu, law=ops.GELU_TANH_LAW)
        yield ops.gemm_gelu(a, w, torch.empty(M, N, dtype=torch.bfloat16, device=DEV), product=gu)
    here = list(calls())
    monkeypatch.setattr(ops, "RING_MIN_ROWS", 1 << 30)
    monkeypatch.setattr(ops, "RING_FEW_ROWS", 1 << 30)
    for i, (got, want) in enumerate(zip(here, calls())):
        scale = want.double().square().mean().sqrt().item()
        assert (got.double() - want.double()).norm().item() <= 2.0 ** -7 * want.double().norm().item(), i
        assert (got.double() - want.double()).abs().max().item() <= 2.0 ** -5 * max(scale, want.abs().max().item()), i


@pytest.mark.parametrize("kind", ["gelu", "gelu_tanh", "relu2"])
def test_activation_of_a_large_product_on_either_side_of_its_line(ops, kind):
    """As a kernel after the library's product and as the epilogue, which results in a view and calls without a buffer keep: the product
    rounded to bf16 either way, from sums of another order (one rounding apart), then the activation."""
    M, N, K = 3001, 8192, 2048
    a, w = operands(M, 8, K)[0], operands(N, 8, K, seed=1)[0] * 0.02
    product, out, held = (torch.empty(M, n, dtype=torch.bfloat16, device=DEV) for n in (N, N, N + 8))
    assert ops.activation_apart(a, w, out, product, kind)
    got = ops.gemm_gelu(a, w, out, kind, product=product)
    z = (a.float() @ w.float().T).double()
    act = {"gelu": lambda x: x * 0.5 * torch.erfc(-x / 2 ** 0.5), "gelu_tanh": lambda x: torch.nn.functional.gelu(x, approximate="tanh"),
           "relu2": lambda x: x.clamp(min=0).square()}[kind]
    want = act(z)
    # z is off by its rounding (2^-8 of it) and the sums' order (K 2^-24 of what a sum of 0.02 sqrt K passes through); slopes to 1.13, relu2 2 z
    slope = 2 * z.abs() if kind == "relu2" else 1.13
    bound = 2.0 ** -8 * want.abs() + (2.0 ** -8 * z.abs() + 1e-4) * (slope + 2.0 ** -8) + 1e-6
    for result in (got, ops.gemm_gelu(a, w, held[:, 8:], kind, product=product), ops.gemm_gelu(a, w, torch.empty_like(out), kind)):
        assert ((result.double() - want).abs() <= bound).all()


def test_a_product_is_asked_about_once(ops, monkeypatch):
    """A step that runs kernel by kernel waits for the host: a product's operands are looked at once, whatever it ends in."""
    a, w, r = operands(300, 2048, 576)
    a2, w2, _ = operands(300, 2048, 8192)                                       # (cut along its inner size)
    asked, ask = [], ops._ring_operands
    monkeypatch.setattr(ops, "_ring_operands", lambda *x: (asked.append(1), ask(*x))[1])
    monkeypatch.setattr(ops, "ring_fits", None)
    half = torch.empty(300, 2048, dtype=torch.bfloat16, device=DEV)
    calls = [lambda: ops.gemm(a, w, r, residual=r), lambda: ops.gemm(a, w, half), lambda: ops.gemm(a2, w2, r, residual=r),
             lambda: ops.gemm_swiglu(a, w, half[:, :1024].contiguous()), lambda: ops.gemm_unfinished(a, w, r, finish=True),
             lambda: ops.gemm_unfinished(a2, w2, r, finish=True)]
    results = [call() for call in calls]
    assert len(asked) == len(calls) and results[-2] is ops.ADDED and isinstance(results[-1][0], ops.RingSums)
    want = r + a.float() @ w.float().T
    assert ops.gemm_unfinished(a, w, r, finish=True) is ops.ADDED
    assert (r - want).abs().max() <= 1e-2


def test_models_that_route_rows_take_no_ring_products(ops, monkeypatch):
    """Every entry point given a pool without ring products, and a step of a model with experts: the bits are those of the other kernels."""
    from runtime.engine import ModelRunner, StepEntry, random_model
    asked, ask = [], ops._ring_operands
    monkeypatch.setattr(ops, "_ring_operands", lambda *x: (asked.append(1), ask(*x))[1])
    M, heads, dim = 500, 8, 64
    a, w, r = operands(M, 3 * heads * dim, 512)
    angle = torch.rand(M, dim // 2, device=DEV)
    cos, sin = angle.cos(), angle.sin()
    half = lambda cols: torch.empty(M, cols, dtype=torch.bfloat16, device=DEV)      # noqa: E731

    def calls(pool):
        yield lambda: ops.gemm(a, w, r.clone(), residual=r, scratch=pool)
        yield lambda: ops.gemm(a, w, half(w.shape[0]), scratch=pool)
        yield lambda: ops.gemm_swiglu(a, w, half(w.shape[0] // 2), scratch=pool)
        yield lambda: ops.gemm_gelu(a, w, half(w.shape[0]), scratch=pool, product=half(w.shape[0]))
        yield lambda: ops.gemm_for_norm(a, w, torch.empty_like(r), lambda n: torch.empty(n, device=DEV), scratch=pool)
        yield lambda: ops.gemm_unfinished(a, w, r.clone(), scratch=pool, finish=True)
    open_, closed = ops.ScratchPool(), ops.ScratchPool(ring=False)
    for i, call in enumerate(calls(open_)):
        call()
        assert len(asked) == i + 1
    kept = [call() for call in calls(closed)]
    assert len(asked) == i + 1 and kept[-1] is None
    assert ops.qkv_rope_fused_ok(a, w, dim, cos, False, open_) and not ops.qkv_rope_fused_ok(a, w, dim, cos, False, closed)
    with pytest.raises(ops.KernelError):
        ops.qkv_rope(a, w, half(heads * dim), torch.zeros(M, dtype=torch.int32, device=DEV), None, cos, sin, None, None, 3 * heads, 0, dim, 16, scratch=closed)
    mlp = {"kind": "moe", "expert": {"ff": 512}, "router": {"experts": 8, "top": 2}}
    raw = {"architecture": "Noresun", "vocab": 1024, "width": 1024, "postln_alpha": 2.0, "norm": {"eps": 1e-5}, "max_positions": 512,
           "embedding": {"scale": 1.0, "bigram": {"buckets": 509, "mul_prev": 13, "mul_cur": 5}},
           "layers": [{"type": "mingru", "mixer": {"width": 1024}, "mlp": mlp}] * 2}
    del asked[:]
    results = []
    for ring in (False, True):
        runner = ModelRunner(random_model(raw, seed=3, std=0.03), n_pages=40, page_size=16, max_requests=2)
        assert not runner.scratch.ring
        runner.scratch.ring = ring
        runner.create("a")
        results.append(runner.step([StepEntry("a", [i * 7 % 1024 for i in range(300)], [0, 150, 299])]).clone())
        assert bool(asked) == ring
    assert not torch.equal(*results)


def test_on_every_replay_of_a_captured_graph(ops):
    M, N, K = 300, 2048, 8192
    a, w, r = operands(M, N, K)
    a.mul_(0.1)
    x, gu = r.clone(), torch.empty(M, N // 2, dtype=torch.bfloat16, device=DEV)

    def step():
        ops.gemm(a, w, x, residual=x)
        ops.gemm_swiglu(a, w, gu)
    step()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    for i in range(4):
        a.copy_(torch.randn(M, K, device=DEV) * 0.1)
        x.copy_(r)
        step()
        torch.cuda.synchronize()
        want = x.clone(), gu.clone()
        x.copy_(r)
        gu.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(x, want[0]) and torch.equal(gu, want[1]), i


def test_gelu_of_every_bf16_number(ops):
    """The gelu of bf16 results against 64 bits over all bf16 numbers from 2^-20 to 16 and their negatives: rounded to the nearest
    bf16 but for sums near a tie (the kernel's 1.4e-5 relative at most against a rounding of 2^-9: fewer than one in a hundred), never
    further than the next one."""
    bits = torch.arange(0x3580, 0x4181, dtype=torch.int32)
    z = torch.cat([bits, bits | 0x8000]).to(torch.int16).view(torch.bfloat16).to(DEV)
    want = 0.5 * z.double() * torch.special.erfc(-z.double() * 0.5 ** 0.5)
    want = torch.where(want.abs() < 1e-36, 0.0, want)
    got = ops.gelu(z, torch.empty_like(z)).double()
    got = torch.where(got.abs() < 1e-36, 0.0, got)
    near = want.float().bfloat16().double()
    assert ((got - want).abs() <= 2.0 ** -7 * want.abs()).all() and (got != near).float().mean().item() < 0.01
    special = torch.tensor([0.0, float("inf"), float("nan")], dtype=torch.bfloat16, device=DEV)
    out = ops.gelu(special, torch.empty_like(special))
    assert out[0] == 0 and out[1] == float("inf") and out[2].isnan()


@pytest.mark.parametrize("M, K, heads, kv, dim, page", [(65, 64, 3, 1, 32, 16), (200, 576, 9, 3, 64, 16), (97, 128, 2, 2, 96, 8), (300, 512, 4, 0, 64, 16),
                                                        (131, 256, 8, 2, 128, 32), (80, 192, 1, 1, 160, 16), (700, 576, 9, 3, 64, 16), (17, 2048, 32, 32, 64, 16), (64, 4096, 32, 8, 128, 16)])
def test_rotation_and_cache_write_in_the_epilogue(ops, M, K, heads, kv, dim, page, monkeypatch):
    """Against the product and the rotary kernel: rows in runs of slots and out of order, rows without a slot, whole pages that stay."""
    a, w, _ = operands(M, (heads + 2 * kv) * dim, K, seed=M)
    g = torch.Generator(device=DEV).manual_seed(M)
    angle = torch.rand(2 * M, dim // 2, generator=g, device=DEV) * 6.3
    cos, sin = angle.cos().contiguous(), angle.sin().contiguous()
    positions = torch.randint(0, 2 * M, (M,), generator=g, device=DEV, dtype=torch.int32)
    pages = M // page + 3
    slots = torch.arange(M, device=DEV, dtype=torch.int32) + page + 3
    slots[M // 2:] = slots[M // 2:].flip(0).clone()
    slots[::17] = -1

    def run():
        keys = torch.full((pages, max(kv, 1), page, dim), 7.0, dtype=torch.bfloat16, device=DEV)
        values = torch.full((pages, max(kv, 1), dim, page), 7.0, dtype=torch.bfloat16, device=DEV)
        pools = (keys, values) if kv else (None, None)
        if ops.qkv_rope_fused_ok(a, w, dim, cos, False):
            q = ops.qkv_rope(a, w, torch.empty(M, heads * dim, dtype=torch.bfloat16, device=DEV), positions, slots if kv else None, cos, sin,
                             *pools, heads, kv, dim, page)
        else:
            rows = ops.gemm(a, w, torch.empty(M, w.shape[0], dtype=torch.bfloat16, device=DEV))
            ops.rope_scatter(rows, positions, slots if kv else None, cos, sin, *pools, heads, kv, dim, page)
            q = rows[:, :heads * dim]
        return q.double(), keys.double(), values.double()
    assert ops.ring_rope_ok(a, w, dim, cos)
    here = run()
    monkeypatch.setattr(ops, "RING_MIN_ROWS", 1 << 30)
    monkeypatch.setattr(ops, "RING_FEW_ROWS", 1 << 30)
    for got, want in zip(here, run()):
        # the other path rounds the product to bf16 before it turns it (2^-8 of either coordinate of a pair) and both round the result
        assert ((got - want).abs() <= 2.0 ** -7 * want.abs() + 2.0 ** -8 * 2 * want.abs().max()).all()
        assert (got - want).norm() <= 2.0 ** -7 * want.norm()


def test_a_result_may_lie_where_the_rows_were(ops):
    """Gate and up, and the gelu, of large weights into the buffer of their rows: the product goes to a buffer of its own first, as it
    did before there were ring products, whose blocks would read rows that others have replaced."""
    a, w, _ = operands(300, 4096, 2048)
    for call, inner in ((lambda x, out: ops.gemm_swiglu(x, w, out), w), (lambda x, out: ops.gemm_gelu(x, w[:2048], out, product=torch.empty_like(out)), w)):
        for shift in (0, 64 * 2048):                    # all of it, and rows that overlap by all but 64
            held = torch.empty(300 * 2048 + shift, dtype=torch.bfloat16, device=DEV)
            x, out = held[:300 * 2048].view(300, 2048).copy_(a), held[shift:].view(300, 2048)
            assert not ops.ring_fits(x, inner, out) and ops.ring_fits(a, inner, torch.empty_like(a))
            want = call(a, torch.empty_like(a)).double()
            got = call(x, out).double()
            # (sums in another order, rounded to bf16 twice: gate and up, and the result)
            assert (got - want).norm() <= 2.0 ** -7 * want.norm() and (got - want).abs().max() <= 2.0 ** -5 * want.abs().max()
    beside = torch.empty(300, 4096, dtype=torch.bfloat16, device=DEV)
    assert not ops.ring_fits(beside[:, :2048], w, beside[:, 2048:])         # (columns of the same rows: told apart no further)


@pytest.mark.parametrize("odd", ["cos", "sin", "q", "keys"])
@pytest.mark.parametrize("M", [64, 200])
def test_rotation_with_operands_between_words(ops, M, odd):
    """Tables, queries or key pages that do not begin on the words the epilogue moves take another route: the layer's projection beside the
    rotary kernel, or up to 64 rows the kernels of few rows."""
    heads, kv, dim, page, K = 32, 32, 64, 16, 2048

    def at_odd(t, name):
        flat = torch.empty(t.numel() + 2, dtype=t.dtype, device=DEV)
        view = flat[1:1 + t.numel()].view(t.shape) if odd == name else flat[:t.numel()].view(t.shape)
        return view.copy_(t)
    a, w, _ = operands(M, (heads + 2 * kv) * dim, K, seed=M)
    angle = torch.rand(2 * M, dim // 2, device=DEV) * 6.3
    cos, sin = at_odd(angle.cos(), "cos"), at_odd(angle.sin(), "sin")
    positions, slots = torch.arange(M, device=DEV, dtype=torch.int32), torch.arange(M, device=DEV, dtype=torch.int32)
    keys = at_odd(torch.zeros(M // page + 1, kv, page, dim, dtype=torch.bfloat16, device=DEV), "keys")
    values = torch.zeros(M // page + 1, kv, dim, page, dtype=torch.bfloat16, device=DEV)
    q = at_odd(torch.zeros(M, heads * dim, dtype=torch.bfloat16, device=DEV), "q")
    if M > 64:
        if odd in ("cos", "sin"):           # (what PagedAttention asks before it chooses)
            assert not ops.qkv_rope_fused_ok(a, w, dim, cos, False, None, sin)
        with pytest.raises(ops.KernelError):
            ops.qkv_rope(a, w, q, positions, slots, cos, sin, keys, values, heads, kv, dim, page)
        return
    ops.qkv_rope(a, w, q, positions, slots, cos, sin, keys, values, heads, kv, dim, page)
    rows = ops.gemm(a, w, torch.empty(M, w.shape[0], dtype=torch.bfloat16, device=DEV))
    ref_keys, ref_values = torch.zeros_like(keys), torch.zeros_like(values)
    ops.rope_scatter(rows, positions, slots, angle.cos(), angle.sin(), ref_keys, ref_values, heads, kv, dim, page)
    for got, want in ((q, rows[:, :heads * dim]), (keys, ref_keys), (values, ref_values)):
        # (rounded to bf16 before the turn on one side only, and both round the result: as in the test above)
        assert ((got.double() - want.double()).abs() <= 2.0 ** -7 * want.double().abs() + 2.0 ** -8 * 2 * want.double().abs().max()).all()


@pytest.mark.parametrize("law", [None, (7.0, 1.702, 1.0), (-1.0, 0.0, 0.0)])
def test_gates_of_every_size_against_64_bits(law):
    """Gates from -1e30 to 1e30 with both signs' smallest, and infinite ones, as products with one term: the activation's own error stays
    below what rounding its result to bf16, eight bits, may cost (2^-8 of it, and 4e-6 for the exponential, whose argument the other two laws
    round before it, times its size)."""
    from runtime.kernels import ops
    k, inter = 64, 128
    a = torch.zeros(80, k, device="cuda:0", dtype=torch.bfloat16)
    for m in range(80):
        a[m, m % k] = 1.0
    g = torch.randn(k, inter, device="cuda:0") * torch.logspace(-3, 1.7, k, device="cuda:0")[:, None]
    g[0, :12] = torch.tensor([0.0, -0.0, 1e-30, -1e-30, 1e-4, -1e-4, 80.0, -80.0, 1000.0, -1000.0, 1e30, -1e30], device="cuda:0")
    g[1, :7] = torch.tensor([-86.0, -87.5, -88.0, -88.5, -89.0, 88.0, 89.0], device="cuda:0")
    g[63] = torch.where(torch.arange(inter, device="cuda:0") % 2 == 0, 3e38, -3e38)
    u = torch.randn(k, inter, device="cuda:0")
    w = torch.cat((g.t(), u.t())).bfloat16().contiguous()
    a[63, 63] = 3e38                                          # (3e38 squared is past the largest float: gates of plus and minus infinity)
    w[inter:, 63] = 1e-38
    out = torch.empty(80, inter, device="cuda:0", dtype=torch.bfloat16)
    ops.gemm_ring_gated(a, w, out, law)
    rows = torch.arange(80, device="cuda:0") % k
    gate, up = w[:inter].t().double()[rows], w[inter:].t().double()[rows]
    gate[rows == 63] *= float("inf")
    up[rows == 63] = (w[inter:, 63].double() * a[63, 63].double()).bfloat16().double()
    limit, slope, shift = law or (0.0, 0.0, 0.0)
    if limit > 0:
        gate, up = gate.clamp(max=limit), up.clamp(-limit, limit) + shift
    z = slope * gate if limit > 0 else 1.5957691216057308 * (gate + 0.044715 * gate ** 3) if limit < 0 else gate
    want, got = gate * torch.sigmoid(z) * up, out.double()
    dull = want.isnan() | want.isinf()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got[want.isinf()], want[want.isinf()])
    # (where exp(-z) is past the largest float the sigmoid is 0; results below the smallest normal number may be)
    bound = want.abs() * (2.0 ** -8 + 4e-6 + 2.0 ** -22 * z.abs().clamp(max=88.0) + (z < -88.72).double()) + 2.0 ** -126
    assert ((got - want).abs() <= bound)[~dull].all()
    near = (z < -87.0) & (z > -88.72)
    assert law is not None or (near.any() and (got[near] != 0).all())
