"""Who may finish whose norm: the rules by which a block leaves the norm between two products to the products themselves, with the
kernels' places taken by torch on the CPU."""
from types import SimpleNamespace

import pytest
import torch

ROWS, WIDTH = 65, 8


@pytest.fixture
def ctx(monkeypatch):
    """A step context whose products always may leave the next norm."""
    from runtime.engine.context import StepContext, Workspace
    from runtime.kernels import ops

    def gemm(a, w, out, residual=None, scratch=None):
        return out.copy_(a.float() @ w.float().T + (0.0 if residual is None else residual))

    def unfinished(a, w, residual, scratch=None, finish=False, leave=None):
        to = None if leave is None or a.shape[0] < ROWS else leave(a, w, residual, ())
        if to is not None:
            gemm(a, w, residual, residual)
            to[1].copy_(residual * to[0])
            to[2].copy_((residual * residual).sum(1)[None])
            return ops.ADDED

    def rmsnorm(x, weight, out, eps, rows=None):
        return out.copy_(x * torch.rsqrt((x * x).mean(1, keepdim=True) + eps) * weight)
    for name, fake in (("gemm", gemm), ("gemm_unfinished", unfinished), ("ring_normed_parts", lambda *a: 1), ("rmsnorm", rmsnorm), ("swiglu_fused_ok", lambda *a: True), ("gemm_swiglu", lambda h, w, out, **k: out.zero_())):
        monkeypatch.setattr(ops, name, fake)
    runner = SimpleNamespace(cache=None, model=SimpleNamespace(dtype=torch.bfloat16), device="cpu", scratch=None, workspace=Workspace("cpu"))
    return StepContext(runner)


def weights(seed):
    return torch.randn(WIDTH, WIDTH, generator=torch.Generator().manual_seed(seed)).bfloat16()


def rms(seed):
    from runtime.parts import RMSNorm
    norm = RMSNorm("n", WIDTH, 1e-5)
    norm.weight = 1.0 + 0.3 * torch.randn(WIDTH, generator=torch.Generator().manual_seed(seed))
    return norm


def read(part, h):
    """What a toy part does with the rows that it is given: their normed form, kept in `got`, and what they were, in `kinds`."""
    from runtime.kernels import ops
    part.kinds.append(type(h).__name__)
    if isinstance(h, ops.ScaledRows):
        h = h.rows.float() * torch.rsqrt(h.sums.sum(0)[:, None] / WIDTH + h.eps)
    part.got.append(h.float().clone())
    return h.bfloat16()


def toys():
    """A mixer and a feed-forward that end with a product and can finish the norm of their rows; with `after` they add that behind the product
    and do not say that it is the last."""
    from runtime.parts.base import FeedForward, Mixer

    class Toy:
        def __init__(self, seed, after=0.0):
            self.w, self.after, self.got, self.kinds = weights(seed), after, [], []

        def takes_scaled(self, rows, ctx):
            return True

        def forward(self, h, residual, ctx, *site, norm=None):
            residual = ctx.add_product(read(self, h), self.w, residual, **({} if self.after else {"last": self}))
            return residual.add_(self.after) if self.after else residual
    return type("ToyMixer", (Toy, Mixer), {}), type("ToyFFN", (Toy, FeedForward), {})


def run(ctx, layers, tap=None, rows=ROWS):
    """Runs the layers as a model does; returns the rows after them and the normed rows that every sublayer should have read."""
    from runtime.models import Model
    torch.manual_seed(0)
    x = torch.randn(rows, WIDTH)
    ctx.layer_tap = tap
    ctx.logit_rows = torch.empty(0)
    model = Model(None, SimpleNamespace(forward=lambda c: x), layers, None, None, max_positions=1, vocab_size=1)
    model.forward(ctx)
    return x


def norm_of(norm, x):
    return x * torch.rsqrt((x * x).mean(1, keepdim=True) + norm.eps) * norm.weight


def layers_of(n, block=None, mixer=None, ffn=None, after={}):
    from runtime.parts import PreNormBlock
    ToyMixer, ToyFFN = toys()
    return [(block or PreNormBlock)(rms(i), (mixer or ToyMixer)(10 + i, after.get("mixer", 0.0)), rms(20 + i), (ffn or ToyFFN)(30 + i, after.get("ffn", 0.0)))
            for i in range(n)]


def watch(blocks, stream=None):
    """What every sublayer should read, found when it runs: [(part, normed rows)]; `stream` receives the residual rows."""
    seen = []
    for block in blocks:
        for part, norm in ((block.mixer, block.mixer_norm), (block.ffn, block.ffn_norm)):
            def spy(h, residual, *rest, part=part, norm=norm, real=part.forward, **kw):
                seen.append((part, norm_of(norm, residual)))
                if stream is not None:
                    stream[:] = [residual]
                return real(h, residual, *rest, **kw)
            part.forward = spy
    return seen


def right(seen, count):
    """Whether every sublayer read what it should (bf16 rows, rounded before their factor or after it)."""
    runs, ok = {}, len(seen) == count
    for part, want in seen:
        n = runs[part] = runs.get(part, -1) + 1
        ok = ok and bool(((part.got[n] - want).abs() <= 0.01 * want.abs() + 1e-6).all())
    return ok


def kinds(blocks):
    return [part.kinds for block in blocks for part in (block.mixer, block.ffn)]


def test_parts_that_end_with_their_product_leave_the_next_norm(ctx):
    blocks = layers_of(2)
    seen = watch(blocks)
    run(ctx, blocks)
    assert right(seen, 4) and kinds(blocks) == [["Tensor"], ["ScaledRows"], ["ScaledRows"], ["ScaledRows"]]


def test_a_part_around_another_is_given_normed_rows(ctx):
    """A feed-forward that answers for another one in all but its forward: what the inner one can finish is not said for the outer one."""
    class Around:
        def __init__(self, inner):
            self.inner = inner

        def __getattr__(self, name):
            return getattr(self.inner, name)

        def forward(self, h, residual, ctx, norm=None):
            return self.inner.forward(h * 1.0, residual, ctx)
    blocks = layers_of(2)
    seen = watch(blocks)
    for block in blocks:
        block.ffn = Around(block.ffn)
    run(ctx, blocks)
    assert right(seen, 4) and kinds(blocks) == [["Tensor"]] * 4


def test_what_others_add_before_a_block_is_in_its_first_norm(ctx):
    """An arrangement made of the pre-norm one, or around it, that adds to the rows before the block reads them: the norm that the block
    before left was of the rows as they were."""
    from runtime.parts import PreNormBlock

    class Before(PreNormBlock):
        def forward(self, residual, ctx, site):
            return super().forward(residual.add_(0.7), ctx, site)

    class Around:
        def __init__(self, inner):
            self.inner = inner

        def __getattr__(self, name):
            return getattr(self.inner, name)

        def forward(self, residual, ctx, site):
            return self.inner.forward(residual.add_(0.7), ctx, site)
    for block, outer in ((Before, None), (None, Around)):
        first, last = layers_of(1) + layers_of(1, block=block)
        seen = watch([first, last])
        run(ctx, [first, outer(last) if outer else last])
        assert right(seen, 4)


def test_products_that_leave_no_norm_are_not_asked_who_reads_it(ctx, monkeypatch):
    """Finding the reader costs host time where a step runs kernel by kernel: only a product that may leave its norm pays for it."""
    from runtime.parts import PreNormBlock
    blocks, asked = layers_of(2), []
    seen, real = watch(blocks), PreNormBlock.reads_next
    monkeypatch.setattr(PreNormBlock, "reads_next", lambda self, *a: (asked.append(self), real(self, *a))[1])
    run(ctx, blocks, rows=ROWS - 1)
    assert right(seen, 4) and not asked
    run(ctx, blocks)
    assert right(seen, 8) and len(asked) == 3         # (the last product has no norm behind it that adds)


@pytest.mark.parametrize("which", ["mixer", "ffn"])
def test_what_a_part_adds_behind_its_product_is_in_the_next_norm(ctx, which):
    """A part that adds to the rows after its last product: sums commute with a product left unfinished, not with a norm taken already."""
    blocks = layers_of(2, after={which: 0.7})
    seen = watch(blocks)
    run(ctx, blocks)
    assert right(seen, 4)


def test_what_others_add_behind_a_part_is_in_the_next_norm(ctx):
    """A mixer around another one, an arrangement made of the pre-norm one, and a caller that looks at the rows between two layers."""
    from runtime.parts import GatedMLP, PreNormBlock
    ToyMixer, ToyFFN = toys()

    class Around(ToyMixer):
        def __init__(self, seed, after):
            super().__init__(seed, after)
            self.inner, self.kinds = ToyMixer(seed), []
            self.got = self.inner.got

        def forward(self, h, residual, ctx, *site, norm=None):
            return self.inner.forward(h, residual, ctx, *site).add_(0.7)

    class More(PreNormBlock):
        def forward(self, residual, ctx, site):
            return super().forward(residual, ctx, site).mul_(0.5)

    class Outer:
        def __init__(self, inner):
            self.inner, self.first_norm, self.first_reader = inner, inner.first_norm, inner.first_reader

        def forward(self, residual, ctx, site):
            return self.inner.forward(residual, ctx, site).mul_(0.5)
    for blocks, outer, tap in ((layers_of(2, mixer=Around), None, None), (layers_of(2, block=More), None, None), (layers_of(2), Outer, None),
                               (layers_of(2), None, lambda index, x: x.mul_(0.5))):
        seen = watch(blocks)
        run(ctx, [outer(b) if outer else b for b in blocks], tap)
        assert right(seen, 4)

    class Halved(GatedMLP):
        def forward(self, h, residual, ctx, norm=None):
            return super().forward(h, residual, ctx, norm=norm).mul_(0.5)
    named = []
    ctx.add_product = lambda a, w, residual, last=None, of=None: (named.append((last, of)), residual)[1]
    for cls in (GatedMLP, Halved):
        part = cls("m", WIDTH, WIDTH)
        part.w_gate_up, part.w_down = torch.cat([weights(1), weights(2)]), weights(3)
        part.forward(torch.zeros(ROWS, WIDTH).bfloat16(), torch.zeros(ROWS, WIDTH), ctx)
        block = PreNormBlock(rms(1), part, rms(2), ToyFFN(3))
        assert named.pop() == (part, GatedMLP)
        assert block.reads_next(part, GatedMLP, ctx) == ((block.ffn_norm, block.ffn) if cls is GatedMLP else None)


def test_a_norm_is_left_to_the_part_that_reads_it_in_this_step_only(ctx, monkeypatch):
    """One norm object before a part of this arrangement and of another, which knows of finished rows only; parts put in the place of
    those that a block was made with; a layer that runs twice."""
    from runtime.kernels import ops
    from runtime.parts import PreNormBlock, SandwichBlock
    from runtime.parts.base import Mixer
    ToyMixer, ToyFFN = toys()

    class Plain(Mixer):
        def __init__(self):
            self.kinds, self.got = [], []

        def output(self, h, ctx, site):
            return read(self, h).float()

        def forward(self, h, residual, ctx, site, norm=None):
            return residual.add_(read(self, h).float())

    def post_norm_add(residual, result, weight, eps, mult, following=None):
        residual.add_(mult * norm_of(SimpleNamespace(weight=weight, eps=eps), result))
        if following is not None:
            ops.rmsnorm(residual, following[0], following[2], following[1])
    monkeypatch.setattr(ops, "post_norm_add", post_norm_add)
    shared = rms(1)
    first, last = (PreNormBlock(norm, ToyMixer(10 + i), rms(20 + i), ToyFFN(30 + i)) for i, norm in enumerate((rms(2), shared)))
    other = SandwichBlock(shared, Plain(), rms(3))
    x = []
    seen = watch([first, last], stream=x)
    spied = other.mixer.output
    other.mixer.output = lambda h, c, site: (seen.append((other.mixer, norm_of(shared, x[0]))), spied(h, c, site))[1]
    run(ctx, [first, other, last])
    assert right(seen, 5) and other.mixer.kinds == ["Tensor"]

    blocks = layers_of(2)
    blocks[1].mixer = Plain()                          # (what it was made with could have finished the norm)
    seen = watch(blocks)
    run(ctx, blocks)
    assert right(seen, 4) and blocks[1].mixer.kinds == ["Tensor"]

    (block,) = layers_of(1)
    seen = watch([block])
    run(ctx, [block, block])
    assert right(seen, 4) and block.mixer.kinds == ["Tensor", "ScaledRows"]
