"""A norm that two ring products make between them, through whole models: steps of so many rows that a block leaves the next part's norm to
its own last product and to that part's first."""
import numpy as np
import pytest
import torch

import plain_llama as P
from conftest import assert_close

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
EPS, THETA, VOCAB = 1e-5, 10000.0, 96


def model_of(width, heads, kv, ff, layers, order=None):
    """A bf16 model of the framework's own attention and feed-forward in the pre-norm arrangement, with the plain weights.  layers: for
    each the options of its parts (out_bias, bias of the feed-forward, own_kv); order: (layer, entry that it reads)."""
    from runtime import make_part
    from runtime.models import Model, ScheduleEntry
    from runtime.parts import LMHead, TokenEmbedding

    def rms(name): return make_part("norm", "rmsnorm", name=name, dim=width, eps=EPS)
    position = make_part("position", "rotary", head_dim=64, theta=THETA, max_positions=1280)
    blocks = [make_part("block", "prenorm", mixer_norm=rms(f"l{i}.n1"), ffn_norm=rms(f"l{i}.n2"),
                        mixer=make_part("mixer", "attention", name=f"l{i}.attn", hidden=width, heads=heads, kv_heads=kv, head_dim=64, position=position,
                                        out_bias=o.get("out_bias", False), own_kv=o.get("own_kv", True)),
                        ffn=make_part("ffn", "gated_mlp", name=f"l{i}.mlp", hidden=width, intermediate=ff, bias=o.get("bias", False)))
              for i, o in enumerate(layers)]
    order = order or [(i, None) for i in range(len(layers))]
    model = Model(None, TokenEmbedding("embed", VOCAB, width), blocks, rms("final"), LMHead("head", VOCAB, width),
                  schedule=[ScheduleEntry(*entry) for entry in order], max_positions=1280, vocab_size=VOCAB)
    g = torch.Generator().manual_seed(width)
    w = {}
    for spec in model.tensor_specs():
        draw = torch.randn(spec.shape, generator=g)
        # (projections keep their input's scale, sublayers add as much as is there, and so does a bias)
        w[spec.name] = (1.0 + 0.2 * draw if len(spec.shape) == 1 and not spec.name.endswith("bias") else draw if spec.name.endswith(("bias", "embed.weight"))
                        else draw * spec.shape[-1] ** -0.5).bfloat16()
    model.bind({name: t.to(DEV) for name, t in w.items()}, torch.bfloat16, torch.device(DEV))
    return model, {name: t.double().numpy() for name, t in w.items()}, order


def plain(w, heads, kv, order, tokens):
    x, T, kept = w["embed.weight"][tokens], len(tokens), []
    pos = np.arange(T)

    def lin(h, name):
        return P.linear(h, w[name + ".weight"]) + w.get(name + ".bias", 0.0)
    for layer, reads in order:
        n = f"l{layer}"
        h = P.rmsnorm(x, w[n + ".n1.weight"], EPS)
        q = P.rope(lin(h, n + ".attn.q_proj").reshape(T, heads, 64), pos, THETA)
        if reads is None:
            kept.append((P.rope(lin(h, n + ".attn.k_proj").reshape(T, kv, 64), pos, THETA), lin(h, n + ".attn.v_proj").reshape(T, kv, 64)))
        else:
            kept.append(kept[reads])
        x = x + lin(P.causal_attention(q, *kept[-1]).reshape(T, heads * 64), n + ".attn.o_proj")
        h = P.rmsnorm(x, w[n + ".n2.weight"], EPS)
        x = x + lin(P.swiglu(lin(h, n + ".mlp.gate_proj"), lin(h, n + ".mlp.up_proj")), n + ".mlp.down_proj")
    return P.linear(P.rmsnorm(x, w["final.weight"], EPS), w["head.weight"])


def logits_of(model, tokens, execution, steps=1):
    """The logits of `tokens` as one portion, of `steps` requests one after the other (under "graph" the later ones are replays)."""
    from runtime.engine import ModelRunner, StepEntry
    runner = ModelRunner(model, n_pages=-(-len(tokens) // 16) + 1, page_size=16, max_requests=1, execution=execution)
    made = []
    for i in range(steps):
        runner.create(i)
        made.append(runner.step([StepEntry(i, list(tokens), list(range(len(tokens))))]).float().cpu().numpy())
        runner.release(i)
    return made


@pytest.fixture
def handed(monkeypatch):
    """How many norms have been left to products so far."""
    from runtime.kernels import ops
    seen, real = [], ops.gemm_ring_normed
    monkeypatch.setattr(ops, "gemm_ring_normed", lambda a, w, *rest, **at: (seen.append(tuple(a.shape)), real(a, w, *rest, **at))[1])
    return seen


SIZES = [(576, 9, 3, 1536, 1000), (1024, 16, 4, 2048, 600)]      # width, heads, key/value heads, feed-forward, rows


@pytest.mark.parametrize("width, heads, kv, ff, rows", SIZES)
def test_a_bias_behind_the_product_is_in_the_norm_after_it(width, heads, kv, ff, rows, handed):
    """Attention with a bias on its output before a feed-forward without, and a feed-forward with biases before attention without: what they add
    behind their last product belongs to the rows that the next norm reads."""
    model, w, order = model_of(width, heads, kv, ff, [{"out_bias": True}, {"bias": True}, {}])
    tokens = np.random.default_rng(rows).integers(0, VOCAB, rows)
    want = plain(w, heads, kv, order, tokens)
    for name in ("l0.attn.o_proj.bias", "l1.mlp.down_proj.bias"):
        assert np.linalg.norm(plain({**w, name: 0.0 * w[name]}, heads, kv, order, tokens) - want) > 0.1 * np.linalg.norm(want), name
    for execution in ("eager", "graph"):
        assert_close(logits_of(model, tokens, execution)[0], want, "bfloat16", execution)
    # left to products: the norms behind the first feed-forward and the last attention
    assert len(handed) >= 2 and len(handed) % 2 == 0


@pytest.mark.parametrize("width, heads, kv, ff, rows", SIZES)
def test_norms_that_products_make_through_a_model(width, heads, kv, ff, rows, handed, monkeypatch):
    """A layer that runs twice and one that reads another's keys: every norm behind a product but the last is left to products, step by step
    and in a captured program, whose replays repeat themselves bit for bit; the logits are as far from 64 bits as with all norms kernels of their own."""
    from runtime.kernels import ops
    layers, order = [{}, {"own_kv": False}, {}], [(0, None), (1, 0), (0, None), (2, None)]
    model, w, order = model_of(width, heads, kv, ff, layers, order)
    tokens = np.random.default_rng(rows).integers(0, VOCAB, rows)
    want = plain(w, heads, kv, order, tokens)
    (eager,) = logits_of(model, tokens, "eager")
    assert len(handed) == 2 * len(order) - 1 and {k for _, k in handed} == {heads * 64, ff}
    made = logits_of(model, tokens, "graph", steps=3)        # (its rows and keys come in rounded numbers: other tiles than step by step)
    assert np.array_equal(made[1], made[0]) and np.array_equal(made[2], made[0])
    assert_close(made[0], want, "bfloat16")
    assert len(handed) % (2 * len(order) - 1) == 0
    monkeypatch.setattr(ops, "ring_normed_parts", lambda *a, **at: 0)
    count = len(handed)
    (apart,) = logits_of(model, tokens, "eager")
    assert len(handed) == count
    assert_close(eager, want, "bfloat16")
    # (both round the rows to bf16 once; which of them is nearer is chance, 5 in 100 over this many)
    off = [np.linalg.norm(got - want) for got in (eager, apart)]
    assert off[0] < 1.05 * off[1]
