"""Products that parts have made together, ahead of them or behind: mixers side by side give what they give one by one, also where
both keep their rows in the same workspace buffers."""

from __future__ import annotations

import ctypes
import random

import pytest
import torch

import kvforge_amd
from kvforge_amd.config.model import ModelConfig
from kvforge_amd.engine.batch import Step, StepEntry, Workspace
from kvforge_amd.engine.runner import ModelRunner
from kvforge_amd.kernels import library, ops
from kvforge_amd.models.transformer import Transformer
from kvforge_amd.parts import (ChannelDelta, FeedForward, GatedDelta, LMHead, Mamba2, Mixer, MixerPair, ModelSpec, NamedRMSNorm, Norm,
                               ParallelBlock, PlainFeedForward, RMSNorm, TokenEmbedding)
from kvforge_amd.parts.base import LayerState, add_product


# ------------------------------------------------------------------------------------- on the CPU, products by torch
class Toy(Mixer):
    """``residual += (x @ w.T)^2 @ w_o.T + sin(x @ w_g.T)`` over rows in buffers of the names ``name`` (``lists``: the first products
    are announced)."""

    def __init__(self, key: str, name: str, buffers: str | None, width: int, lists: bool = True) -> None:
        g = torch.Generator().manual_seed(width + ord(key))
        self.prefix, self.name, self.buffers, self.lists = key, name, buffers, lists
        self.w, self.w_g, self.w_o = (torch.randn(*s, generator=g) for s in ((width, 24), (24, 24), (24, width)))

    def plainly(self, x):
        return (x @ self.w.T) ** 2 @ self.w_o.T + torch.sin(x @ self.w_g.T)

    def _products(self, x, step):
        return [((self.prefix, k), x, w, step.ws.buf(self.name + k, (x.shape[0], w.shape[0]), torch.float32), "store")
                for k, w in (("rows", self.w), ("gates", self.w_g))]

    def input_products(self, x, step):
        return self._products(x, step) if self.lists else []

    def forward(self, x, step, layer, residual):
        step.settle()
        products = self._products(x, step)
        if self.lists:
            step.make(products)
        else:
            for _, a, w, out, _how in products:
                ops.gemm(a, w, out)
        rows, gates = (p[3] for p in products)
        residual += torch.sin(gates)
        add_product(step, rows ** 2, self.w_o, residual)


@pytest.fixture
def by_torch(monkeypatch):
    """Products as torch makes them, and how many went into each launch of several."""
    sizes = []

    def gemm(a, w, out, accumulate=False, **_):
        out.copy_(out + a @ w.T if accumulate else a @ w.T)

    def group(products):
        sizes.append(len(products))
        for a, w, out, how in reversed(products):     # (in any order: they run at the same time)
            gemm(a, w, out, how == "add")
    for name, f in (("gemm", gemm), ("gemm_group", group), ("gemm_group_takes", lambda a, w, out: a.shape[0] <= 16),
                    ("is_library_product", lambda a, w: False), ("k_halves_pay", lambda a, w: False)):
        monkeypatch.setattr(ops, name, f)
    monkeypatch.setattr(ops, "parts_count", lambda a, w: 0)
    return sizes


def _step():
    step = Step()
    step.ws, step.act_dtype = Workspace("cpu"), torch.float32
    return step


@pytest.mark.parametrize("early", [False, True])     # whether a block has asked for the products before the pair does
@pytest.mark.parametrize("left,right,launches", [
    (("a", "", "toy", 40), ("b", "", "toy", 40), [2, 2]),             # one make: the same memory
    (("a", "", "toy", 24), ("b", "", "toy", 56), [2, 2]),             # ... and the wider one makes it move
    (("a", "", "toy", 56), ("b", "", "toy", 24), [2, 2]),
    (("a", "", "toy", 40, False), ("b", "", "toy", 40), [2]),         # the first says nothing of its products
    (("a", "", None, 40), ("b", "", None, 40), [2, 2]),               # makes that do not say what they use
    (("a", "", "one", 40), ("b", "", "two", 40), [2, 2]),             # makes that say so wrongly
    (("a", "", "one", 24), ("b", "", "two", 56), [3, 2]),
    (("a", "left_", "one", 40), ("b", "right_", "two", 56), [4])])
def test_mixers_side_by_side_as_one_by_one(by_torch, left, right, launches, early):
    for rows in (1, 7, 16, 17):
        by_torch.clear()
        x = torch.randn(rows, 24, generator=torch.Generator().manual_seed(rows))
        pair, got, step = MixerPair(Toy(*left), Toy(*right)), torch.zeros(rows, 24), _step()
        want = pair.left.plainly(x) + pair.right.plainly(x)
        if early and rows <= 16:
            step.make_early(pair.input_products(x, step))
        pair.forward(x, step, LayerState(), got)
        step.settle()
        torch.testing.assert_close(got, want, rtol=1e-5, atol=1e-3)
        assert not step.made and by_torch == (launches if rows <= 16 else [])


class ToyNorm(Norm):
    def __init__(self) -> None:
        self.prefix = "n"

    def forward(self, x, out, rows=None, add=None):
        if add is not None:
            x += add
        out.copy_(x)


class ToyFeedForward(FeedForward):
    """``sin(x @ w.T) @ w_o.T`` for the stream, and the rows ``x @ w_r.T`` for ``seen``, which may ride with a product of the mixer's;
    ``uses``: whether it looks for the products that it has announced."""

    settles_residual = True

    def __init__(self, uses: bool = True) -> None:
        g = torch.Generator().manual_seed(5)
        self.prefix, self.uses, self.seen = "f", uses, []
        self.w, self.w_o, self.w_r = (torch.randn(*s, generator=g) for s in ((32, 24), (24, 32), (16, 24)))

    def input_products(self, x, step):
        return [(("f", "first"), x, self.w, step.ws.buf("f_first", (x.shape[0], 32), torch.float32), "store")]

    def ready_products(self, x, step):
        return [(("f", "ready"), x, self.w_r, step.ws.buf("f_ready", (x.shape[0], 16), torch.float32), "store")]

    def forward(self, x, step, residual):
        step.settle()
        if self.uses:
            step.make(self.input_products(x, step))
            step.make(self.ready_products(x, step))
            self.seen.append(step.ws.buf("f_ready", (x.shape[0], 16), torch.float32).clone())
        add_product(step, torch.sin(x @ self.w.T), self.w_o, residual)


def test_products_ride_with_the_mixers_last_one_and_none_may_be_left_over(by_torch):
    for rows in (1, 16, 17):
        by_torch.clear()
        x, step, ffn = torch.randn(rows, 24, generator=torch.Generator().manual_seed(rows)), _step(), ToyFeedForward()
        mixer = Toy("a", "", "toy", 40)
        got = x.clone()
        ParallelBlock(ToyNorm(), mixer, ffn, 24).forward(got, step, LayerState())
        step.settle()
        torch.testing.assert_close(got, x + mixer.plainly(x) + torch.sin(x @ ffn.w.T) @ ffn.w_o.T, rtol=1e-5, atol=1e-3)
        torch.testing.assert_close(ffn.seen[0], x @ ffn.w_r.T, rtol=1e-5, atol=1e-4)
        assert by_torch == ([3, 2] if rows <= 16 else []) and not step.riders     # first products; last one and rider
    with pytest.raises(RuntimeError, match="not used.*first"):
        ParallelBlock(ToyNorm(), Toy("a", "", "toy", 40), ToyFeedForward(uses=False), 24).forward(
            torch.randn(4, 24), _step(), LayerState())


STORE_F32, STORE_BF16, ADD, PAIRS = range(4)      # what becomes of a product


@pytest.mark.parametrize("rows", [1, 3, 16])
def test_products_of_one_launch_lie_apart(rows):
    """Results of a launch against memory written out: a product is refused where it writes what another writes or reads."""
    apart = ctypes.CDLL(library.build_module("gemm_bf16")).kvf_gemm_bf16_group_apart
    rng = random.Random(rows)
    seen = set()
    for _ in range(3000):
        items, writes, reads = [], [], []
        for _ in range(rng.randint(1, 4)):
            n, k, epi = rng.choice([4, 8, 16]), rng.choice([8, 16]), rng.choice([STORE_F32, STORE_BF16, ADD, PAIRS])
            size, cols = 4 if epi in (STORE_F32, ADD) else 2, n // 2 if epi == PAIRS else n
            ldc, lda = (cols if rows == 1 else rng.choice([cols, 16, 24])), (k if rows == 1 else rng.choice([k, 24]))
            ldc = max(ldc, cols)
            a, c = 4096 + 16 * rng.randint(0, 100), 4096 + 4 * rng.randint(0, 400) + rng.choice([0, 1 << 16])
            items += [a, 64, c, n, k, lda, ldc, epi]
            reads.append({a + 2 * (r * lda + i) + b for r in range(rows) for i in range(k) for b in range(2)})
            writes.append({c + size * (r * ldc + i) + b for r in range(rows) for i in range(cols) for b in range(size)})
        clash = any(x & y for i, x in enumerate(writes) for y in writes[:i]) or any(x & y for x in writes for y in reads)
        said = apart((ctypes.c_longlong * len(items))(*items), len(items) // 8, rows)
        assert not (said and clash), items
        seen.add((bool(said), clash))
    assert seen >= {(True, False), (False, True)}
    column = lambda at, first: [4096, 64, at + 4 * first, 16, 64, 64, 48, STORE_F32]  # noqa: E731
    if rows > 1:
        for firsts, want in (((0, 16, 32), 1), ((32, 0, 16), 1), ((0, 8), 0), ((0, 40), 0), ((0, 0), 0), ((0, 48), 0)):
            items = sum((column(1 << 20, f) for f in firsts), [])
            assert apart((ctypes.c_longlong * len(items))(*items), len(firsts), rows) == want, firsts


@pytest.mark.gpu
def test_a_launch_of_several_products_refuses_memory_that_two_of_them_use():
    a, wide = torch.ones(3, 512, dtype=torch.bfloat16, device="cuda"), torch.zeros(3, 48, device="cuda")
    w = ops.StreamedWeight(torch.ones(16, 256, dtype=torch.bfloat16, device="cuda"))
    for products in ([(a[:, :256], w, wide[:, :16], "store"), (a[:, :256], w, wide[:, 8:24], "add")],
                     [(a[:, :256], w, a[:, 400:416], "store"), (a[:, :256], w, wide[:, :16], "store")]):
        with pytest.raises(ops.KernelError, match="what another one writes"):
            ops.gemm_group(products)
    assert bool((wide == 0).all()) and bool((a == 1).all())
    ops.gemm_group([(a[:, :256], w, wide[:, f:f + 16], "store") for f in (0, 32, 16)])
    assert bool((wide == 256).all())


# ------------------------------------------------------------------------------------- on the GPU, whole models
class OneByOne(MixerPair):
    """The two mixers one after the other, each with launches of its own."""

    def input_products(self, x, step):
        return []

    def forward(self, x, step, layer, residual):
        outs = []
        for m, state, name in zip((self.left, self.right), self._layers(layer), ("one_left", "one_right")):
            if self.norms is None:
                m.forward(x, step, state, residual)
                continue
            step.settle()
            step.fresh = step.ws.buf(name, tuple(residual.shape), torch.float32)
            outs.append(step.fresh)
            m.forward(x, step, state, step.fresh)
        if self.norms is not None:
            ops.rms_add_two(residual, outs[0], self.weights[0], outs[1], self.weights[1], self.norms[0].eps)


class PairConfig(ModelConfig):
    def __init__(self, d):
        super().__init__(architecture="ToyPairForCausalLM", vocab_size=96, max_position_embeddings=256)
        self.d = d

    @classmethod
    def from_dict(cls, d):
        return cls(d)

    def to_dict(self):
        return self.d


def _memory(kind, name, h):
    cls, heads, dim = kind
    more = dict(norm_parts=2) if cls is Mamba2 else dict(a_rank=16, g_rank=32) if cls is ChannelDelta else {}
    return cls(name, h, heads, 2, dim, 32, 4, norm_eps=1e-5, **more)


def _build(cfg):
    d, h = cfg.d, 256
    pair_cls = OneByOne if d["one_by_one"] else MixerPair
    blocks = []
    for i in range(2):
        norms = tuple(NamedRMSNorm(f"l.{i}.out_{s}", h, 1e-5) for s in "lr") if d["normed"] else None
        pair = pair_cls(*(_memory(k, f"l.{i}.{s}", h) for k, s in zip(d["kinds"], "lr")), norms=norms)
        blocks.append(ParallelBlock(RMSNorm(f"l.{i}.n", h, 1e-5), pair, PlainFeedForward(f"l.{i}.ff", h, 256), h))
    return ModelSpec(config=cfg, embedding=TokenEmbedding("embed", 96, h), blocks=blocks, final_norm=RMSNorm("norm", h, 1e-5),
                     head=LMHead("head", 96, h), positions=[])


@pytest.mark.gpu
@pytest.mark.parametrize("normed", [False, True])
@pytest.mark.parametrize("kinds", [((Mamba2, 8, 16), (GatedDelta, 8, 16)), ((GatedDelta, 4, 16), (Mamba2, 8, 32)),
                                   ((ChannelDelta, 4, 32), (ChannelDelta, 4, 32))])
def test_memories_of_one_make_side_by_side_as_one_by_one(kinds, normed):
    """Prompts of 1, 8 and 16 tokens and steps of 1, 8 and 16 requests behind longer ones: the same bits as from two mixers with
    launches of their own."""
    kvforge_amd.register_architecture("ToyPairForCausalLM", PairConfig, _build)
    logits = []
    for one_by_one in (True, False):
        cfg = PairConfig({"kinds": kinds, "normed": normed, "one_by_one": one_by_one})
        model = Transformer.from_random(cfg, 3, torch.bfloat16, "cuda")
        runner = ModelRunner(model, 16, 64, max_num_seqs=16, max_num_batched_tokens=256, max_model_len=64)
        g, out = torch.Generator().manual_seed(1), []
        ids = lambda n: torch.randint(0, 96, (n,), generator=g).tolist()  # noqa: E731
        for n in (1, 8, 16):
            runner.cache.allocate(f"p{n}", n)
            out.append(runner.step([StepEntry(f"p{n}", ids(n), 0, "all")]).clone())
            runner.cache.free(f"p{n}")
        for r in range(16):
            runner.cache.allocate(f"r{r}", 20)
        out.append(runner.step([StepEntry(f"r{r}", ids(9 + r % 3), 0) for r in range(16)]).clone())
        at = [9 + r % 3 for r in range(16)]
        for rows in (16, 8, 1, 8):
            out.append(runner.step([StepEntry(f"r{r}", ids(1), at[r]) for r in range(rows)]).clone())
            at = [p + (r < rows) for r, p in enumerate(at)]
        logits.append(torch.cat(out).cpu())
    assert bool(logits[0].isfinite().all()) and float(logits[0].std()) > 0
    assert torch.equal(*logits)
