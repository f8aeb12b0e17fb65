"""What the compiled modules say of themselves without a GPU, and what is planned from it: where the matrix-core
attention kernels read a key's row, how items of wide heads are put together, which kernels the routed experts'
sizes choose, and which route products of some rows take."""

from __future__ import annotations

import ctypes
from types import SimpleNamespace

import pytest
import torch

from kvforge_amd.engine.batch import Step, Workspace
from kvforge_amd.kernels import library, ops
from kvforge_amd.parts import attention, block
from kvforge_amd.parts.base import Norm, add_product
from kvforge_amd.parts.norm import NamedRMSNorm, RMSNorm


@pytest.mark.parametrize("d", range(16, 257, 16))
@pytest.mark.parametrize("pages,KV,bs", [(1, 1, 8), (2, 3, 16)])
def test_every_fragment_of_a_key_lies_in_its_row(d, pages, KV, bs):
    """A key's row is d / 8 fragments of 16 bytes, and a step takes four of them, one a lane group.  A step that
    reaches past the row (d / 16 odd) reads inside it all the same: behind the last head's last slot of the last
    page the tensor ends."""
    fragment = ctypes.CDLL(library.build_module("attn_mfma")).kvf_attn_mfma_key_fragment
    steps, row = (d // 16 + 1) // 2, d // 8
    size = pages * KV * bs * row
    for page in range(pages):
        for head in range(KV):
            for slot in range(bs):
                base = ((page * KV + head) * bs + slot) * row
                read = [base + fragment(d, c, group) for c in range(steps) for group in range(4)]
                assert all(base <= at < base + row and at < size for at in read)
                assert read[:row] == list(range(base, base + row))


@pytest.mark.parametrize("experts,ff,k,few,more", [
    (4, 512, 1024, 64, 192), (8, 1024, 1024, 40, 64), (8, 3584, 2048, 12, 20), (8, 2048, 4096, 12, 16), (16, 512, 1024, 32, 48),
    (32, 1024, 2048, 5, 6), (64, 256, 1024, 6, 20), (512, 2048, 4096, 5, 6)])
def test_routed_experts_change_kernels_where_tiles_of_many_rows_pay(experts, ff, k, few, more):
    """``few`` and ``more`` rows an expert, either side of where the two take the same time: few or small experts, which
    leave most of the chip to tiles of many rows idle, change late.  Sizes whose products pass 32 bits too."""
    many = ctypes.CDLL(library.build_module("moe")).kvf_moe_grouped_many_rows
    assert [many(rows * experts, experts, ff, k) for rows in (2, few, more, 4096)] == [0, 0, 1, 1]


@pytest.mark.parametrize("pairs,own,library_s", [
    # what the library makes in whole rounds of large tiles, whatever K; many rows of large weights; either side of the most that is taken
    (0, [(2048, 1024, 512), (2048, 2048, 2048), (2048, 4096, 2048), (66, 28672, 4096), (333, 1024, 512), (777, 6144, 1024)],
     [(2048, 8192, 2048), (2048, 8192, 8192), (1013, 16384, 2048), (1013, 16384, 4096), (2048, 16384, 4096), (430, 28672, 2048), (512, 28672, 4096),
      (2048, 28672, 4096), (2048, 2048, 8192)]),
    (1, [(2048, 16384, 2048), (66, 16384, 2048), (2048, 4096, 2048), (100, 28672, 4096), (512, 1024, 512), (1300, 16384, 2048)],
     [(1771, 28672, 4096), (1013, 28672, 4096), (2048, 28672, 4096), (2048, 8192, 8192), (2048, 6144, 14336), (1300, 28672, 4096)])])
def test_products_of_many_rows_that_the_library_makes_as_fast_are_left_to_it(pairs, own, library_s):
    """Sizes that were timed both ways, faster in tiles and not."""
    takes = ctypes.CDLL(library.build_module("gemm_tile")).kvf_gemm_tile_takes
    assert [size for size in own if not takes(*size, pairs)] == [] and [size for size in library_s if takes(*size, pairs)] == []


@pytest.mark.parametrize("m,n,k,split", [(33, 128256, 2048, False), (64, 128256, 2048, False), (65, 128256, 2048, True), (64, 25016, 704, False),
                                         (95, 16384, 2048, False), (96, 16384, 2048, True), (767, 2048, 8192, False), (768, 2048, 8192, True),
                                         (768, 2048, 511, False), (768, 2048, 512, True), (33, 16, 64, False)])
def test_32_bit_products_on_split_operands_take_enough_rows(m, n, k, split):
    """Either side of every line of the rule: 64 rows, 6,144 outputs a compute unit (of 256), K of 512."""
    assert (ctypes.CDLL(library.build_module("gemm_generic")).kvf_gemm_generic_split_takes(m, n, k) >= 0) == split


@pytest.mark.parametrize("m,n,k,best", [(1434, 4096, 192, 1), (893, 6144, 128, 0), (1518, 3072, 64, 0), (1705, 6144, 512, 0), (1638, 5120, 256, 3),
                                        (2072, 1536, 64, 2), (343, 1536, 64, 5), (423, 5120, 128, 3)])
def test_tiles_of_the_fused_projection_where_k_is_short(m, n, k, best):
    """The tile that was timed the fastest of the six is taken."""
    assert ctypes.CDLL(library.build_module("gemm_tile")).kvf_gemm_tile_qkv_tile(m, n, k) == best


@pytest.mark.parametrize("q_lens,H,KV,pairs", [([33], 16, 1, False), ([256, 1], 16, 1, False), ([512], 32, 1, False),
                                               ([513], 32, 1, True), ([200, 200, 200], 32, 8, True), ([64], 8, 8, False)])
def test_items_of_wide_heads_go_in_pairs_where_they_are_more_than_the_compute_units(monkeypatch, q_lens, H, KV, pairs):
    monkeypatch.setattr(attention, "compute_units", lambda device: 256)
    seqs = [b for b, q in enumerate(q_lens) if q > 1]
    step = SimpleNamespace(prefill_seqs=seqs, scratch={}, device=None, q_lens=q_lens, start_pos=[0] * len(q_lens),
                           upload_ints=lambda ints: torch.tensor(ints, dtype=torch.int32))
    part = SimpleNamespace(H=H, KV=KV, d=224)
    work, per_item = attention.PagedAttention._prefill_work(part, step, torch.bfloat16, 16)
    assert per_item == 64 and bool((work[:, 2] >= 0).any()) == pairs
    items = sorted((b, i) for b, *both in work.tolist() for i in both if i >= 0)
    assert items == [(b, i) for b in seqs for i in range(-(-q_lens[b] * (H // KV) // 64))]


@pytest.mark.parametrize("dk", [1, 31, 32, 33, 96, 97, 128, 129, 192, 250, 256])
def test_the_scratch_of_channel_decays_holds_whole_heads(dk):
    """What the kernels write is as wide as what is given to them."""
    padded = ctypes.CDLL(library.build_module("chdelta")).kvf_chdelta_padded(dk)
    shapes = ops.chdelta_scratch(5, 2, 3, dk, 16)
    assert padded % 32 == 0 and padded - 32 < dk <= padded
    assert shapes["Kd"][0] == shapes["Qd"][0] == (5, 3, padded) and shapes["E"][0] == (2, 3, padded)
    assert shapes["Kw"][0] == (2, 3, padded, ops.ssm_chunk_len(dk))


@pytest.mark.parametrize("m,n,k,own", [
    (33, 16384, 2048, True), (56, 24576, 2048, True), (57, 24576, 2048, False), (64, 65536, 2048, True), (64, 128256, 2048, True),
    (33, 16368, 2048, False), (65, 128256, 2048, False), (33, 32768, 1024, False), (33, 24576, 2304, False),
    (48, 128256, 2112, False), (33, 16384, 4096, False), (64, 24576, 2056, True), (64, 128256, 4104, True)])
def test_products_that_stream_in_place_of_the_library(monkeypatch, m, n, k, own):
    """33 to 64 rows over tiled weights, either side of every line of the rule; over plain weights, and where the product
    is added to what is there, the library takes them all."""
    monkeypatch.setattr(ops, "compute_units", lambda device: 256)
    w = object.__new__(ops.StreamedWeight)
    w.shape, w.dtype, w.plain = (n, k), torch.bfloat16, SimpleNamespace(shape=(n, k), dtype=torch.bfloat16)
    a = torch.empty(m, k, dtype=torch.bfloat16)
    assert ops.streams_in_place_of_library(a, w) == own and ops.is_library_product(a, w) == (not own)
    assert ops.is_library_product(a, w.plain)
    routes = []
    monkeypatch.setattr(ops, "_gemm_operands", lambda a, w, out, n_out: (m, n, k, k, n))
    monkeypatch.setattr(ops, "_w_args", lambda w: (0, 1))
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops, "_fn", lambda module, name, types: lambda *args: routes.append(module) or 0)
    monkeypatch.setattr(ops, "_library_product", lambda *args: routes.append("library"))
    out = SimpleNamespace(dtype=torch.float32, data_ptr=lambda: 0)
    ops.gemm(a, w, out)
    ops.gemm(a, w, out, accumulate=True)
    assert routes == ["gemm_bf16" if own else "library", "library"]


@pytest.mark.parametrize("rows,n,k,settled,route", [
    (17, 2048, 2048, True, "added"), (23, 3072, 3072, True, "added"), (24, 3072, 3072, True, "parts"),
    (17, 2048, 2048, False, "parts"), (17, 2048, 4096, True, "parts"), (33, 2048, 2048, True, "parts"),
    (16, 2048, 2048, False, "added"), (65, 2048, 2048, False, "owed")])
def test_products_go_in_parts_where_what_reads_them_next_pays_for_it(monkeypatch, rows, n, k, settled, route):
    """Parts that the next reader cannot take cost an add kernel: few rows are then added by the product's own kernel."""
    took = []
    monkeypatch.setattr(ops, "parts_count", lambda a, w: 4 if 16 < a.shape[0] <= 64 else 0)
    monkeypatch.setattr(ops, "gemm_parts", lambda a, w, parts: took.append("parts"))
    monkeypatch.setattr(ops, "k_halves_pay", lambda a, w: False)
    monkeypatch.setattr(ops, "gemm", lambda a, w, out, accumulate=False, owed=None: took.append("added" if accumulate else "owed"))
    step = Step()
    step.ws, step.settled_next = Workspace("cpu"), settled
    monkeypatch.setattr(step, "owe", lambda stream, product: None)
    add_product(step, torch.empty(rows, k, dtype=torch.bfloat16), torch.empty(n, k, dtype=torch.bfloat16), torch.empty(rows, n))
    assert took == [route]


@pytest.mark.parametrize("feed_forward,pair,after,wanted", [
    (True, True, False, [True, True]), (True, False, False, [True, False]), (True, False, True, [True, True]),
    (False, False, False, [False]), (False, False, True, [True])])
def test_a_parallel_block_says_who_settles_what_its_sublayers_owe(monkeypatch, feed_forward, pair, after, wanted):
    said = []
    sub = SimpleNamespace(settles_residual=False, state_spec=None, forward=lambda *args: said.append(args[1].settled_next))
    ffn = SimpleNamespace(settles_residual=False, forward=lambda x, step, residual: said.append(step.settled_next))
    norm = SimpleNamespace(adds_bias=False, takes_parts=True, forward=lambda *args, **kw: None)
    then = SimpleNamespace(forward=lambda residual, step, bias=None: said.append(("after", step.settled_next)))
    part = block.ParallelBlock(norm, sub, ffn if feed_forward else None, 8, after=then if after else None,
                               ffn_norm=norm if pair else None)
    monkeypatch.setattr(part, "_norms_pair", lambda: pair)
    monkeypatch.setattr(ops, "rmsnorm_pair", lambda *args, **kw: None)
    part.norm = part.ffn_norm = SimpleNamespace(weight=None, eps=0.0, adds_bias=False, takes_parts=True, forward=norm.forward)
    if not pair:
        part.ffn_norm = None
    step = Step()
    step.ws = Workspace("cpu")
    part.forward(torch.zeros(3, 8), step, None)
    assert said == wanted + ([("after", False)] if after else []) and not step.settled_next


@pytest.mark.parametrize("n", [1, 16, 4096])
@pytest.mark.parametrize("m", [17, 64])
def test_no_product_goes_in_parts_below_the_least_k(m, n):
    """What the host leaves unasked is what the kernel's rule refuses."""
    count = ctypes.CDLL(library.build_module("gemm_bf16")).kvf_gemm_bf16_parts_count
    assert not any(count(m, n, k) for k in range(8, ops.PARTS_MIN_K, 8))


@pytest.mark.parametrize("n,KV,window,chunk,in_order", [
    (41, 8, None, None, True), (32, 8, None, None, False), (33, 8, None, None, True), (41, 8, 512, None, False),
    (41, 8, None, 512, False), (257, 1, None, None, True), (256, 1, None, None, False)])
def test_layers_alike_share_the_plan_of_single_tokens(monkeypatch, n, KV, window, chunk, in_order):
    """The step's order is taken where the workgroups outnumber the compute units and every layer sees whole contexts; it is
    worked out once a step for layers alike, and again for ones that are not and for a step filled anew."""
    monkeypatch.setattr(attention, "compute_units", lambda device: 256)
    asked = []

    def layer(**other):
        part = object.__new__(attention.PagedAttention)
        part.__dict__.update(dict(H=32, KV=KV, window=window, chunk=chunk, keep_first=0), **other)
        part._decode_cuts = lambda step, on_matrix_cores: asked.append(part) or 1
        return part

    step = Step()
    step.device, step.n_decode = None, n
    parts = [layer(), layer(), layer(window=64), layer(H=64)]
    plans = [p._decode_plan(step, True) for p in parts * 2]
    assert plans == [(1, in_order), (1, in_order), (1, False), (1, in_order)] * 2
    assert asked == [parts[0], parts[2], parts[3]]
    assert parts[1]._decode_plan(step, False) == (1, in_order) and asked[3:] == [parts[1]]
    step.scratch = {}
    parts[1]._decode_plan(step, True)
    assert asked[4:] == [parts[1]]


@pytest.mark.parametrize("config", ["llama", "rudorax", "depolix"])
def test_a_model_that_the_last_level_cache_holds_is_read_through_it(monkeypatch, config):
    """Every matrix in tiles that the parts of a model hold is found, and all are marked, or none, by what they are worth together."""
    import kvforge_amd
    from kvforge_amd.config import presets
    from kvforge_amd.models.transformer import Transformer
    cfg = {"llama": lambda: kvforge_amd.preset_dict("tiny-b"),
           "rudorax": lambda: presets.rudorax_stack(vocab=300, width=64, pairs=1, heads=4, kv_heads=2, dim=16, window=24, lstm_heads=2,
                                                    lstm_dim=32, lstm_vdim=32, ff=32, experts=4, top=2, identity=1, shared_ff=32,
                                                    max_positions=512),
           "depolix": lambda: presets.depolix_stack(vocab=300, width=64, groups=1, heads=4, latent_dim=16, rot_dim=16, q_rank=32,
                                                    kv_rank=32, att_heads=4, att_kv_heads=2, att_dim=16, window=24, mem_heads=4,
                                                    mem_kv_heads=2, mem_dim=16, mem_vdim=16, gate_rank=16, ff=64, moe_ff=32,
                                                    experts=4, top=2, max_positions=512)}[config]()
    made = []

    def streamed(w):
        if w is None or w.dtype != torch.bfloat16 or w.dim() != 2:
            return w
        made.append(ops.StreamedWeight(w.contiguous()))
        return made[-1]
    monkeypatch.setattr(ops, "streamed", streamed)
    model = Transformer.from_random(cfg, 3, torch.bfloat16, "cpu")
    held = {t.data_ptr() for p in model.spec.all_parts() for t in p.held_tensors()}
    assert made and {w.tiles.data_ptr() for w in made} <= held and {w.cached for w in made} == {True}
    total = sum(w.tiles.nbytes for w in made)
    for limit, cached in ((total - 1, False), (total, True)):
        monkeypatch.setattr(ops, "LAST_LEVEL_BYTES", limit)
        del made[:]
        model = Transformer.from_random(cfg, 3, torch.bfloat16, "cpu")
        assert sum(w.tiles.nbytes for w in made) == total and {w.cached for w in made} == {cached}


class Centred(Norm):
    """No RMS norm, though it has a weight vector and an eps."""

    def __init__(self, weight):
        self.weight, self.eps = weight, 1e-5

    def forward(self, x, out, rows=None, add=None):
        out.copy_(torch.nn.functional.layer_norm(x, x.shape[1:], self.weight, None, self.eps))


class Doubled(RMSNorm):
    def forward(self, x, out, rows=None, add=None, bias=None):
        out.copy_(2.0 * x)


def test_two_norms_of_one_stream_are_one_kernel_only_if_they_are_rms_norms():
    """Norms of other kinds, two of one kind among them, are each asked for their rows."""
    g = torch.Generator().manual_seed(1)
    x, weights = torch.randn(17, 8, generator=g), [torch.randn(8, generator=g) for _ in range(2)]
    got = []
    sub = SimpleNamespace(settles_residual=False, state_spec=None, forward=lambda rows, *args: got.append(rows.clone()))
    ffn = SimpleNamespace(settles_residual=False, forward=lambda rows, *args: got.append(rows.clone()))
    step = Step()
    step.ws, step.act_dtype = Workspace("cpu"), torch.float32
    block.ParallelBlock(Centred(weights[0]), sub, ffn, 8, ffn_norm=Centred(weights[1])).forward(x, step, None)
    for rows, w in zip(got, weights):
        assert torch.equal(rows, torch.nn.functional.layer_norm(x, (8,), w, None, 1e-5))

    def rms(cls, eps=1e-5, dtype=torch.float32):
        norm = cls("n", 8, eps)
        norm.weight = torch.ones(8, dtype=dtype)
        return norm

    def together(a, b):
        return block.ParallelBlock(a, sub, ffn, 8, ffn_norm=b)._norms_pair()
    assert together(rms(RMSNorm), rms(NamedRMSNorm))
    for other in (rms(RMSNorm, 1e-6), rms(RMSNorm, dtype=torch.bfloat16), rms(Doubled), Centred(weights[0]), None):
        assert not together(rms(RMSNorm), other)
    assert not together(rms(Doubled), rms(Doubled))
