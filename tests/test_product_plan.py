"""The host-side plan of a matrix product (how many float32 shares of k): no
device is needed for it.  A decode step captured as a graph of 128 or 256 rows
stands for any number of sequences up to that; graph and kernel-by-kernel
execution agree bit for bit only if the plan is the same for all of them."""

import pytest

from shrike_amd.kernels import ops

MATRICES = [(4608, 3584), (3584, 3584), (3584, 18944), (5120, 13824), (7168, 5120), (5120, 5120),
            (152064, 3584), (503, 128), (2100, 16400)]


@pytest.mark.parametrize("m, k", MATRICES)
def test_the_plan_is_the_same_for_every_row_count_of_a_graph_bucket(m, k):
    for lo, hi in ((1, 16), (17, 32), (33, 64), (65, 128), (129, 256)):
        plans = {ops.gemm_splits(n, m, k) for n in range(lo, hi + 1)}
        assert len(plans) == 1, f"rows {lo}..{hi} of [{m}, {k}]: {sorted(plans)}"


@pytest.mark.parametrize("m, k", MATRICES)
def test_shares_keep_enough_of_k(m, k):
    """Every share has at least 16 tiles of 32 of k, and there are at most 16 shares."""
    for n in (1, 8, 16, 24, 64, 100, 256, 512, 2048, 4096):
        s = ops.gemm_splits(n, m, k)
        assert 1 <= s <= 16
        assert s == 1 or -(-k // 32) // s >= 16


SMALL = [(896, 896), (1152, 896), (896, 4864), (1000, 2056), (512, 3584), (2048, 2048), (1536, 1536), (256, 40), (10, 3584), (64, 520),
         (1, 64), (300, 8192)]


@pytest.mark.parametrize("m, k", SMALL)
def test_small_matrices_are_planned_alike_for_every_row_count_of_a_graph_bucket(m, k):
    for lo, hi in ((1, 16), (17, 32), (33, 64), (65, 128), (129, 256)):
        assert len({(ops.gemm_splits(n, m, k), ops.gemm_keeps_float32(n, m, k), ops.gemm_parts(n, m, k))
                    for n in range(lo, hi + 1)}) == 1, f"rows {lo}..{hi}"


def test_small_matrices_formed_whole_reach_their_reader_in_float32():
    """What the staged kernels would leave as float32 shares is not rounded to bfloat16 for being formed whole."""
    for m, k, ns in ((896, 896, (17, 64)), (1152, 896, (17, 64)), (896, 4864, (65, 256)), (512, 3584, (65, 300))):
        for n in ns:
            assert ops.gemm_splits(n, m, k) == 1 and ops.gemm_keeps_float32(n, m, k), (m, k, n)
    assert ops.gemm_splits(64, 896, 4864) > 1 and not ops.gemm_keeps_float32(64, 896, 4864)  # shares are float32 anyway
    # never split, never kept: one token, large matrices, a short k
    for m, k, n in ((896, 896, 1), (152064, 3584, 8), (18944, 3584, 4096), (896, 128, 64)):
        assert ops.gemm_splits(n, m, k) == 1 and not ops.gemm_keeps_float32(n, m, k), (m, k, n)


def test_a_long_k_is_shared_where_one_walk_along_it_takes_longer():
    for n in (17, 64):
        assert ops.gemm_splits(n, 512, 1024) == 1 and ops.gemm_splits(n, 512, 2048) == 2 and ops.gemm_splits(n, 512, 3584) == 4
        assert ops.gemm_splits(n, 256, 8192) == 8 and ops.gemm_splits(n, 896, 4864) >= 2
    # few rows: whole, but not a long k in a handful of workgroups or in more than the compute units take at once
    assert ops.gemm_splits(1501, 10, 3584) == 1 and ops.gemm_splits(256, 32, 8192) == 1
    assert ops.gemm_splits(65, 16, 8192) > 1 and ops.gemm_splits(1501, 64, 8192) > 1 and ops.gemm_splits(4096, 64, 3584) > 1
    # small matrices: not where the staged kernels' larger tiles fill the chip
    assert ops.gemm_splits(1119, 1024, 2048) == 2 and ops.gemm_splits(640, 256, 14336) > 8
    # rows that are no whole 16-byte pieces keep the shares of the kernels that take them
    assert ops.gemm_splits(64, 896, 4860) == ops.gemm_splits(64, 896, 4861) > 1


def test_matrices_that_fill_the_chip_are_not_split():
    assert ops.gemm_splits(8, 152064, 3584) == 1      # 9504 row blocks
    assert ops.gemm_splits(4096, 18944, 3584) == 1    # 592 tiles of 256 x 256
    assert ops.gemm_splits(8, 3584, 18944) > 1        # 224 row blocks, a long k
    assert ops.gemm_splits(512, 5120, 13824) > 1      # 80 tiles of 256 x 128


def test_small_matrices_of_a_decode_step_take_few_shares():
    """Up to 16 tokens, a matrix below 96 MiB: the count of shares that keeps the busiest
    compute unit's workgroups shortest, each share costing something by itself."""
    assert ops.gemm_splits(8, 3584, 3584) == 2    # 112 pairs of row blocks: 224 workgroups, one each
    assert ops.gemm_splits(8, 4608, 3584) == 3    # 144 pairs: 2 shares would give 32 compute units two each
    assert ops.gemm_splits(8, 5120, 5120) == 3
    assert ops.gemm_splits(8, 7168, 5120) == 1    # 224 pairs fill the chip unsplit
    assert ops.gemm_splits(8, 3584, 18944) == 9   # 130 MiB: a matter of bandwidth, many workgroups
    assert ops.gemm_splits(8, 896, 896) == 1      # 28 k-tiles: too few to share


def test_key_splits_of_decode_attention_depend_on_the_buckets_only():
    """A graph is captured for a bucket of sequences and of context; every step
    that it replays must split the keys as the captured one did."""
    from shrike_amd.engine.context import bucket
    from shrike_amd.parts.attention import decode_splits

    for kv_heads in (1, 4, 8):
        for seqs_lo, seqs_hi in ((1, 1), (3, 4), (5, 8), (33, 64), (129, 256)):
            for ctx_lo, ctx_hi in ((1, 256), (257, 512), (2049, 4096), (16385, 32768)):
                plans = {decode_splits(s, kv_heads, c)
                         for s in (seqs_lo, seqs_hi) for c in (ctx_lo, (ctx_lo + ctx_hi) // 2, ctx_hi)}
                assert len(plans) == 1
                (n,) = plans
                assert 1 <= n <= 64 and n <= max(1, bucket(ctx_hi, 256) // 256)
    assert decode_splits(8, 4, 2100) == 8 and decode_splits(64, 4, 4000) == 1 and decode_splits(1, 4, 100) == 1


def test_non_temporal_loads_from_a_size_on_and_alike_within_a_bucket():
    from shrike_amd.parts.attention import decode_streams

    # 7B heads: 8 sequences at 2,100 keys stay as they were, 64 of them or 8 at 16,000 stream
    assert not decode_streams(8, 4, 128, 2100) and not decode_streams(1, 4, 128, 4000)
    assert decode_streams(64, 4, 128, 2100) and decode_streams(8, 4, 128, 16000) and decode_streams(16, 4, 128, 2100)
    # a window bounds what is read
    assert not decode_streams(64, 4, 128, 100000, window=256)
    for seqs_lo, seqs_hi in ((3, 4), (5, 8), (33, 64), (129, 256)):
        for ctx_lo, ctx_hi in ((257, 512), (2049, 4096), (16385, 32768)):
            assert len({decode_streams(s, 4, 128, c) for s in (seqs_lo, seqs_hi) for c in (ctx_lo, ctx_hi)}) == 1


def test_decode_graphs_are_keyed_by_buckets_and_few():
    """The key of a decode graph: batch bucket, table widths in steps of 64
    pages, and what the parts' launches depend on (here the split of the keys).
    Walking batch sizes and contexts far and wide makes a few dozen keys, not
    one per context length."""
    import numpy as np
    import torch

    from shrike_amd.cache import CacheManager
    from shrike_amd.config import AttentionSpec, BlockSpec, ModelSpec, RMSNormSpec, SwiGLUSpec
    from shrike_amd.engine.runner import GRAPH_BATCH_BUCKETS, ModelRunner, StepEntry
    from shrike_amd.engine.runtime import Runtime
    from shrike_amd.models import DecoderModel

    norm = RMSNormSpec(eps=1e-6)
    mixer = AttentionSpec(num_heads=28, num_kv_heads=4, head_dim=128, qkv_bias=True, out_bias=False, scale=0.1)
    block = BlockSpec(name="model.layers.0", mixer=mixer, ffn=SwiGLUSpec(intermediate_size=64),
                      mixer_norm=norm, ffn_norm=norm)
    model = DecoderModel(ModelSpec(architecture="t", hidden_size=3584, vocab_size=100, blocks=(block,),
                                   final_norm=norm, tie_word_embeddings=False))
    model.blocks[0].mixer.dtype = torch.bfloat16  # what load() would set
    cache = CacheManager(model.cache_specs(), 16, 1 << 20)  # book-keeping only, nothing allocated
    runner = ModelRunner(model, cache, Runtime("cuda:0", torch.bfloat16))
    keys = {}
    for batch in (1, 2, 3, 8, 9, 60, 64, 65, 200, 256):
        seqs = [cache.new_sequence() for _ in range(batch)]
        for ctx in (1, 100, 256, 257, 1000, 1024, 1025, 2047, 2049, 4000, 4097, 8000):
            for s in seqs:
                cache.append(s, 0, ctx)
            entries = [StepEntry(s, [0], ctx - 1, [0]) for s in seqs]
            key = runner._graph_key(entries)
            assert key[0] == next(b for b in GRAPH_BATCH_BUCKETS if b >= batch)
            assert key[1] == (-(-(-(-ctx // 16)) // 64) * 64,)
            keys.setdefault(key, []).append((batch, ctx))
        for s in seqs:
            cache.free(s)
    assert len(keys) <= 64  # of 120 (batch, context) pairs over 8 batch buckets and 6 table widths
    # more than 256 rows, a portion, or a row that wants no logits: no graph
    seqs = [cache.new_sequence() for _ in range(2)]
    for s in seqs:
        cache.append(s, 0, 8)
    assert runner._graph_key([StepEntry(seqs[0], [0, 1], 0, [1])]) is None
    assert runner._graph_key([StepEntry(seqs[0], [0], 0, [])]) is None
    assert runner._graph_key([StepEntry(seqs[0], [0], 0, [0])] * 257) is None
    assert np.all([len(v) >= 1 for v in keys.values()])


def test_prompt_portions_are_launched_heaviest_first():
    """The list of workgroups that the attention part hands to the prefill
    kernel: runs of queries of every portion, each exactly once, the one whose
    last query reads the most keys first."""
    import numpy as np

    from shrike_amd.parts.attention import QUERY_TILE, heavy_first, portion_runs

    q_lens, starts = np.array([1, 1, 300, 40, 2048]), np.array([77, 5, 1900, 0, 0])
    run = 2 * QUERY_TILE
    seqs, q0 = portion_runs(q_lens[2:], 2, run)
    assert sorted(zip(seqs.tolist(), q0.tolist())) == (
        [(2, q) for q in range(0, 300, run)] + [(3, q) for q in range(0, 40, run)] + [(4, q) for q in range(0, 2048, run)])
    keys = starts[seqs] + q0 + run
    order = heavy_first(keys)
    assert sorted(order.tolist()) == list(range(seqs.size))
    assert (np.diff(keys[order]) <= 0).all()
    # the 300-token portion at position 1,900 reads more keys than the whole prompt's last run
    assert seqs[order][0] == 2 and q0[order][0] == 288
    assert (seqs[order][-1], q0[order][-1]) in ((3, 0), (4, 0))


def test_shares_of_a_portions_keys():
    from shrike_amd.parts.attention import portion_splits

    assert portion_splits(512, 1000) == 1  # a whole 2,048-token prompt: enough workgroups already
    assert portion_splits(128, 264) == 1   # 512 queries from position 0: too few keys to share
    assert portion_splits(128, 1800) == 4 and portion_splits(256, 3600) == 2
    assert portion_splits(32, 8000) == 16 and portion_splits(4, 100000) == 64
    assert portion_splits(0, 5) == 1


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("m, k", MATRICES)
def test_a_product_in_two_parts_is_the_same_for_every_row_count_of_a_graph_bucket(m, k, gated):
    """A product of many tokens may run as two (whole rounds of tiles, then the
    rest): graphs of 128 and 256 rows must decide as every row count they stand for."""
    for lo, hi in ((65, 128), (129, 256)):
        assert len({ops.gemm_parts(n, m, k, gated) for n in range(lo, hi + 1)}) == 1
    assert ops.gemm_parts(64, m, k, gated) == 1


def test_where_a_product_runs_in_two_parts():
    assert ops.gemm_parts(512, 18944, 3584, True) == 2    # 296 tiles of 256 x 256: 256 + 40
    assert ops.gemm_parts(2048, 18944, 3584, True) == 1   # 1,184 tiles: the rest would take a round of its own anyway
    assert ops.gemm_parts(512, 3584, 18944) == 1          # shares of k instead
    assert ops.gemm_parts(2048, 13824, 5120, True) == 2   # 864 tiles: three whole rounds, then 96 tiles' rows in smaller tiles


def test_scratch_of_float32_decode_attention_stays_near_what_is_in_use():
    """A context that crosses every table width up to 128k tokens, in a workspace whose graphs keep what it outgrew."""
    import torch

    from shrike_amd.engine.context import Workspace
    from shrike_amd.engine.runner import GRAPH_TABLE_QUANTUM
    from shrike_amd.kernels import ops
    from shrike_amd.parts.attention import F32_SPLIT_SCRATCH, f32_split_floats

    page, heads, kv_heads, dim = 16, 14, 2, 64
    for rows in (1, 4):
        space, live = Workspace("cpu", keep_outgrown=True), 0
        for width in range(GRAPH_TABLE_QUANTUM, 8192 + 1, GRAPH_TABLE_QUANTUM):
            floats = f32_split_floats(rows, heads, kv_heads, dim, width * page)
            assert floats >= ops.attention_partial_floats(rows, heads, dim, width, page)
            live = max(live, 4 * space.get("p", (floats,), torch.float32).numel())
        assert live == 4 * rows * heads * 512 * (dim + 2)
        assert space.nbytes() <= 2 * live and space.generation <= 10
    # none for one block, for rows that fill the chip, or beyond the limit
    assert f32_split_floats(1, heads, kv_heads, dim, 256) == 0 and f32_split_floats(1, heads, kv_heads, dim, 257) > 0
    assert f32_split_floats(256, heads, kv_heads, dim, 4096) == 0
    for rows in (1, 8, 64, 255):
        for keys in (1 << 12, 1 << 17, 1 << 20, 1 << 24):
            assert 4 * f32_split_floats(rows, 28, 1, 128, keys) <= F32_SPLIT_SCRATCH


def test_the_reserve_counts_scratch_that_grows_with_the_context():
    import torch

    from shrike_amd.config import AttentionSpec, BlockSpec, EngineConfig, ModelSpec, RMSNormSpec, SwiGLUSpec
    from shrike_amd.engine.llm_engine import context_reserve
    from shrike_amd.models import DecoderModel

    norm = RMSNormSpec(eps=1e-6)
    mixer = AttentionSpec(num_heads=14, num_kv_heads=2, head_dim=64, qkv_bias=True, out_bias=False, scale=0.1)
    block = BlockSpec(name="model.layers.0", mixer=mixer, ffn=SwiGLUSpec(intermediate_size=64), mixer_norm=norm, ffn_norm=norm)
    model = DecoderModel(ModelSpec(architecture="t", hidden_size=896, vocab_size=100, blocks=(block,), final_norm=norm,
                                   tie_word_embeddings=False))
    cfg = EngineConfig(max_running=100)
    model.blocks[0].mixer.dtype = torch.bfloat16
    assert context_reserve(model, cfg, 32768) == 0
    model.blocks[0].mixer.dtype = torch.float32
    row = 14 * 128 * 66 * 4  # bytes a row at 32,768 keys
    assert context_reserve(model, cfg, 32768) == 2 * 255 * row + 128 * row  # buckets 1 to 128, the largest once more
    assert context_reserve(model, EngineConfig(max_running=1), 32768) == 3 * row
    assert context_reserve(model, cfg, 100) == 0


def test_the_reserve_counts_mixers_side_by_side():
    import torch

    from shrike_amd.config import AttentionSpec
    from shrike_amd.config.specs import ParallelMixerSpec
    from shrike_amd.parts.base import build_part

    small = AttentionSpec(num_heads=2, num_kv_heads=1, head_dim=32, qkv_bias=False, out_bias=False, scale=0.1)
    large = AttentionSpec(num_heads=14, num_kv_heads=2, head_dim=64, qkv_bias=False, out_bias=False, scale=0.1)
    both = build_part("mixer", ParallelMixerSpec(branches=(("left", small), ("right", large)), eps=1e-6, scale=1.0), 896, "m")
    for _, mixer in both.branches:
        mixer.dtype = torch.float32
    assert both.context_scratch_bytes(3, 32768) == 3 * 14 * 128 * 66 * 4
    assert both.context_scratch_bytes(3, 200) == 0


def test_float32_single_tokens_of_one_block_of_keys_are_one_launch():
    """A graph of 64 pages' tables stands for contexts of up to 1,024 tokens: those of one block have one of their own."""
    import torch

    from shrike_amd.cache import CacheManager
    from shrike_amd.config import AttentionSpec, BlockSpec, ModelSpec, RMSNormSpec, SwiGLUSpec
    from shrike_amd.engine.runner import ModelRunner, StepEntry
    from shrike_amd.engine.runtime import Runtime
    from shrike_amd.models import DecoderModel

    norm = RMSNormSpec(eps=1e-6)
    mixer = AttentionSpec(num_heads=14, num_kv_heads=2, head_dim=64, qkv_bias=True, out_bias=False, scale=0.1)
    block = BlockSpec(name="model.layers.0", mixer=mixer, ffn=SwiGLUSpec(intermediate_size=64), mixer_norm=norm, ffn_norm=norm)
    model = DecoderModel(ModelSpec(architecture="t", hidden_size=896, vocab_size=100, blocks=(block,), final_norm=norm,
                                   tie_word_embeddings=False))
    model.blocks[0].mixer.dtype = torch.float32
    cache = CacheManager(model.cache_specs(), 16, 1 << 10)
    runner = ModelRunner(model, cache, Runtime("cuda:0", torch.float32))
    keys = {}
    for ctx in (1, 200, 256, 257, 300, 1024, 1025):
        seqs = [cache.new_sequence() for _ in range(2)]
        cache.append(seqs[0], 0, ctx)
        cache.append(seqs[1], 0, 1)
        keys[ctx] = runner._graph_key([StepEntry(seqs[0], [0], ctx - 1, [0]), StepEntry(seqs[1], [0], 0, [0])])
        for s in seqs:
            cache.free(s)
    assert keys[1] == keys[200] == keys[256] != keys[257] == keys[300] == keys[1024] != keys[1025]


# (query heads, key/value heads, head size, portions [(queries, position)], whether the kernel with 32 rows a wavefront serves
# them; us of the other kernel and of it)
PROMPT_KERNELS = [
    (28, 4, 128, [(512, 6000)], True),         # 98 -> 84
    (28, 4, 128, [(512, 2000)], True),         # 50 -> 47
    (28, 4, 128, [(8192, 0)], True),           # 682 -> 575
    (28, 4, 128, [(100, 8000)] * 4, True),     # 100 -> 76
    (40, 8, 128, [(170, 5000)] * 3, True),     # 202 -> 103
    (16, 1, 128, [(12, 6000)] * 32, True),     # 59 -> 46
    (14, 2, 64, [(512, 16000)], True),         # 77 -> 68
    (16, 4, 64, [(8192, 0)], True),            # 282 -> 231
    # portions that fill few of a workgroup's rows
    (28, 4, 128, [(8, 2000)] * 64, False),     # 60 / 80
    (28, 4, 128, [(12, 6000)] * 32, False),    # 94 / 140
    (40, 8, 128, [(8, 2000)] * 16, False),     # 33 / 46
    (32, 8, 128, [(20, 2000)] * 16, False),    # 38 / 50
    (32, 8, 128, [(30, 4000)] * 16, False),    # 69 / 95
    (32, 8, 128, [(17, 16000), (9, 14000)], False),  # 34 / 46
    (14, 2, 64, [(12, 6000)] * 32, False),     # 35 / 49
    (16, 4, 64, [(30, 4000)] * 16, False),     # 29 / 37
    # the last queries of one prompt in one workgroup, one to a compute unit
    (16, 4, 128, [(4096, 0)], False),          # 130 / 140
    (16, 1, 128, [(4096, 0)], False),          # 125 / 139
    (14, 2, 64, [(4096, 0)], False),           # 95 / 108
    # few keys, or few workgroups
    (28, 4, 128, [(512, 0)], False), (28, 4, 128, [(40, 3000)], False),
]


@pytest.mark.parametrize("heads, kv_heads, head_dim, steps, rows", PROMPT_KERNELS)
def test_prompt_portions_take_the_kernel_that_serves_them_sooner(heads, kv_heads, head_dim, steps, rows):
    import numpy as np
    import torch

    from shrike_amd.config import AttentionSpec
    from shrike_amd.engine.context import StepShape
    from shrike_amd.parts.attention import QUERY_TILE, PagedAttention

    mixer = PagedAttention(AttentionSpec(num_heads=heads, num_kv_heads=kv_heads, head_dim=head_dim, qkv_bias=False, out_bias=False,
                                         scale=0.1), 256, "m")
    mixer.dtype, mixer.dist_bias = torch.bfloat16, None
    queries, starts = (np.array(x) for x in zip(*steps))
    shape = StepShape(np.concatenate([[1, 1], queries]), np.concatenate([[5, 70], starts]), 16)
    mixer.prepare(shape)
    plan = shape.notes[mixer.plan_key]
    assert plan.kernel == "shared" and (plan.small == 2) == rows and plan.first_token == 2
    # every query once, whichever kernel it is
    run = (ops.attention_prefill_rows_queries(heads, kv_heads, head_dim) if rows
           else QUERY_TILE * ops.attention_prefill_shared_tiles(heads, kv_heads, head_dim, small=bool(plan.small)))
    listed = sorted(zip(shape.extras[plan.seq_name].tolist(), shape.extras[plan.q0_name].tolist()))
    assert listed == [(2 + i, q) for i, n in enumerate(queries) for q in range(0, int(n), run)] and len(listed) == plan.count


def test_experts_of_any_size_keep_the_kernel_for_long_lists():
    assert ops.moe_experts_tiles(131200, 64, 8192, 2, 2)  # 2^31 activations and more
    assert ops.moe_experts_tiles(70000, 32768, 64, 8, 2)  # elements of the tokens' rows
    assert ops.moe_experts_tiles(128, 32768, 65536, 1, 1)  # of a matrix
    assert ops.moe_experts_tiles(64, 64, 64, 8, 2) is None and ops.moe_experts_tiles(1501, 3584, 4736, 8, 2, 2) == ((256, 128), (256, 192))


def test_rows_that_are_not_aligned_take_the_shares_of_their_own_kernels():
    """As many as for a k that is no whole number of 16-byte pieces, which the same kernels take."""
    for n, m, k in ((1000, 5120, 13824), (512, 3584, 18944), (100, 3584, 3584), (300, 896, 4864), (64, 896, 4864), (8, 3584, 18944),
                    (1501, 10, 3584), (2048, 4608, 3584)):
        assert ops.gemm_splits(n, m, k, aligned=False) == ops.gemm_splits(n, m, k - 4)
        assert ops.gemm_keeps_float32(n, m, k, aligned=False) == ops.gemm_keeps_float32(n, m, k - 4)
    assert ops.gemm_splits(1000, 5120, 13824) == 1 and ops.gemm_splits(1000, 5120, 13824, aligned=False) == 3


def test_a_deferred_product_is_planned_for_the_rows_that_it_gets(monkeypatch):
    from types import SimpleNamespace

    import torch

    from shrike_amd.engine.runtime import Runtime

    runtime, calls = Runtime("cpu", torch.bfloat16), []
    monkeypatch.setattr(ops, "gemm_tiled_weight", lambda x, wt, m, k, out, **more: calls.append(more["splits"]))
    ctx = SimpleNamespace(buffer=lambda name, shape, dtype: torch.empty(shape, dtype=dtype))
    weight = SimpleNamespace(tiled=1, rows=5120, cols=13824)
    rows = torch.empty(512, 13824 + 8, dtype=torch.bfloat16)
    for x, aligned in ((rows[:, :13824], True), (rows[:, 4:13828], False), (rows.flatten()[: 512 * 13828].view(512, 13828)[:, :13824], False)):
        assert ops.rows_aligned(x) == aligned
        out = runtime.linear_deferred(ctx, "p", x, weight)
        assert out.parts.shape[0] == calls[-1] == ops.gemm_splits(512, 5120, 13824, aligned)
    assert len(set(calls)) == 2


def test_shares_of_few_rows_and_a_long_k_are_priced_with_what_the_dies_fetch():
    """The price is that of an order in which every eighth tile was a die's (with the reading norm, 896 x 18944 at 2,048 tokens 128 us in three shares of
    128 x 192, 75 in four of 128 x 256).  In runs of neighbours, the products alone: 896 x 18944 69 in three and 65 in four, 640 x 18944 52 in four
    of 128 x 192 and 48 in six, 1152 x 18944 97 in two of 128 x 192 and 84 in three."""
    for n, m, k, old in ((2048, 896, 18944, (3, (128, 192))), (2048, 640, 18944, (4, (128, 192))), (2048, 1152, 18944, (2, (128, 192))),
                         (2048, 896, 9472, (3, (128, 192))), (777, 2304, 9472, (4, (256, 128)))):
        splits = ops.gemm_splits(n, m, k)
        assert (splits, *ops.gemm_tiles(n, m, k, False, splits)) != old, (n, m, k)
    # numbers of tiles that divide among the dies, one or two rows of them, a shorter k: as without that price
    assert ops.gemm_splits(512, 3584, 18944) == 3 and ops.gemm_splits(128, 3584, 18944) == 9 and ops.gemm_splits(2048, 3584, 18944) == 1
    assert ops.gemm_splits(1119, 896, 4864) == 3
