"""Host-side choices of the kernel wrappers that need no GPU: how a product's K is cut into parts
and how many key splits the decode attention takes."""

from __future__ import annotations

import re
import subprocess

import pytest

from forge_engine_amd.engine import runner
from forge_engine_amd.kernels import build, ops


@pytest.mark.parametrize("steps", [1, 3, 4, 7, 20, 32, 76, 500])
@pytest.mark.parametrize("blocks", [1, 3, 40, 96, 160, 1000])
@pytest.mark.parametrize("most", [1, 4, 16])
def test_parts_of_k_are_never_empty_and_respect_their_bounds(steps, blocks, most):
    parts = ops._mid_parts(steps, blocks, most)
    assert 1 <= parts <= most
    per_part = -(-steps // parts)
    assert (parts - 1) * per_part < steps          # the last part still has a step
    assert parts == 1 or per_part >= 4 or steps < 8   # a part is at least four steps long


def test_parts_of_k_for_the_large_model():
    # Qwen3-4B: q/k/v (20 steps, 96 blocks of 64 rows), output (32, 40), down (76, 40)
    assert ops._mid_parts(20, 96, most=4) == 2
    assert ops._mid_parts(32, 40) == 6
    assert ops._mid_parts(76, 40) == 6


@pytest.mark.parametrize("m", [1, 8, 16, 40, 64, 100, 256, 384])
@pytest.mark.parametrize("n", [64, 320, 2560, 4096, 5120, 6144])
@pytest.mark.parametrize("k", [64, 512, 2560, 4096, 9728, 25600])
@pytest.mark.parametrize("block_rows,most", [(64, 16), (32, 4), (128, 16)])
def test_parts_of_the_product_for_portions(m, n, k, block_rows, most):
    parts = ops._wide_parts(m, n, k, block_rows, most)
    steps = k // 64
    assert 1 <= parts <= most
    per_part = -(-steps // parts)
    assert (parts - 1) * per_part < steps                    # no part without steps
    assert parts == 1 or per_part >= 8                       # a part is at least eight 64-steps long


def test_blocks_of_the_products_for_few_rows_fill_the_chip():
    # Qwen3-4B at up to 16 rows: output and down projections in six parts of 40 blocks (240 of 256 CUs)
    assert ops._wide_parts(8, 2560, 4096) == 6 and ops._wide_parts(8, 2560, 9728) == 6
    # q/k/v in blocks of 32 weight rows: 192 blocks a part, four parts (768 = three rounds of 256), never more than
    # the four that the attention launch adds up
    assert ops._wide_parts(8, 6144, 2560, 32, most=4) == 4 and ops._wide_parts(8, 6144, 4096, 32, most=4) == 4
    # Qwen3-8B: 64 blocks a part, four parts fill 256 CUs
    assert ops._wide_parts(8, 4096, 4096) == 4 and ops._wide_parts(8, 4096, 12288) == 4
    # gate/up: columns a block so that the blocks fill rounds of one a CU (9728 / 40 = 244, 12288 / 48 = 256)
    assert ops._gate_block_columns(9728) == 40 and ops._gate_block_columns(12288) == 48


@pytest.mark.parametrize("num_decode,kv_heads,max_ctx,expect", [
    (8, 8, 1040, 4), (1, 8, 2048, 16), (64, 8, 1040, 1), (1, 8, 64, 1), (1, 1, 100000, 64),
])
def test_key_splits_of_the_decode_attention(num_decode, kv_heads, max_ctx, expect):
    assert ops.decode_splits(num_decode, kv_heads, max_ctx) == expect


def test_the_fused_decode_attention_serves_what_it_says():
    import torch
    ok = dict(q_heads=32, kv_heads=8, head_dim=128, rotary_dim=128, block_size=16)
    assert ops.decode_prepare_supported(torch.bfloat16, **ok)
    assert not ops.decode_prepare_supported(torch.float32, **ok)
    for change in (dict(head_dim=96, rotary_dim=96), dict(rotary_dim=64), dict(q_heads=80), dict(block_size=8),
                   dict(block_size=48), dict(q_heads=30)):
        assert not ops.decode_prepare_supported(torch.bfloat16, **{**ok, **change}), change


def test_split_counters_outlive_their_growth():
    """A captured graph keeps the address of the counters it was recorded with: when a step needs
    more of them, the old buffer must stay alive (and zero) beside the new one."""
    import torch

    workspace = ops.Workspace()
    cpu = torch.device("cpu")
    first = workspace.split_counters(cpu, 64)
    address = first.data_ptr()
    assert workspace.split_counters(cpu, 4096) is first           # no growth: the same buffer
    grown = workspace.split_counters(cpu, 100000)
    assert grown.numel() >= 100000 and grown.data_ptr() != address
    assert any(old is first for old in workspace._retired)        # still referenced, so never handed to another tensor
    assert first.data_ptr() == address and int(first.abs().sum()) == 0
    assert workspace.split_counters(cpu, 5000) is grown           # and later launches use the larger one


def test_workspaces_are_per_owner():
    import torch

    a, b = ops.Workspace(), ops.Workspace()
    cpu = torch.device("cpu")
    with ops.use_workspace(a):
        mine = ops._split_counters(cpu, 8)
        with ops.use_workspace(b):
            assert ops._split_counters(cpu, 8) is not mine
        assert ops._split_counters(cpu, 8) is mine
    assert ops._split_counters(cpu, 8) is not mine                # outside: the default of (device, stream)


def test_every_count_of_key_splits_that_a_decode_step_can_take_is_one_that_the_gpu_tests_launch():
    import kernel_refs
    seen = set()
    for batch in list(range(1, 66)) + [96, 128, 255, 256]:
        for kv_heads in (1, 2, 3, 4, 5, 8, 16, 40, 64):
            for ctx in [1, 31, 32, 33, 127, 128, 129] + [64 * n for n in range(1, 1025)]:
                seen.add(ops.decode_splits(batch, kv_heads, ctx))
    assert seen <= set(kernel_refs.DECODE_SPLITS_TESTED)
    assert {1, 16, 17, 64} <= seen and max(seen) == 64 and min(seen) == 1
    # the table-width bound of a captured decode step (a multiple of 64 pages of 16 tokens) at batch 1 and 2 past
    # 1,024 tokens, and at batch 1 past 4,096: the merges of 9 to 16 splits and of 17 to 64
    assert ops.decode_splits(1, 8, 2048) == 16 and ops.decode_splits(2, 8, 2048) == 16
    assert ops.decode_splits(1, 8, 8192) == 32 and ops.decode_splits(1, 1, 16384) == 64


@pytest.mark.parametrize("window", [None, 1, 9, 40])
def test_the_two_references_of_paged_attention_agree(window):
    """The reference by whole matrices (used where sequences are thousands of tokens long) against
    the one that goes token by token: mixed batch, shuffled pages, a window whose passed pages were
    given back."""
    import kernel_refs
    import torch
    g = torch.Generator().manual_seed(5)
    q_heads, kv_heads, head_dim, block_size = 6, 2, 8, 4
    seqs = [(0, 7), (13, 1), (5, 9), (30, 0), (0, 1)]
    total = sum(n for _, n in seqs)
    pages = [-(-(b + n) // block_size) for b, n in seqs]
    order = torch.randperm(sum(pages) + 2, generator=g).tolist()
    table = torch.full((len(seqs), max(pages)), -1, dtype=torch.int32)
    at = 0
    for s, count in enumerate(pages):
        table[s, :count] = torch.tensor(order[at:at + count], dtype=torch.int32)
        at += count
    if window:   # pages that every query's window has passed
        for s, (before, n) in enumerate(seqs):
            table[s, :max(0, before - window + 1) // block_size] = -1
    kp = torch.randn(sum(pages) + 2, kv_heads, block_size, head_dim, generator=g)
    vp = torch.randn(sum(pages) + 2, kv_heads, head_dim, block_size, generator=g)
    q = torch.randn(total, q_heads * head_dim + 5, generator=g)
    cu = torch.tensor([0] + torch.tensor([n for _, n in seqs]).cumsum(0).tolist(), dtype=torch.int32)
    ctx = torch.tensor([b + n for b, n in seqs], dtype=torch.int32)
    kw = dict(q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim, scale=0.3, window=window)
    slow = kernel_refs.paged_attention(q, kp, vp, torch.empty(total, q_heads * head_dim), cu, ctx, table,
                                       num_seqs=len(seqs), max_q_len=9, **kw)
    fast = kernel_refs.paged_attention_by_matrices(q, kp, vp, cu, ctx, table, **kw)
    torch.testing.assert_close(fast, slow, atol=1e-5, rtol=1e-5)


def test_a_library_that_is_missing_and_cannot_be_built_fails_loudly(monkeypatch, tmp_path):
    """No fallback: without a compiled library and without a compiler, loading raises, and so does
    the preparation of a model's libraries; a file at the library's place that was built from other
    sources is not opened in its stead."""
    from forge_engine_amd.kernels import build, library

    monkeypatch.setattr(build, "library_dirs", lambda: [tmp_path])
    monkeypatch.setattr(library, "_LOADED", {})

    def no_compiler() -> str:
        raise build.KernelBuildError("hipcc not found: the HIP kernels cannot be compiled")

    monkeypatch.setattr(build, "find_hipcc", no_compiler)
    assert not library.is_built("rowwise")
    with pytest.raises(library.KernelUnavailable, match="not built and could not be compiled.*hipcc not found"):
        library.load("rowwise")
    with pytest.raises(library.KernelUnavailable, match="hipcc not found"):
        library.ensure_built(["rowwise", "sample"], announce=False)
    stale = build.library_path("rowwise", tmp_path)
    stale.write_bytes(b"\x7fELF built from sources with another hash")
    assert not library.is_built("rowwise")
    with pytest.raises(library.KernelUnavailable):
        library.load("rowwise")
    assert "rowwise" not in library._LOADED
    with pytest.raises(build.KernelBuildError, match="no kernel source"):
        build.compile_one("no_such_kernel", tmp_path)


def test_a_library_whose_source_changes_before_it_is_loaded_is_built_again(monkeypatch, tmp_path):
    from forge_engine_amd.kernels import library

    source = tmp_path / "probe.hip"
    source.write_text("before")
    compiled = []

    def compile_many(names, **_):
        for name in names:
            compiled.append(name)
            build.library_path(name, tmp_path).write_bytes(build.source_hash(name).encode())

    monkeypatch.setattr(build, "SOURCE_DIR", tmp_path)
    monkeypatch.setattr(build, "library_dirs", lambda: [tmp_path])
    monkeypatch.setattr(build, "compile_many", compile_many)
    for text, count in (("before", 1), ("before", 1), ("after", 2), ("after", 2)):
        source.write_text(text)
        library.ensure_built(["probe"], announce=False)
        assert len(compiled) == count and library.is_built("probe"), text
    build.library_path("probe", tmp_path).unlink()
    library.ensure_built(["probe"], announce=False)
    assert len(compiled) == 3


def test_operands_on_the_cpu_are_refused_before_anything_is_loaded():
    import torch

    h = torch.zeros(2, 8)
    with pytest.raises(ops.KernelError, match="no CPU path"):
        ops.add_rmsnorm(h, None, torch.ones(8), 1e-6, torch.empty(2, 8))
    with pytest.raises(ops.KernelError, match="no CPU path"):
        ops.linear(torch.zeros(2, 8), torch.zeros(4, 8))


def test_the_product_that_stores_bfloat16_needs_blocks_enough_beyond_64_rows():
    # q/k/v of Qwen3-4B and 8B (6144 weight rows) fill the chip at 65 to 256 rows; of Qwen3-0.6B and 1.7B (4096) they do not
    for rows in (65, 128, 129, 256):
        assert ops._wide_store_pays(rows, 6144) and ops._wide_store_pays(rows, 5120)
        assert not ops._wide_store_pays(rows, 4096) and not ops._wide_store_pays(rows, 2048)
    for rows in (17, 32, 64):
        assert ops._wide_store_pays(rows, 4096, 2048) and ops._wide_store_pays(rows, 7168, 5120)
        assert not ops._wide_store_pays(rows, 8192, 6144)       # 100 MB of weight: the library's


@pytest.mark.parametrize("source", ["lds_tile.h", "gemm_lds.h", "moe.hip", "gemm_f32.hip"])
def test_loads_in_assembly_leave_no_register_in_flight(source):
    """A load in an assembly statement that writes a register is waited for in the same statement: to the compiler the register is
    written there and then, and it may copy it or give it away.  (Loads into LDS write no register.)"""
    text = (build.SOURCE_DIR / source).read_text()
    statements = [m.group(0) for m in re.finditer(r"asm volatile\(.*?\);", text, re.S)]
    for statement in statements:
        code = "".join(re.findall(r'"((?:[^"\\]|\\.)*)"', statement.split(" : ")[0]))
        if re.search(r"\b(ds_read|ds_load|global_load|buffer_load|flat_load|s_load)", code.replace("global_load_lds_dwordx4", "")):
            assert re.search(r"s_waitcnt (lgkmcnt|vmcnt)\(0\)$", code), statement
    if source in ("lds_tile.h", "gemm_f32.hip"):
        assert statements


def test_which_logits_go_through_lds():
    """Both sides of every line (rows, weight rows, K), see the rule."""
    pays = ops._lds_head_pays
    for rows, weight_rows, k in ((1, 131072, 2048), (8, 151936, 2560), (8, 131072, 3584), (9, 131072, 4096), (8, 131072, 4160), (16, 151936, 5120),
                                 (17, 131072, 2048), (64, 256000, 2048), (64, 131072, 4096), (17, 151936, 2560), (32, 200064, 5120)):
        assert pays(rows, weight_rows, k), (rows, weight_rows, k)
    for rows, weight_rows, k in ((1, 131071, 2048), (1, 131072, 1984), (1, 151936, 4096), (8, 256000, 4096), (8, 151936, 3648), (65, 131072, 2048),
                                 (17, 256000, 2560), (17, 131072, 5120), (33, 151936, 2560), (64, 200064, 5120), (17, 131072, 6144), (64, 151936, 6144)):
        assert not pays(rows, weight_rows, k), (rows, weight_rows, k)


def test_which_gated_products_go_through_lds():
    """Both sides of every line of the rule: the rounds that the planned blocks make, rows, columns, K."""
    pays = ops._lds_gate_pays
    taken = ((1, 3072, 1024), (8, 9728, 2560), (2, 2064, 2432), (983, 960, 2880), (128, 9728, 2496), (8, 17408, 5120), (16, 12288, 5120), (5, 4096, 4096), (5, 12288, 4096),
             (17, 9728, 2560), (64, 9728, 2560), (32, 14336, 8192), (65, 17408, 5120), (128, 6144, 2048), (256, 9728, 2560), (192, 9728, 2560),
             (384, 3072, 1024), (700, 3072, 1024), (1536, 256, 1024), (80, 512, 5184), (320, 1536, 4096), (320, 4864, 4096))
    left = ((8, 13824, 2560), (1, 14336, 2048), (4, 4096, 4096), (8, 17408, 4096), (64, 11008, 2048), (32, 16384, 4096),
            (128, 9728, 2560), (96, 12288, 4096), (80, 256, 8192), (320, 9728, 2560), (320, 3072, 4096), (1536, 1024, 8192),
            (1537, 256, 1024), (4096, 256, 4096), (8192, 256, 8192), (769, 3072, 1024))
    for size in taken:
        assert pays(*size), size
    for size in left:
        assert not pays(*size), size


def test_which_updates_go_through_lds():
    for size in ((1, 3072, 1024), (16, 5120, 10240), (17, 8192, 4096), (256, 8192, 4096), (384, 3584, 1024), (384, 6144, 5120), (640, 4096, 8192), (768, 3584, 8192), (271, 6320, 3136),
                 (1024, 2560, 9728), (1024, 5120, 25600), (384, 8192, 16384)):
        assert ops._lds_update(*size) is not None, size
    for size in ((1, 3088, 4096), (1, 6144, 12288), (16, 5120, 10176), (257, 3840, 4096), (320, 4096, 4096), (384, 6144, 4864), (385, 3072, 4096),
                 (769, 3072, 9728), (641, 3840, 9728), (1025, 2560, 9728), (768, 4096, 8192), (257, 8192, 16128)):
        assert ops._lds_update(*size) is None, size


def test_which_projections_in_parts_go_through_lds():
    for rows, weight_rows, k in ((1, 4096, 1024), (4, 6144, 2048), (4, 6144, 2560), (4, 5120, 4096), (4, 6144, 4160), (5, 8192, 4096), (64, 6144, 2560),
                                 (17, 6144, 2560), (32, 6144, 2560), (24, 6144, 4096), (17, 4096, 1024), (32, 12288, 1024), (64, 25344, 1024)):
        tile, parts = ops._lds_in_parts(rows, weight_rows, k)
        assert 1 <= parts <= 4                                   # at most what the attention launch adds up
        if rows > 16:                                            # one round of the chip
            assert -(-rows // ops.LDS_TILES[tile][0]) * -(-weight_rows // ops.LDS_TILES[tile][1]) * parts <= 256, (rows, weight_rows, k)
    for size in ((1, 4112, 1024), (4, 6144, 4096), (4, 5136, 3072), (1, 6160, 2048), (64, 6144, 4288), (65, 4096, 1024)):
        assert ops._lds_in_parts(*size) is None, size


def test_which_stored_products_go_through_lds():
    for size in ((9, 1024, 1024), (5, 8192, 2048), (17, 2048, 1024), (192, 3072, 8192), (256, 6144, 2560), (512, 4096, 1024), (320, 4096, 2048),
                 (385, 4096, 2048), (384, 3568, 2048), (329, 3864, 3008), (384, 4096, 1984), (288, 3584, 6144)):
        assert ops._lds_store_pays(*size), size
    for size in ((4, 4096, 2048), (8, 8208, 2048), (8, 4096, 1984), (17, 2032, 1024), (193, 3072, 8192), (257, 4112, 1024), (513, 2048, 1024),
                 (321, 4096, 2048), (384, 3584, 2048), (288, 3328, 6144), (64, 10240, 5120)):
        assert not ops._lds_store_pays(*size), size


def test_which_products_of_portions_leave_the_library():
    """Both sides of the lines of 256 and 512 rows (rows, weight rows, K): beyond them all of these are the library's."""
    for size in ((512, 4096, 1024), (512, 4096, 2560), (512, 3072, 4096), (256, 6144, 2560), (256, 10240, 2048)):
        assert ops._lds_store_pays(*size), size
    for size in ((513, 4096, 1024), (768, 4096, 2048), (640, 4096, 2560), (768, 3584, 4096), (513, 3072, 4096), (257, 6144, 2560), (289, 6144, 2560),
                 (384, 7168, 3072), (384, 10240, 2048), (385, 8192, 2048), (512, 8192, 1024), (640, 6144, 2048)):
        assert not ops._lds_store_pays(*size), size


def test_parts_of_products_do_not_move_with_the_tiles_times(monkeypatch):
    """How many parts of K a product is summed in settles its bits: pinned, and the same whatever the tiles are said to take."""
    sizes = (((110, 1024, 2048), 4), ((130, 1024, 2048), 4), ((160, 1024, 3072), 4), ((256, 1024, 3072), 3), ((90, 2048, 2048), 3), ((300, 2048, 6144), 2),
             ((700, 2048, 6144), 3), ((110, 2560, 9728), 3), ((130, 2560, 9728), 3), ((160, 2560, 9728), 3), ((64, 2560, 9728), ops._lds_update(64, 2560, 9728)[1]))
    gates = ((80, 9728, 2560), (96, 12288, 4096), (64, 11008, 2048), (256, 9728, 2560), (361, 3072, 1024), (900, 3072, 1024))
    routes = [ops._lds_gate_pays(*size) for size in gates]
    assert routes == [False, False, False, True, True, False]
    for times in (1.0, 0.5, 2.0):
        monkeypatch.setattr(ops, "LDS_TILES", {tile: (rows, columns, held, one * times, two * (times if rows > 64 else 1.0))
                                               for tile, (rows, columns, held, one, two) in ops.LDS_TILES.items()})
        ops._lds_plan.cache_clear()
        assert all(ops._lds_update(*size)[1] == parts for size, parts in sizes)
        assert [ops._lds_gate_pays(*size) for size in gates] == routes
    monkeypatch.undo()
    ops._lds_plan.cache_clear()


def test_plans_are_found_once_for_all_lengths_of_as_many_tiles():
    """Portions of every length up to 1,024: a plan a weight and multiple of 32, the same for all lengths that make these tiles."""
    before = ops._lds_plan.cache_info().misses
    plans = {}
    for rows in range(17, 1025):
        plan = ops.lds_plan(rows, 2568, 4160, 4 * 2568, 8, summed=True)
        assert plans.setdefault(-(-rows // 32), plan) == plan
    assert ops._lds_plan.cache_info().misses - before <= 32
    for rows in range(1, 17):                                # (few rows: by the count itself)
        tile, parts = ops.lds_plan(rows, 2568, 4160, 4 * 2568, 8, summed=True)
        assert ops.LDS_TILES[tile][0] == 16 and 1 <= parts <= 8


def test_key_runs_that_a_caller_asks_for():
    assert ops._runs_asked_for(None, None) is None and ops._runs_asked_for(3, None) == 3 and ops._runs_asked_for(None, 5) == -5
    for bad in ((0, None), (-4, None), (None, 0), (None, -4), (2, 4), (2, 0)):
        with pytest.raises(ops.KernelError):
            ops._runs_asked_for(*bad)


@pytest.mark.parametrize("rows,weight_rows,k,before,split", [
    (20, 512, 6144, 16.4, 46.4), (21, 256, 5120, 14.1, 39.2), (32, 512, 5120, 29.1, 41.1), (47, 768, 6144, 38.6, 46.5), (17, 512, 2048, 10.7, 17.3),
    (60, 4096, 1024, 52.0, 10.5), (60, 4096, 2048, 62.0, 19.0), (17, 6144, 4096, 59.8, 35.7), (18, 6144, 1024, 25.6, 12.1)])
def test_float32_products_of_17_to_64_rows_take_the_kernel_that_was_measured_to_be_faster(rows, weight_rows, k, before, split):
    assert ops._split_pays(rows, weight_rows, k, 1) == (split < before)


def test_float32_products_of_more_rows_take_the_more_exact_kernel_unless_it_is_far_slower():
    for size in ((65, 4096, 1024), (92, 4608, 2048), (96, 768, 8192), (298, 1024, 1024), (655, 768, 12288), (700, 4096, 1024), (700, 6144, 1024),
                 (1024, 4096, 2048), (200, 4096, 512)):
        assert ops._split_pays(*size, 1), size
    for size in ((65, 300, 256), (371, 512, 256), (17, 6144, 256), (48, 3200, 512), (86, 1536, 352)):
        assert not ops._split_pays(*size, 1), size


def test_which_float32_products_of_few_rows_take_a_ring_for_each_wave():
    """Both sides of every line (rows, weight rows or columns, K), see the rules."""
    for taken, left, pays in (
            (((9, 64, 1024), (16, 512, 2048), (9, 768, 3072), (9, 768, 8192), (16, 1024, 4096), (9, 1024, 12288), (12, 1280, 12288), (16, 8192, 2048), (8, 2048, 1152)),
             ((9, 64, 2048), (16, 512, 3072), (15, 256, 12288), (9, 512, 8192), (16, 768, 4096), (16, 768, 12288), (16, 1024, 6144), (1, 2048, 2048), (8, 1536, 1024), (9, 4096, 224)),
             ops._ring_float32_pays),
            (((1, 64, 1024), (8, 512, 2048), (4, 768, 2816), (1, 1024, 3072), (8, 1024, 8192), (1, 1280, 12288), (9, 256, 4096), (16, 512, 12288), (9, 64, 3072)),
             ((2, 256, 9728), (8, 256, 2048), (1, 512, 3072), (8, 768, 4096), (1, 1024, 6144), (8, 1024, 12288), (9, 256, 6144), (16, 64, 4096), (1, 4096, 224)),
             ops._ring_gate_float32_pays),
            (((1, 4096, 1024), (8, 4096, 2048), (1, 2560, 9728), (4, 768, 1152), (16, 2050, 1056)), ((1, 2048, 2048), (8, 1024, 4096), (4, 512, 1024), (9, 512, 4096)),
             ops._unscaled_float32_pays)):
        assert [size for size in taken if not pays(*size)] == [] and [size for size in left if pays(*size)] == []


def test_which_updates_are_left_to_the_product_with_the_norm_behind_it():
    """Both sides of every line (rows, weight rows, K), see the rules; every size of a decode step that was measured faster stays."""
    for taken, left, pays in (
            (((1, 1024, 25600), (4, 512, 11264), (8, 1536, 25600), (5, 512, 8192), (16, 768, 8192), (8, 1024, 11264), (12, 2048, 12288), (16, 2048, 11264),
              (16, 2560, 9728), (16, 4096, 12288), (16, 5120, 25600), (8, 2560, 9728), (1, 1024, 2048)),
             ((1, 512, 12288), (8, 1024, 17408), (8, 768, 17408), (12, 1280, 12288), (12, 2048, 17408), (16, 768, 9728), (16, 1280, 9728), (16, 2560, 14336),
              (16, 4096, 25600)), ops._update_norm_pays),
            (((8, 1024, 3072), (1, 2048, 6144), (4, 2048, 8192), (8, 2304, 25600), (1, 2560, 9728), (9, 512, 25600), (16, 2048, 6144)),
             ((8, 1024, 4096), (4, 1024, 8192), (1, 1536, 6144), (8, 2048, 12288), (1, 512, 2048)), ops._update_norm_float32_pays)):
        assert [size for size in taken if not pays(*size)] == [] and [size for size in left if pays(*size)] == []


def test_which_projections_of_few_rows_come_whole_from_a_ring():
    for size in ((1, 512, 2048), (16, 2047, 1024), (8, 2048, 12288), (9, 2048, 3072), (16, 2560, 3712), (12, 3072, 4352), (16, 3585, 9728), (16, 6144, 4096)):
        assert ops._ring_parts_pays(*size), size
    for size in ((1, 512, 2112), (9, 2048, 4096), (16, 2560, 9728), (16, 3584, 6144), (1, 6152, 2560)):
        assert not ops._ring_parts_pays(*size), size


def test_lanes_of_a_recurrences_column():
    for columns, heads, seqs in ((64, 4, 1), (64, 4, 4), (128, 8, 1), (256, 4, 1), (1, 1, 256)):
        assert ops._recurrence_lanes(columns, heads, seqs) == 64, (columns, heads, seqs)
    for columns, heads, seqs in ((257, 4, 1), (64, 4, 5), (128, 4, 3), (256, 4, 2), (257, 8, 6)):
        assert ops._recurrence_lanes(columns, heads, seqs) == 32, (columns, heads, seqs)


def test_which_steps_of_a_recurrence_are_one_launch():
    pays = ops.linear_recurrence_step_pays
    for seqs, heads, key_dim, columns in ((1, 8, 128, 257), (1, 1, 128, 513), (1, 1, 256, 144), (1, 2, 16, 513), (5, 1, 256, 513), (1, 5, 256, 513), (2, 3, 200, 513)):
        assert pays(seqs, heads=heads, key_dim=key_dim, columns=columns), (seqs, heads, key_dim, columns)
    for seqs, heads, key_dim, columns in ((1, 1, 256, 513), (2, 1, 256, 513), (4, 1, 200, 145), (1, 4, 132, 400)):
        assert not pays(seqs, heads=heads, key_dim=key_dim, columns=columns), (seqs, heads, key_dim, columns)


def test_which_float32_values_go_to_blocks_of_their_own():
    """(tokens, sequences, query heads, key heads, head size): both sides of every line."""
    for case in ((17, 1, 32, 8, 128), (17, 8, 8, 2, 256), (24, 24, 16, 8, 128), (64, 64, 16, 8, 256), (17, 17, 4, 1, 64), (200, 200, 16, 4, 64)):
        assert ops._few_values_apart(*case), case
    for case in ((16, 1, 16, 8, 128), (17, 9, 8, 2, 256), (64, 64, 8, 2, 256), (128, 128, 8, 2, 256), (17, 17, 32, 8, 128), (64, 64, 2, 1, 128),
                 (23, 23, 16, 8, 128), (63, 63, 16, 8, 256)):
        assert not ops._few_values_apart(*case), case


def test_float32_updates_of_short_k_keep_the_kernel_they_had():
    for size in ((34, 3072, 576), (80, 768, 320), (123, 2560, 256), (56, 6144, 256), (724, 256, 512)):
        assert not ops._split_pays(*size, ops.SPLIT_MOST_PARTS), size
    for size in ((700, 1024, 2048), (700, 1024, 3072), (700, 2048, 6144), (20, 1024, 3072), (100, 1024, 2048), (60, 4096, 2048), (17, 2560, 4096)):
        assert ops._split_pays(*size, ops.SPLIT_MOST_PARTS), size


@pytest.mark.parametrize("compute", ["bfloat16", "float32"])
@pytest.mark.parametrize("stored", ["bfloat16", "float32"])
def test_rows_without_their_factors_go_to_matrices_of_their_own_dtype_only(stored, compute):
    """A matrix that a checkpoint stores in 32 bits stays so in a bfloat16 model, beside others that are not: what reads its rows from a norm
    widens them, which no product that applies the factors does."""
    from types import SimpleNamespace

    import torch

    from forge_engine_amd.parts import BuildContext
    from forge_engine_amd.parts.attention import GroupedQueryAttention
    from forge_engine_amd.parts.mlp import SwiGLU

    ctx = BuildContext(torch.device("cpu"), getattr(torch, compute))
    mlp = SwiGLU(ctx, "mlp", hidden_size=1024, intermediate_size=1024)
    mlp.gate_up_weight = torch.zeros(2048, 1024, dtype=getattr(torch, stored))
    assert mlp.takes_unscaled(4) == (stored == compute)
    mixer = GroupedQueryAttention.__new__(GroupedQueryAttention)
    mixer.ctx, mixer.general, mixer.qkv_bias, mixer.qkv_weight = ctx, False, None, torch.zeros(2048, 1024, dtype=getattr(torch, stored))
    mixer.position = SimpleNamespace(rotary=lambda: None)
    batch = SimpleNamespace(num_decode=None)
    assert mixer.takes_unscaled(12, batch, None) == (stored == compute)


def _reads_in_flight_at_barriers(listing: str) -> dict[str, list[int]]:
    """Per kernel of a gfx950 listing and barrier in it, the most reads of LDS that may be under way there over all paths that lead to it."""
    kernels: dict[str, list[str]] = {}
    code = None
    for line in listing.splitlines():
        if start := re.match(r"(_Z\w+):", line):
            code = kernels.setdefault(start.group(1), [])
        elif re.match(r"\.Lfunc_end", line):
            code = None
        elif code is not None and (text := line.split(";")[0].strip()):
            code.append(text)
    found = {}
    for name, code in kernels.items():
        label_at = {text[:-1]: i for i, text in enumerate(code) if re.fullmatch(r"\.LBB\w+:", text)}
        most, barriers, work = {0: 0}, {}, [0]
        while work:                         # each walk goes on to the next jump's target, or to where it learns nothing new
            i = work.pop()
            pending = most[i]
            while True:
                text = code[i]
                if text.startswith(("ds_read", "ds_load")):
                    pending = min(pending + 1, 64)
                elif wait := re.match(r"s_waitcnt\b.*lgkmcnt\((\d+)\)", text):
                    pending = min(pending, int(wait.group(1)))
                elif text.startswith("s_barrier"):
                    barriers[i] = max(barriers.get(i, 0), pending)
                jump = re.match(r"s_c?branch\S*\s+(\.LBB\w+)", text)
                if jump and most.get(label_at[jump.group(1)], -1) < pending:
                    most[label_at[jump.group(1)]] = pending
                    work.append(label_at[jump.group(1)])
                i += 1
                if text.startswith(("s_endpgm", "s_branch")) or i == len(code):
                    break
                if code[i].startswith(".LBB"):
                    if most.get(i, -1) >= pending:
                        break
                    most[i] = pending
        found[name] = list(barriers.values())
    return found


@pytest.mark.parametrize("source", ["gemm_split", "gemm_planes", "gemm_f32", "moe"])
def test_no_read_of_lds_is_under_way_at_a_barrier_behind_which_its_buffer_is_filled(source, tmp_path):
    """A wave that passes such a barrier requests loads into the buffer that it or another has just read: the compiler keeps reads before
    the barrier, but waits for them only where they are used, which it may move behind it.  (``gemm_tile``, whose buffers are filled two
    barriers later, reads across them.)"""
    listing = tmp_path / f"{source}.s"
    flags = [flag for flag in build.HIPCC_FLAGS if flag != "-shared"]
    subprocess.run([build.find_hipcc(), *flags, "-S", "--cuda-device-only", "-o", str(listing), str(build.SOURCE_DIR / f"{source}.hip")],
                   check=True, capture_output=True)
    found = _reads_in_flight_at_barriers(listing.read_text())
    assert any(found.values())
    assert {name: at for name, at in found.items() if any(at)} == {}


def _that_leave_m0_as_it_is() -> list[str]:
    return sorted(path.stem for path in build.SOURCE_DIR.glob("*.hip") if '#include "lds_load.h"' in path.read_text())


def test_only_one_place_leaves_m0_as_it_is():
    """A statement that changes m0 without putting it back, in lds_load.h; the warning that the compiler may not honour it is off there alone."""
    assert {"gemm_big", "gemm_planes"} <= set(_that_leave_m0_as_it_is()) and not any("inline-asm" in flag for flag in build.HIPCC_FLAGS)
    for path in [*build.SOURCE_DIR.glob("*.hip"), *build.SOURCE_DIR.glob("*.h")]:
        text = path.read_text()
        assert ('"m0"' in text or "-Winline-asm" in text) == (path.name == "lds_load.h"), path.name
        for statement in re.findall(r'asm volatile\("([^"]*\bs_mov_b32 m0[^"]*)"', text):
            assert path.name == "lds_load.h" or statement.endswith("s_mov_b32 m0, %0"), path.name


@pytest.mark.parametrize("source", _that_leave_m0_as_it_is())
def test_loads_into_lds_have_m0_to_themselves(source, tmp_path):
    """Nothing but the loads into LDS touches m0, which they leave as it is, and nothing goes to scratch memory."""
    listing = tmp_path / f"{source}.s"
    flags = [flag for flag in build.HIPCC_FLAGS if flag != "-shared"]
    subprocess.run([build.find_hipcc(), *flags, "-S", "--cuda-device-only", "-o", str(listing), str(build.SOURCE_DIR / f"{source}.hip")],
                   check=True, capture_output=True)
    text = listing.read_text()
    lines = [line.split(";")[0].strip() for line in text.splitlines()]
    uses = [line for line in lines if re.search(r"\bm0\b", line)]
    assert uses and all(line.startswith("s_mov_b32 m0, s") for line in uses)
    assert not any(line.startswith(("scratch_", "buffer_store", "buffer_load")) for line in lines)


def test_which_loads_pass_the_caches_is_known_when_a_product_is_compiled(tmp_path):
    """Loads of the products through LDS pass the caches (nt) in an instance of each tile for one tile of x.  Which of them do is known when the
    kernel is compiled, but for the share of a step that begins inside the first operand: without one, the instances have as many loads
    and branches as the others."""
    listing = tmp_path / "gemm_wide.s"
    flags = [flag for flag in build.HIPCC_FLAGS if flag != "-shared"]
    subprocess.run([build.find_hipcc(), *flags, "-S", "--cuda-device-only", "-o", str(listing), str(build.SOURCE_DIR / "gemm_wide.hip")],
                   check=True, capture_output=True)
    kernels = re.findall(r"^(_Z\w*gemm_lds_kernel\w+):(.*?)^\.Lfunc_end", listing.read_text(), re.M | re.S)
    assert kernels
    past, shapes = {}, {}
    for name, code in kernels:
        mi, ni, wm, wn, kg, *_ = (int(v) for v in re.findall(r"Li(\d+)E", name))
        assert "global_load_lds_dwordx4" in code
        past.setdefault((mi, ni, wm, wn), set()).add(bool(re.search(r"global_load_lds_dwordx4 .*\bnt\b", code)))
        if 2 * mi * wm % (wm * wn * kg) == 0:
            shapes.setdefault(re.match(r"(.*)Lb[01]EEE", name).group(1), set()).add((code.count("global_load_lds_dwordx4"), code.count("s_cbranch")))
    assert shapes and all(len(kinds) == 1 for kinds in shapes.values())
    assert len(past) == 14 and all(kinds == {False, True} for kinds in past.values())


def test_tiles_of_96_rows_pass_the_caches_for_one_tile_of_x_too(tmp_path):
    """Every tile and ending of the library of these tiles has both instances, whose weight rows pass the caches and whose all stay."""
    listing = tmp_path / "gemm_lds96.s"
    flags = [flag for flag in build.HIPCC_FLAGS if flag != "-shared"]
    subprocess.run([build.find_hipcc(), *flags, "-S", "--cuda-device-only", "-o", str(listing), str(build.SOURCE_DIR / "gemm_lds96.hip")],
                   check=True, capture_output=True)
    past = {}
    for name, code in re.findall(r"^(_Z\w*gemm_lds_kernel\w+):(.*?)^\.Lfunc_end", listing.read_text(), re.M | re.S):
        mi, ni, wm, wn, _, _, ending = (int(v) for v in re.findall(r"Li(\d+)E", name))
        past.setdefault((16 * mi * wm, 16 * ni * wn, ending), set()).add(bool(re.search(r"global_load_lds_dwordx4 .*\bnt\b", code)))
    assert set(past) == {tuple(ops.LDS_TILES[tile][:2]) + (ending,) for tile in ops.LDS_TILES if ops.LDS_TILES[tile][0] == 96 for ending in (0, 1, 2)}
    assert all(kinds == {False, True} for kinds in past.values())


def test_values_of_long_pages_stay_in_the_caches(tmp_path):
    """The decode attention has instances whose values pass the caches, for pages in which an instruction takes whole lines of them, and
    others whose loads all stay there, for pages in which two waves share a line."""
    listing = tmp_path / "attention_decode.s"
    flags = [flag for flag in build.HIPCC_FLAGS if flag != "-shared"]
    subprocess.run([build.find_hipcc(), *flags, "-S", "--cuda-device-only", "-o", str(listing), str(build.SOURCE_DIR / "attention_decode.hip")],
                   check=True, capture_output=True)
    kernels = re.findall(r"^(_Z\w*paged_decode_kernel\w+):(.*?)^\.Lfunc_end", listing.read_text(), re.M | re.S)
    forms = {}
    for name, code in kernels:
        head, past = re.match(r"(.*)Lb([01])EEv", name).groups()
        loads = len(re.findall(r"global_load_lds_dwordx4 v\[\d+:\d+\], off nt", code))      # (a wave's address for keys, a lane's for values)
        assert loads == (2 * int(re.search(r"ILi(\d+)E", name).group(1)) // 16 if past == "1" else 0)      # the first block's and the next one's
        forms.setdefault(head, set()).add(past)
    assert forms and all(kinds == {"0", "1"} for kinds in forms.values())


@pytest.mark.parametrize("rows,weight_rows,k,most_parts,split,planes,made", [
    (768, 1024, 1024, 1, 21.6, 25.9, 20.0), (560, 6976, 512, 1, 38.5, 46.9, None), (403, 1024, 2048, 6, 25.9, 29.6, 23.1), (92, 2560, 2560, 6, 21.1, 24.9, None),
    (934, 1536, 512, 1, 17.0, 19.9, 14.5), (78, 3828, 3828, 1, 54.9, 63.9, 64.0), (700, 6144, 1024, 1, 68.0, 59.0, 52.0), (700, 2048, 6144, 6, 130.0, 100.0, 96.0)])
def test_float32_products_of_prompts_take_planes_where_they_were_measured_to_be_faster(rows, weight_rows, k, most_parts, split, planes, made):
    """us, the weight coming from memory: through gemm_split, through planes with the pass over the rows, and without it."""
    assert isinstance(ops._product_plan(rows, weight_rows, k, most_parts, True)[0], tuple) == (planes < split)
    assert made is None or isinstance(ops._product_plan(rows, weight_rows, k, most_parts, True, made=True)[0], tuple) == (made < split)


def test_float32_plans_of_planes_are_shared_by_the_lengths_of_a_fragment_of_rows():
    before = ops._planes_instead.cache_info().misses
    for rows in range(497, 513):
        assert ops._product_plan(rows, 2056, 4104, 6, True) == ops._product_plan(512, 2056, 4104, 6, True)
    assert ops._planes_instead.cache_info().misses - before == 1
    for rows, planes in ((64, True), (81, True), (512, False)):      # ... and gemm_split's own by the length itself
        assert ops._product_plan(rows, 1024, 4096, 6, planes) == ops._split_plan(rows, 1024, 4096, 6)


def test_float32_plans_of_planes_lose_no_precision():
    """Over the sizes of prompts: never the long sums of the largest tiles where gemm_split's plan gathers its own, and never longer ones than its."""
    for rows in (66, 96, 130, 250, 333, 500, 700, 1400):
        for n, k, most_parts in ((4096, 1024, 1), (6144, 1024, 1), (12288, 2048, 1), (4096, 2048, 1), (1024, 2048, 6), (1024, 3072, 6), (2048, 6144, 6), (2560, 9728, 6)):
            for made in (False, True):
                (tile, parts), (split, split_parts) = ops._product_plan(rows, n, k, most_parts, True, made), ops._split_plan(rows, n, k, most_parts)
                if not isinstance(tile, tuple):
                    assert (tile, parts) == (split, split_parts)
                elif tile[0] * tile[1] > 10:
                    assert ops.SPLIT_TILES[split][2] == 64 and 0.75 * k / parts <= k / split_parts


def test_rows_of_decode_steps_are_turned_away_unseen():
    """Whether rows come with their parts is asked of every part of every layer: by the rows first, which say no for any decode step."""
    for rows in (1, 17, 64):
        assert not ops.takes_split(rows, None) and not ops.takes_split(rows, None, update=True) and ops._made_plan(rows, 4096, 1024, False) is None
    assert ops._made_plan(700, 4096, 1024, False) == ops._product_plan(700, 4096, 1024, 1, True, made=True)
    assert ops._made_plan(700, 1024, 3072, True) == ops._product_plan(700, 1024, 3072, ops.SPLIT_MOST_PARTS, True, made=True)
    assert ops._made_plan(700, 1024, 1000, False) is None and ops._made_plan(700, 4096, 8256, False) is None
    assert ops._big_update_parts(2048, 2560, 8128) == 0 and ops._big_update_parts(2048, 2560, 8192) == 3


@pytest.mark.parametrize("elements,dtype,captured,hidden", [
    (100_925_440, "bfloat16", 1288, 1289), (50_331_648, "bfloat16", 2582, 2583), (15_728_640, "bfloat16", 4096, 8266),
    (15_728_640, "float32", 1271, 1272), (50_331_648, "float32", 397, 398)])
def test_steps_whose_launches_the_gpu_hides_are_known_by_their_size(elements, dtype, captured, hidden):
    """Both sides of the line, by the tokens and the model alone: no clock has a say in which of two forms of a step runs."""
    import types

    import torch

    step = types.SimpleNamespace(_products_per_token=elements, dtype=getattr(torch, dtype))
    assert not runner.ModelRunner._launches_hidden(step, captured) and runner.ModelRunner._launches_hidden(step, hidden)


def test_products_per_token_count_what_a_token_is_multiplied_with():
    """A layer's matrices, of the experts those that a token is sent to; no lookups, no norms, no head."""
    import torch

    from forge_engine_amd.config import load_model_config
    from forge_engine_amd.engine import build_model
    from forge_engine_amd.parts.base import BuildContext
    from forge_engine_amd.parts.moe import RoutedExperts

    dense = {"architectures": ["Qwen3ForCausalLM"], "model_type": "qwen3", "hidden_act": "silu", "vocab_size": 320, "hidden_size": 96,
             "intermediate_size": 160, "num_hidden_layers": 3, "num_attention_heads": 6, "num_key_value_heads": 2, "head_dim": 64,
             "max_position_embeddings": 128, "rms_norm_eps": 1e-6, "rope_theta": 10000.0, "tie_word_embeddings": False, "eos_token_id": None}
    model = build_model(load_model_config(dense), dtype="bfloat16", device=torch.device("cpu"))
    assert model.products_per_token() == 96 * (6 + 2 + 2) * 64 + 6 * 64 * 96 + 3 * 96 * 160
    ctx = BuildContext(torch.device("cpu"), torch.bfloat16)
    experts = RoutedExperts(ctx, "m", hidden_size=48, experts=8, top=2, intermediate_size=80, limit=1.0, shared_size=32)
    assert experts.products_per_token(experts.param_specs()) == 8 * 48 + 2 * 3 * 48 * 80 + 3 * 48 * 32


def test_float32_decode_attention_sizes_and_splits():
    import torch

    ok = dict(q_heads=16, kv_heads=8, head_dim=128, rotary_dim=128, block_size=16)
    assert ops.decode_f32_supported(torch.float32, **ok) and ops.decode_f32_supported(torch.float32, **{**ok, "head_dim": 64, "rotary_dim": 64})
    assert not ops.decode_f32_supported(torch.bfloat16, **ok)
    for change in ({"head_dim": 256, "rotary_dim": 256}, {"rotary_dim": 64}, {"q_heads": 72}, {"q_heads": 12}, {"block_size": 8}, {"block_size": 48}):
        assert not ops.decode_f32_supported(torch.float32, **{**ok, **change}), change
    for (sequences, kv_heads, reach), splits in (((1, 8, 1024), 8), ((1, 8, 100), 1), ((4, 8, 1024), 8), ((8, 8, 1024), 4), ((1, 8, 8192), 32), ((1, 1, 100000), 64), ((64, 8, 4096), 1)):
        assert ops.decode_f32_splits(sequences, kv_heads, reach) == splits, (sequences, kv_heads, reach)
