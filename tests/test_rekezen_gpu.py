"""Rekezen on the GPU: its kernels alone against their plain references (tests/kernel_refs.py), and
the model against the plain implementation (tests/plain_rekezen.py) in float32 and bfloat16 over
traces that cut the same requests in different ways."""

from __future__ import annotations

import pytest
import torch

import kernel_refs as refs
import rekezen_util as ku
import replay_util as ru

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

CONFIGS = dict(ku.CONFIGS, M=ku.MEDIUM)
LENGTHS = {"A": (5, 1, 14, 27, 90), "B": (2, 9, 21, 33, 64), "C": (7, 18, 3, 1, 40), "M": (4, 45, 150, 83, 1)}
BLOCKS = dict(ku.BLOCK_SIZE, M=16)


def close(got, want, dtype):
    if dtype == torch.float32:
        torch.testing.assert_close(got.float().cpu(), want.float(), rtol=2e-5, atol=2e-5)
    else:
        torch.testing.assert_close(got.float().cpu(), want.float(), rtol=2e-2, atol=2e-2)


# ------------------------------------------------------------------ kernels alone

@pytest.mark.parametrize("streams,width,parts", [(1, 40, 0), (3, 48, 1), (4, 256, 3), (8, 130, 2), (2, 4096, 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_hyper_norm_kernel(streams, width, parts, dtype):
    from forge_engine_amd.kernels import ops
    g = torch.Generator().manual_seed(streams * 100 + width)
    rows = 37
    x = torch.randn(streams, rows, width, generator=g) * 3
    update = None if parts == 0 else (torch.randn(rows, width, generator=g) if parts == 1 else torch.randn(parts, rows, width, generator=g))
    mix = torch.eye(streams) + 0.2 * torch.randn(streams, streams, generator=g)
    share, read = torch.randn(streams, generator=g), torch.randn(streams, generator=g)
    weight, bias = 1 + 0.1 * torch.randn(width, generator=g), 0.1 * torch.randn(width, generator=g)
    for use_mix, use_read, rms, chosen in ((True, True, False, None), (False, False, True, None), (True, False, False, [5, 0, 36, 5])):
        want_x = x.clone()
        pick = None if chosen is None else torch.tensor(chosen, dtype=torch.int32)
        n = rows if chosen is None else len(chosen)
        want = refs.hyper_norm(want_x, update, mix if use_mix else None, share if use_mix else None, read if use_read else None,
                               weight, None if rms else bias, 1e-5, torch.empty(n, width, dtype=dtype), rows=pick,
                               store=chosen is None, rms=rms)
        got_x = x.clone().to(DEV)
        got = ops.hyper_norm(got_x, None if update is None else update.to(DEV), mix.to(DEV) if use_mix else None,
                             share.to(DEV) if use_mix else None, read.to(DEV) if use_read else None, weight.to(DEV),
                             None if rms else bias.to(DEV), 1e-5, torch.empty(n, width, dtype=dtype, device=DEV),
                             rows=None if pick is None else pick.to(DEV), store=chosen is None, rms=rms)
        close(got, want, dtype)
        close(got_x, want_x, torch.float32)
    if update is not None:      # the update alone, nothing read
        want_x, got_x = x.clone(), x.clone().to(DEV)
        refs.hyper_norm(want_x, update, mix, share, None, None, None, 0.0, None)
        ops.hyper_norm(got_x, update.to(DEV), mix.to(DEV), share.to(DEV), None, None, None, 0.0, None)
        close(got_x, want_x, torch.float32)


@pytest.mark.parametrize("rows", [8, 37, 513, 600])          # up to 512 rows of 2,048 and more take more threads a row
@pytest.mark.parametrize("streams,width", [(1, 1024), (4, 1024), (4, 1028), (3, 2044), (1, 2048), (4, 2048), (4, 2052), (2, 4096), (4, 4096), (2, 4100)])
def test_hyper_norm_has_the_bits_of_the_general_kernel(streams, width, rows):
    """Rows with an update in up to four parts go to a kernel that requests all of a row's operands before it uses any; with a fifth part
    (of zeros here) they go to the general one.  The same bits in the streams and in the rows, on both sides of every line between
    instances, with and without each operand that may be absent; and the plain reference's values, five parts of numbers among them."""
    from forge_engine_amd.kernels import ops
    g = torch.Generator().manual_seed(streams * 10000 + width + rows)
    mix = torch.eye(streams) + 0.2 * torch.randn(streams, streams, generator=g)
    share, read = torch.randn(streams, generator=g), torch.randn(streams, generator=g)
    weight, bias, shift = 1 + 0.1 * torch.randn(width, generator=g), 0.1 * torch.randn(width, generator=g), torch.randn(width, generator=g)
    dev = lambda t: None if t is None else t.to(DEV)
    for parts in (0, 1, 2, 4, 5):
        x = torch.randn(streams, rows, width, generator=g) * 3
        update = torch.randn(parts, rows, width, generator=g) if parts else None
        five = torch.zeros(5, rows, width)
        if parts:
            five[:parts] = update
        for use_mix, use_read, rms, use_shift, dtype in ((True, True, False, False, torch.bfloat16), (False, False, True, True, torch.float32),
                                                         (True, False, False, True, torch.float32), (False, True, True, False, torch.bfloat16)):
            use_mix = use_mix and (parts > 0 or use_shift)      # without either the streams are left as they are
            rest = (mix if use_mix else None, share if use_mix else None, read if use_read else None, weight, None if rms else bias)
            results = []
            for brought in (update, five):
                got_x, out = dev(x).clone(), torch.full((rows, width), float("nan"), dtype=dtype, device=DEV)
                ops.hyper_norm(got_x, dev(brought), *(dev(t) for t in rest), 1e-5, out, rms=rms, shift=dev(shift if use_shift else None))
                results.append((got_x, out))
            for here, there in zip(*results):
                assert torch.equal(here.view(torch.int16), there.view(torch.int16)), (parts, use_mix, use_read, rms, use_shift)
            want_x = x.clone()
            want = refs.hyper_norm(want_x, update, *rest, 1e-5, torch.empty(rows, width, dtype=dtype), rms=rms, shift=shift if use_shift else None)
            close(results[0][1], want, dtype)
            close(results[0][0], want_x, torch.float32)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_token_pair_embedding_kernel(dtype):
    from forge_engine_amd.kernels import ops
    g = torch.Generator().manual_seed(5)
    vocab, hidden, buckets = 70, 24, 13
    table, pairs = torch.randn(vocab, hidden, generator=g).to(dtype), torch.randn(buckets + 1, hidden, generator=g).to(dtype)
    # three sequences: one from its first token, one going on (its first token of the step reads the slot), one single token
    ids = torch.tensor([3, 9, 9, 60, 1, 2, 69], dtype=torch.int32)
    positions = torch.tensor([0, 1, 2, 7, 8, 9, 4], dtype=torch.int32)
    token_seq = torch.tensor([0, 0, 0, 1, 1, 1, 2], dtype=torch.int32)
    cu_q = torch.tensor([0, 3, 6, 7], dtype=torch.int32)
    slots = torch.tensor([2, 0, 3], dtype=torch.int32)
    previous = torch.tensor([[41], [7], [55], [12], [0]], dtype=torch.int32)
    want_prev, want = previous.clone(), torch.empty(7, hidden)
    refs.embed_token_pairs(ids, table, pairs, positions, token_seq, cu_q, slots, want_prev, want, num_seqs=3, buckets=buckets,
                           mul_prev=1000003, mul_cur=77)
    got_prev, got = previous.clone().to(DEV), torch.empty(7, hidden, device=DEV)
    ops.embed_token_pairs(ids.to(DEV), table.to(DEV), pairs.to(DEV), positions.to(DEV), token_seq.to(DEV), cu_q.to(DEV), slots.to(DEV),
                          got_prev, got, num_seqs=3, buckets=buckets, mul_prev=1000003, mul_cur=77)
    assert torch.equal(got.cpu(), want) and torch.equal(got_prev.cpu(), want_prev)
    assert want_prev[:, 0].tolist() == [2, 7, 9, 69, 0]


@pytest.mark.parametrize("heads,kv_heads,dim,vdim,rot", [(4, 2, 16, 24, 8), (6, 2, 128, 128, 64), (2, 2, 12, 20, 12), (3, 1, 64, 8, 0)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_whole_norm_rope_write_kernel(heads, kv_heads, dim, vdim, rot, dtype):
    from forge_engine_amd.kernels import ops
    g = torch.Generator().manual_seed(heads + dim)
    tokens, block, pages = 9, 4, 12
    width = heads * dim + kv_heads * (dim + vdim) + 5
    qkv = (torch.randn(tokens, width, generator=g) * 2).to(dtype)
    qw, kw = 1 + 0.2 * torch.randn(heads * dim, generator=g), 1 + 0.2 * torch.randn(kv_heads * dim, generator=g)
    inv_freq = torch.rand(max(rot // 2, 1), generator=g)[:rot // 2]
    positions = torch.tensor([0, 1, 2, 3, 4, 17, 18, 19, 1000], dtype=torch.int32)
    token_seq = torch.tensor([0, 0, 0, 0, 0, 1, 1, 1, 2], dtype=torch.int32)
    table = torch.full((3, 251), -1, dtype=torch.int32)
    table[0, :2] = torch.tensor([3, 7])
    table[1, 4] = 1
    table[2, 250] = 11
    for write_kv in (True, False):
        want_k, want_v = torch.zeros(pages, kv_heads, block, dim, dtype=dtype), torch.zeros(pages, kv_heads, vdim, block, dtype=dtype)
        want_q = torch.empty(tokens, heads * dim, dtype=dtype)
        args = dict(q_heads=heads, kv_heads=kv_heads, head_dim=dim, value_dim=vdim, rotary_dim=rot, eps=1e-5, magnitude=1.3, write_kv=write_kv)
        refs.whole_norm_rope_write(qkv, qw, kw, inv_freq, positions, token_seq, table, want_k, want_v, want_q, **args)
        got_k, got_v, got_q = torch.zeros_like(want_k, device=DEV), torch.zeros_like(want_v, device=DEV), torch.empty_like(want_q, device=DEV)
        ops.whole_norm_rope_write(qkv.to(DEV), qw.to(DEV), kw.to(DEV), inv_freq.to(DEV), positions.to(DEV), token_seq.to(DEV), table.to(DEV),
                                  got_k, got_v, got_q, **args)
        # position 1000 turns by up to 1000 radians: float32 angles differ in their last bits
        for got, want in ((got_q, want_q), (got_k, want_k), (got_v, want_v)):
            torch.testing.assert_close(got.float().cpu(), want.float(), rtol=2e-2 if dtype == torch.bfloat16 else 1e-4,
                                       atol=2e-2 if dtype == torch.bfloat16 else 5e-4)
        assert write_kv or not bool(got_k.any())


@pytest.mark.parametrize("heads,kv_heads,dim,vdim", [(4, 2, 16, 24), (8, 2, 128, 128), (2, 2, 12, 20)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_masked_attention_with_cap_and_head_gates(heads, kv_heads, dim, vdim, dtype):
    from forge_engine_amd.kernels import ops
    g = torch.Generator().manual_seed(dim)
    block, pages = 8, 40
    q_lens, ctx = [1, 5, 30, 1], [70, 5, 47, 1]
    tokens = sum(q_lens)
    q = (torch.randn(tokens, heads * dim, generator=g) * 2).to(dtype)
    gate = torch.randn(tokens, heads + 3, generator=g).to(dtype)[:, 2:2 + heads]
    keys = torch.randn(pages, kv_heads, block, dim, generator=g).to(dtype)
    values = torch.randn(pages, kv_heads, vdim, block, generator=g).to(dtype)
    cu_q = torch.tensor([0, 1, 6, 36, 37], dtype=torch.int32)
    ctx_len = torch.tensor(ctx, dtype=torch.int32)
    perm = torch.randperm(pages, generator=g).to(torch.int32)
    table = torch.full((4, 9), -1, dtype=torch.int32)
    at = 0
    for s, n in enumerate(ctx):
        need = -(-n // block)
        table[s, :need] = perm[at:at + need]
        at += need
    args = dict(num_seqs=4, max_q_len=30, q_heads=heads, kv_heads=kv_heads, head_dim=dim, value_dim=vdim, scale=0.9, softcap=2.5,
                head_gate=True)
    want = refs.masked_attention(q, keys, values, torch.empty(tokens, heads * vdim, dtype=dtype), cu_q, ctx_len, table, gate=gate, **args)
    got = ops.masked_attention(q.to(DEV), keys.to(DEV), values.to(DEV), torch.empty(tokens, heads * vdim, dtype=dtype, device=DEV),
                               cu_q.to(DEV), ctx_len.to(DEV), table.to(DEV), gate=gate.to(DEV), num_decode=2, max_ctx=72, **args)
    close(got, want, dtype)


@pytest.mark.parametrize("tokens,hidden,experts,top,inner", [(1, 48, 5, 2, 20), (37, 64, 3, 1, 36), (150, 256, 6, 2, 96), (70, 40, 4, 4, 100), (600, 128, 4, 2, 160)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_mixture_of_experts_kernels(tokens, hidden, experts, top, inner, dtype):
    from forge_engine_amd.kernels import ops
    g = torch.Generator().manual_seed(tokens + experts)
    x = torch.randn(tokens, hidden, generator=g).to(dtype)
    router, bias = (torch.randn(experts, hidden, generator=g) * 0.5).to(dtype), torch.randn(experts, generator=g)
    gate_up = (torch.randn(experts, 2 * inner, hidden, generator=g) * 0.3).to(dtype)
    down = (torch.randn(experts, hidden, inner, generator=g) * 0.2).to(dtype)
    want_chosen, want_weights = refs.moe_route(x, router, bias, top)
    chosen, weights = ops.moe_route(x.to(DEV), router.to(DEV), bias.to(DEV), top)
    assert torch.equal(chosen.cpu(), want_chosen)
    torch.testing.assert_close(weights.cpu(), want_weights, rtol=1e-4, atol=1e-5)
    want = refs.moe_experts(x, want_chosen, want_weights, gate_up, down, torch.empty(top, tokens, hidden), limit=1.2, alpha=1.702)
    got = ops.moe_experts(x.to(DEV), chosen, weights, gate_up.to(DEV), down.to(DEV), torch.empty(top, tokens, hidden, device=DEV),
                          limit=1.2, alpha=1.702)
    close(got, want, dtype)
    for extra in (torch.randn(tokens, hidden, generator=g), torch.randn(3, tokens, hidden, generator=g)):   # what every token gets beside
        want = refs.moe_experts(x, want_chosen, want_weights, gate_up, down, torch.empty(top, tokens, hidden), limit=1.2, alpha=1.702,
                                extra=extra)
        got = ops.moe_experts(x.to(DEV), chosen, weights, gate_up.to(DEV), down.to(DEV), torch.empty(top, tokens, hidden, device=DEV),
                              limit=1.2, alpha=1.702, extra=extra.to(DEV))
        close(got, want, dtype)
    shared = (torch.randn(2 * inner, hidden, generator=g) * 0.3).to(dtype)
    close(ops.linear_gated(x.to(DEV), shared.to(DEV), limit=0.8, alpha=1.702), refs.linear_gated(x, shared, limit=0.8, alpha=1.702), dtype)


# (rows, columns, K, the tile): one of every tile, columns that fill no tile of gate and up rows, K of an odd count of steps
BOUNDED = [(5, 1024, 2048, 9), (8, 2048, 2048, 9), (16, 2047, 1024, 9), (9, 2500, 1024, 10), (16, 1030, 4096, 9), (12, 4100, 1088, 11), (13, 8192, 1024, 12), (9, 9728, 1024, 13),
           (16, 10001, 1088, 13)]


@pytest.mark.parametrize("rows", [17, 90, 361, 500])
def test_bounded_gate_of_more_rows_stands_behind_its_product(rows):
    """Beyond 16 rows, whatever tile the product takes (one of 96 rows among them): the activation is a launch of its own."""
    from forge_engine_amd.kernels import ops
    g = torch.Generator().manual_seed(rows)
    columns, k = 2048, 1024
    assert rows != 361 or ops.LDS_TILES[ops.lds_plan(rows, 2 * columns, k, 4 * columns)[0]][0] == 96
    x = torch.randn(rows, k, generator=g).bfloat16().to(DEV)
    weight = (torch.randn(2 * columns, k, generator=g) * 2 * k ** -0.5).bfloat16().to(DEV)
    got = ops.linear_gated(x, weight, limit=1.5, alpha=1.702)
    both, want = ops.linear(x, weight, ring=False), torch.empty_like(got)
    ops._call("moe", "fe_gated_act", ops._ptr(both), ops._ptr(want), ops.c_int(ops._code(both.dtype)), ops.c_int(rows), ops.c_int(columns),
              ops.c_float(1.5), ops.c_float(1.702), ops._stream())
    assert torch.equal(got, want)


@pytest.mark.parametrize("rows,columns,k,tile", BOUNDED)
def test_bounded_gate_in_its_product(rows, columns, k, tile, monkeypatch):
    """The bits of the product as ``linear`` makes it and a launch of the activation behind it."""
    from forge_engine_amd.kernels import ops
    assert {case[3] for case in BOUNDED} == {9, 10, 11, 12, 13} and ops.lds_plan(rows, 2 * columns, k, 4 * columns)[0] == tile
    g = torch.Generator().manual_seed(rows + columns)
    x = torch.randn(rows, k, generator=g).bfloat16().to(DEV)
    weight = (torch.randn(2 * columns, k, generator=g) * 2 * k ** -0.5).bfloat16().to(DEV)
    calls = []
    real = ops._call
    monkeypatch.setattr(ops, "_call", lambda library, name, *args: (calls.append(name), real(library, name, *args)))
    got = ops.linear_gated(x, weight, limit=1.5, alpha=1.702)
    assert calls == ["fe_gemm_lds_bounded"]
    calls.clear()
    both, want = ops.linear(x, weight, ring=False), torch.empty_like(got)
    ops._call("moe", "fe_gated_act", ops._ptr(both), ops._ptr(want), ops.c_int(ops._code(both.dtype)), ops.c_int(rows), ops.c_int(columns),
              ops.c_float(1.5), ops.c_float(1.702), ops._stream())
    assert calls == ["fe_gemm_wide", "fe_gated_act"] and torch.equal(got, want)


@pytest.mark.parametrize("tile", [9, 10, 11, 12, 13])
@pytest.mark.parametrize("rows,columns,k", [(1, 1, 64), (1, 7, 64), (16, 9, 128), (15, 33, 1024), (2, 130, 832)])
def test_bounded_gate_of_the_smallest_products(rows, columns, k, tile):
    """One row, one step of K, fewer columns than a fragment has, a weight of rows further apart: every tile against the bits of its own
    bfloat16 product and a launch of the activation."""
    from forge_engine_amd.kernels import ops
    g = torch.Generator().manual_seed(rows + columns)
    x = torch.randn(rows, k, generator=g).bfloat16().to(DEV)
    weight = (torch.randn(2 * columns, k + 8, generator=g) * 2 * k ** -0.5).bfloat16().to(DEV)[:, :k]
    c_int, ptr = ops.c_int, ops._ptr
    got = torch.full((rows + 1, columns), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops._call("gemm_wide", "fe_gemm_lds_bounded", ptr(x), ptr(weight), ptr(got), c_int(rows), c_int(columns), c_int(k), ops.c_longlong(weight.stride(0)),
              ops.c_longlong(columns), c_int(tile), ops.c_float(1.5), ops.c_float(1.702), ops._stream())
    both, want = ops.gemm_lds(x, weight, "bf16", tile=tile), torch.empty(rows, columns, dtype=torch.bfloat16, device=DEV)
    ops._call("moe", "fe_gated_act", ptr(both), ptr(want), c_int(ops._code(both.dtype)), c_int(rows), c_int(columns), ops.c_float(1.5), ops.c_float(1.702),
              ops._stream())
    assert torch.equal(got[:rows], want) and bool(got[rows].isnan().all())


# keys in one run, a few, more than sixteen; a gate a head and one an element; rows of q, gate and output of other strides
@pytest.mark.parametrize("form", ["plain", "capped", "sloped", "table", "sink"])
@pytest.mark.parametrize("dim,per_head,contexts", [(128, True, (1, 33, 700, 16)), (64, False, (40, 3, 1, 257, 90)), (128, False, (4000,)), (64, True, (9,) * 20)])
def test_gate_in_the_decode_kernel(dim, per_head, contexts, form, monkeypatch):
    """Single tokens: the bits of the attention and a launch of the gate, in one."""
    from forge_engine_amd.kernels import ops
    n, heads, kv_heads, page = len(contexts), 8, 2, 16
    g = torch.Generator().manual_seed(dim + n)
    pages = [-(-c // page) for c in contexts]
    table = torch.zeros(n, max(pages), dtype=torch.int32)
    order = torch.randperm(sum(pages), generator=g).int()
    for i, count in enumerate(pages):
        table[i, :count] = order[sum(pages[:i]):sum(pages[:i]) + count]
    keys = torch.randn(sum(pages), kv_heads, page, dim, generator=g).bfloat16().to(DEV)
    values = torch.randn(sum(pages), kv_heads, dim, page, generator=g).bfloat16().to(DEV)
    q = torch.randn(n, heads * dim + 64, generator=g).bfloat16().to(DEV)[:, :heads * dim]
    gate = torch.randn(n, heads * (1 if per_head else dim) + 3, generator=g).bfloat16().to(DEV)[:, 3:]
    kinds = {"plain": {}, "capped": {"softcap": 20.0}, "sloped": {"slopes": torch.rand(heads, generator=g).to(DEV) * 0.1},
             "table": {"dist_bias": torch.randn(heads, 50, generator=g).to(DEV)}, "sink": {"sink": torch.randn(heads, generator=g).to(DEV)}}
    where = (torch.arange(n + 1, dtype=torch.int32, device=DEV), torch.tensor(contexts, dtype=torch.int32, device=DEV), table.to(DEV))
    how = dict(num_seqs=n, max_q_len=1, q_heads=heads, kv_heads=kv_heads, head_dim=dim, value_dim=dim, scale=dim ** -0.5, num_decode=n,
               max_ctx=max(contexts), **kinds[form])
    got = torch.empty(n, heads * dim + 2, dtype=torch.bfloat16, device=DEV)[:, :heads * dim]
    calls = []
    real = ops._call
    monkeypatch.setattr(ops, "_call", lambda library, name, *args: (calls.append(name), real(library, name, *args)))
    ops.masked_attention(q, keys, values, got, *where, gate=gate, head_gate=per_head, factor=1.25, **how)
    assert calls == ["fe_paged_attention_decode_gated"]
    apart, want = (torch.empty(n, heads * dim, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    ops.masked_attention(q, keys, values, apart, *where, **how)
    ops._sigmoid_gate(apart, gate, want, heads, dim, dim, per_head, 1.25)
    assert torch.equal(got, want)


def test_gate_of_wide_heads_is_for_a_launch_of_its_own():
    """Heads of 256 have no gated decode kernel: refused before a launch, whatever else the call has."""
    from forge_engine_amd.kernels import ops
    q, pages = torch.zeros(2, 512, dtype=torch.bfloat16, device=DEV), torch.zeros(2, 1, 16, 256, dtype=torch.bfloat16, device=DEV)
    cu, ctx, table = (torch.tensor(v, dtype=torch.int32, device=DEV) for v in ([0, 1, 2], [3, 9], [[0], [1]]))
    how = dict(num_seqs=2, max_q_len=1, q_heads=2, kv_heads=1, head_dim=256, scale=1.0, num_decode=2, max_ctx=9)
    for more in ({}, {"softcap": 5.0}, {"slopes": torch.zeros(2, device=DEV)}):
        with pytest.raises(ops.KernelError, match="heads of 64 and 128"):
            ops.paged_attention(q, pages, pages.transpose(2, 3).contiguous(), torch.empty_like(q), cu, ctx, table, gate=(q, 1, 1.0), **how, **more)


# the smallest, most tokens, experts, pairs and choices, and one of each too many
@pytest.mark.parametrize("scoring,biased", [("softmax", True), ("sigmoid", False)])
@pytest.mark.parametrize("tokens,experts,top", [(1, 1, 1), (8, 8, 2), (64, 64, 4), (16, 17, 16), (64, 3, 3), (65, 8, 2), (8, 65, 2), (33, 64, 8)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_routing_with_its_plan_chooses_as_without(tokens, experts, top, scoring, biased, dtype):
    from forge_engine_amd.kernels import ops
    g = torch.Generator().manual_seed(tokens + experts)
    x, router = torch.randn(tokens, 128, generator=g).to(DEV, dtype), torch.randn(experts, 128, generator=g).to(DEV, dtype)
    router[experts // 2] = router[0]           # equal logits: the lowest index
    bias = torch.randn(experts, generator=g).to(DEV) if biased else None
    chosen, weights = ops.moe_route(x, router, bias, top, scoring)
    none, got_weights, plan = ops.moe_route_plan(x, router, bias, top, scoring)
    assert torch.equal(got_weights, weights)
    if tokens > 64 or experts > 64 or tokens * top > 256:
        assert plan is None and torch.equal(none, chosen)
        return
    flat = chosen.reshape(-1).long()
    counts = torch.bincount(flat, minlength=experts)
    assert none is None and torch.equal(plan[0][1:], torch.cumsum(counts, 0).int()) and int(plan[0][0]) == 0
    assert torch.equal(plan[1], torch.argsort(flat, stable=True).int())


@pytest.mark.parametrize("tokens,hidden,experts,top,inner", [
    (3, 96, 130, 2, 33), (40, 128, 70, 3, 100),                 # more experts than a wave has lanes, few rows each
    (65, 160, 2, 1, 70), (150, 64, 3, 2, 130),                  # 32 to 100 rows an expert
    (190, 224, 2, 2, 129), (300, 96, 1, 1, 260),                # 190 and 300: the wider tiles
    (1030, 192, 4, 1, 34),
    (130, 1440, 3, 1, 2080), (130, 1440, 3, 1, 2083), (130, 1441, 3, 1, 2080),      # blocks enough for 64 x 64
    (300, 1440, 2, 1, 736), (300, 1440, 2, 1, 739), (300, 1441, 2, 1, 736),         # ... for 64 x 128
    (1300, 5152, 4, 1, 1312), (1300, 5152, 4, 1, 1315), (1300, 5153, 4, 1, 1312)])  # ... and steps enough for 256 x 128
@pytest.mark.parametrize("weight_input", [False, True])
def test_grouped_products_tiles(tokens, hidden, experts, top, inner, weight_input):
    """Every tile of the grouped products, rows and columns beside its edges, K ending in half a step, some experts without
    rows: against the same products in 64 bits, with the middle rounded to bfloat16 as the kernels round it."""
    from forge_engine_amd.kernels import ops
    g = torch.Generator(device=DEV).manual_seed(tokens + inner)

    def draw(*shape, scale=1.0):
        return (torch.randn(*shape, generator=g, device=DEV) * scale).bfloat16()

    x, gate_up, down = draw(tokens, hidden), draw(experts, 2 * inner, hidden, scale=hidden ** -0.5), draw(experts, hidden, inner, scale=inner ** -0.5)
    chosen = torch.rand(tokens, experts, generator=g, device=DEV).argsort(1)[:, :top].int()
    if experts > 1:
        chosen[chosen == experts - 1] = 0 if top == 1 else experts - 1      # (one choice a token: the last expert gets nothing)
    weights = torch.rand(tokens, top, generator=g, device=DEV)
    got = ops.moe_experts(x, chosen, weights, gate_up, down, torch.full((top, tokens, hidden), float("nan"), device=DEV), limit=2.0,
                          alpha=1.702, weight_input=weight_input)
    want = torch.zeros(top, tokens, hidden, dtype=torch.float64, device=DEV)
    for k in range(top):
        for e in chosen[:, k].unique().tolist():
            mine = (chosen[:, k] == e).nonzero().flatten()
            both = x[mine].double() @ gate_up[e].double().t()
            w = weights[mine, k, None].double()
            if weight_input:
                both = both * w
            gate, up = both[:, :inner].clamp(max=2.0), both[:, inner:].clamp(-2.0, 2.0)
            act = (gate * torch.sigmoid(1.702 * gate) * (up + 1.0)).float().bfloat16().double()
            want[k, mine] = act @ down[e].double().t() * (1.0 if weight_input else w)
    # the middle may round the other way where a float32 sum lies beside a tie: 2^-8 of one of `inner` terms of size inner^-0.5 each
    torch.testing.assert_close(got.double(), want, atol=2e-2, rtol=1e-3)
    assert float((got.double() - want).norm() / want.norm()) < 1e-3


# blocks for less than all CUs and for just as many, pairs an expert up to a tile's rows and one more, and all but a few with one expert,
# whose tiles then share its weight rows beside experts that are one tile
@pytest.mark.parametrize("tokens,experts,top,hidden,inner,most", [(1, 8, 1, 320, 1024, 1), (1, 8, 1, 320, 8160, 1), (1, 8, 1, 320, 8192, 1), (2, 4, 2, 4096, 288, 2), (64, 4, 2, 1024, 2048, 64),
                                                                  (65, 4, 2, 1024, 2048, 65), (60, 8, 2, 1088, 1024, 60), (250, 8, 2, 1024, 2080, 250)])
def test_grouped_products_whose_weights_pass_the_caches(tokens, experts, top, hidden, inner, most):
    from forge_engine_amd.kernels import ops
    g = torch.Generator(device=DEV).manual_seed(tokens + inner)
    x = torch.randn(tokens, hidden, generator=g, device=DEV).bfloat16()
    gate_up = (torch.randn(experts, 2 * inner, hidden, generator=g, device=DEV) * hidden ** -0.5).bfloat16()
    down = (torch.randn(experts, hidden, inner, generator=g, device=DEV) * inner ** -0.5).bfloat16()
    chosen = torch.zeros(tokens, top, dtype=torch.int32, device=DEV)       # the first expert takes `most` tokens, a second choice goes round
    if top > 1:
        chosen[:, 1] = 1 + torch.arange(tokens, device=DEV).int() % (experts - 1)
    weights = torch.rand(tokens, top, generator=g, device=DEV)
    got = ops.moe_experts(x, chosen, weights, gate_up, down, torch.full((top, tokens, hidden), float("nan"), device=DEV), limit=2.0, alpha=1.702)
    for k in range(top):
        mine = chosen[:, k].long()
        both = torch.stack([x[i].double() @ gate_up[e].double().t() for i, e in enumerate(mine.tolist())])
        gate, up = both[:, :inner].clamp(max=2.0), both[:, inner:].clamp(-2.0, 2.0)
        act = (gate * torch.sigmoid(1.702 * gate) * (up + 1.0)).float().bfloat16().double()
        want = torch.stack([act[i] @ down[e].double().t() for i, e in enumerate(mine.tolist())]) * weights[:, k, None].double()
        torch.testing.assert_close(got[k].double(), want, atol=2e-2, rtol=1e-3)
        assert float((got[k].double() - want).norm() / want.norm()) < 1e-3
    assert int((chosen == 0).sum()) == most


def test_which_tile_a_grouped_product_takes():
    """Both sides of every line: rows an expert, blocks, steps, for the gated product and the other; and that the sizes above
    reach every tile."""
    from forge_engine_amd.kernels import library
    tile = library.load("moe").fe_moe_tile
    for gated, tokens, top, experts, n, k, want in (
            (1, 130, 1, 3, 2080, 1440, 64064), (0, 130, 1, 3, 1440, 2080, 64064), (1, 300, 1, 2, 736, 1440, 64128), (0, 300, 1, 2, 1440, 736, 64128),
            (1, 1300, 1, 4, 1312, 5152, 256128), (0, 1300, 1, 4, 5152, 1312, 256128),
            (1, 32, 1, 1, 65536, 2048, 32064), (1, 33, 1, 1, 65536, 2048, 64064), (1, 96, 1, 1, 65536, 2048, 64064), (1, 97, 1, 1, 65536, 2048, 64128),
            (1, 255, 1, 1, 65536, 2048, 64128), (1, 256, 1, 1, 65536, 2048, 256128), (1, 256, 1, 1, 65536, 2016, 64128), (0, 256, 1, 1, 65536, 736, 64128),
            (0, 256, 1, 1, 65536, 768, 256128), (0, 256, 1, 1, 20352, 768, 64128), (0, 256, 1, 1, 20353, 768, 256128),
            (0, 128, 1, 1, 4096, 768, 64064), (0, 64, 1, 1, 4096, 768, 32064), (0, 64, 1, 1, 4097, 768, 64064), (0, 128, 1, 1, 4097, 768, 64128), (1, 400, 1, 4, 64, 64, 32064)):
        assert tile(gated, tokens, top, experts, n, k) == want, (gated, tokens, top, experts, n, k)


# ------------------------------------------------------------------ the model

@pytest.fixture(scope="module")
def folders(tmp_path_factory):
    return {name: ku.write_model(raw, 31, tmp_path_factory.mktemp(f"rekezen_{name}")) for name, raw in CONFIGS.items()}


@pytest.fixture(scope="module")
def plain_cache():
    return {}


def expected(name, folder, cache, requests):
    key = (name, tuple(sorted((k, tuple(v)) for k, v in requests.items())))
    if key not in cache:
        cache[key] = ku.plain_logits(folder, requests)
    return cache[key]


def requests_of(name, seed, lengths):
    return ru.make_requests({"vocab_size": CONFIGS[name]["vocab"]}, seed, lengths)


TRACES = {
    "whole": ru.trace_whole,
    "tail": lambda r: ru.trace_tail(r, 32),
    "portions": ru.trace_portions,
    "mixed": lambda r: ru.trace_mixed(r, 5, max_live=4),
}


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", list(CONFIGS))
@pytest.mark.parametrize("mode", list(TRACES))
def test_replay_matches_plain(name, mode, dtype, folders, plain_cache, tmp_path):
    requests = requests_of(name, 3, LENGTHS[name])
    trace = TRACES[mode](requests)
    print(f"replay {name} {mode} {dtype}: {len(trace.steps)} steps", flush=True)
    got = ru.run_trace(folders[name], dtype, trace, tmp_path, block_size=BLOCKS[name])
    worst = ku.compare(got, expected(name, folders[name], plain_cache, requests), dtype)
    print(f"  worst difference {worst:.3e}", flush=True)


def sharp(folder, target, factor=6.0):
    """A copy of a model whose attention is sharp (larger norm weights on q, no cap below the scores'
    range), so that one key among hundreds, however far back, moves the logits."""
    import json
    from safetensors.torch import save_file
    raw, weights = ku.folder_weights(folder)
    for index, layer in enumerate(raw["layers"]):
        weights[f"l{index}.mix.q.norm"] = weights[f"l{index}.mix.q.norm"] * factor
        if "softcap" in layer["mixer"]:
            layer["mixer"]["softcap"] = 40.0
    target.mkdir(parents=True, exist_ok=True)
    (target / "config.json").write_text(json.dumps(raw))
    save_file({n: t.contiguous() for n, t in weights.items()}, str(target / "model.safetensors"))
    return target


def test_far_tokens_reach_the_logits(folders, tmp_path):
    """A control on the weights made above: with them, changing the third token of 500 changes the
    last token's logits by more than the float32 bound of these tests."""
    folder = sharp(folders["M"], tmp_path / "sharp")
    cfg, weights = ku.folder_weights(folder)
    tokens = requests_of("M", 8, (500,))["r0"]
    other = list(tokens)
    other[2] = (other[2] + 1) % cfg["vocab"]
    a, b = ku.plain.forward(tokens, weights, cfg)[-1], ku.plain.forward(other, weights, cfg)[-1]
    assert float((a - b).abs().max()) > 1000 * (1e-5 + 1e-4 * float(a.abs().max()))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_long_requests_with_sharp_attention(dtype, folders, tmp_path):
    """Prompts of several hundred tokens whose far keys matter: whole, then the last 40 tokens one by
    one (across page borders), then in portions, then three at once."""
    folder = sharp(folders["M"], tmp_path / "sharp")
    requests = requests_of("M", 9, (500, 333, 129))
    want = ku.plain_logits(folder, requests)
    for mode, trace in (("whole", ru.trace_whole(requests)), ("tail", ru.trace_tail(requests, 40)),
                        ("portions", ru.trace_portions(requests, sizes=(64, 17, 2, 130, 3, 48, 16, 2, 33), want_all=False)),
                        ("mixed", ru.trace_mixed(requests, 11, max_live=3))):
        print(f"sharp {mode} {dtype}: {len(trace.steps)} steps", flush=True)
        got = ru.run_trace(folder, dtype, trace, tmp_path / mode, block_size=16)
        # scores of up to 40 turn an error of one part in 10**7 in a key into one of some parts in 10**5 in a
        # softmax weight: float32 differs from the plain implementation by up to 1e-4 here (the plain
        # implementation in float32 does too); a key left out moves these logits by a hundred times that
        ku.compare(got, want, dtype, fraction=0.1, float32_factor=10.0)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("block_size", [4, 16, 32])
@pytest.mark.parametrize("heads,kv_heads,dim,vdim", [(4, 2, 32, 16), (6, 3, 64, 64), (8, 1, 128, 128)])
def test_one_far_key_among_hundreds_is_found(dtype, block_size, heads, kv_heads, dim, vdim):
    """Keys whose scores dominate sit at the first position, just before and at page borders and hundreds
    of positions back: the attention kernels (matrix cores for heads of 64 and 128 in bfloat16 with pages
    of 16 or more, the vector ALU otherwise) against the plain capped attention, for a prompt's portion
    behind cached keys and for single tokens; with a cap that the dominant scores reach."""
    from forge_engine_amd.kernels import ops
    g = torch.Generator().manual_seed(dim + block_size)
    length, cached = 420, 391          # the portion's 29 tokens lie behind 391 cached ones
    q = torch.randn(length, heads, dim, generator=g)
    k = torch.randn(length, kv_heads, dim, generator=g)
    v = torch.randn(length, kv_heads, vdim, generator=g)
    for far in (0, block_size - 1, block_size, 7 * block_size - 1, 7 * block_size, 200, cached - 1, cached):
        k[far] *= 5.0
    q, k, v = (t.to(dtype) for t in (q, k, v))
    cap, scale = 9.0, 0.3
    want = ku.plain.capped_causal_attention(q.double(), k.double(), v.double(), scale=scale, softcap=cap)
    gates = torch.randn(length, heads, generator=g).to(dtype)
    want = (want * torch.sigmoid(gates.double())[:, :, None]).reshape(length, heads * vdim).float()
    pages = -(-length // block_size)
    perm = torch.randperm(pages + 3, generator=g)[:pages].to(torch.int32)
    key_pages = torch.zeros(pages + 3, kv_heads, block_size, dim, dtype=dtype)
    value_pages = torch.zeros(pages + 3, kv_heads, vdim, block_size, dtype=dtype)
    for p in range(length):
        key_pages[perm[p // block_size], :, p % block_size] = k[p]
        value_pages[perm[p // block_size], :, :, p % block_size] = v[p]
    key_pages, value_pages = key_pages.to(DEV), value_pages.to(DEV)
    table = perm.view(1, -1).to(DEV)
    common = dict(q_heads=heads, kv_heads=kv_heads, head_dim=dim, value_dim=vdim, scale=scale, softcap=cap, head_gate=True)
    # the portion
    out = torch.empty(length - cached, heads * vdim, dtype=dtype, device=DEV)
    ops.masked_attention(q[cached:].reshape(length - cached, -1).to(DEV), key_pages, value_pages, out,
                         torch.tensor([0, length - cached], dtype=torch.int32, device=DEV), torch.tensor([length], dtype=torch.int32, device=DEV),
                         table, num_seqs=1, max_q_len=length - cached, gate=gates[cached:].to(DEV), num_decode=0, max_ctx=length, **common)
    close(out, want[cached:], dtype)
    # single tokens: the same request at eight of its lengths, as eight sequences of one step
    places = [0, block_size - 1, block_size, 7 * block_size, 201, cached - 1, cached, length - 1]
    n = len(places)
    out = torch.empty(n, heads * vdim, dtype=dtype, device=DEV)
    ops.masked_attention(q[places].reshape(n, -1).to(DEV), key_pages, value_pages, out,
                         torch.arange(n + 1, dtype=torch.int32, device=DEV), torch.tensor([p + 1 for p in places], dtype=torch.int32, device=DEV),
                         table.expand(n, -1).contiguous(), num_seqs=n, max_q_len=1, gate=gates[places].to(DEV), num_decode=n,
                         max_ctx=length, **common)
    close(out, want[places], dtype)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_captured_steps_equal_eager_steps_and_long_decoding(dtype, folders):
    """A prompt and then 150 single tokens, two requests side by side: steps replayed from captured graphs
    against the same steps run eagerly, and both against the plain implementation."""
    from forge_engine_amd.engine import ModelRunner, StepEntry, load_model
    _, model = load_model(folders["M"], dtype=dtype, device=DEV)
    requests = requests_of("M", 21, (160, 171))
    want = ku.plain_logits(folders["M"], requests)
    results = {}
    for graphs in (True, False):
        runner = ModelRunner(model, block_size=16, block_capacity=40, num_state_slots=3, use_graphs=graphs, eager_sightings=1)
        got = {}
        for name in requests:
            runner.begin(name)
        at = {"r0": 10, "r1": 21}
        logits = runner.step([StepEntry(n, requests[n][:at[n]], [at[n] - 1]) for n in requests])
        for row, n in zip(logits, requests):
            got[(n, at[n] - 1)] = row.cpu().clone()
        for _ in range(150):
            logits = runner.step([StepEntry(n, [requests[n][at[n]]], [0]) for n in requests])
            for row, n in zip(logits, requests):
                got[(n, at[n])] = row.cpu().clone()
                at[n] += 1
        assert runner.graph_replays >= (140 if graphs else 0) and (graphs or runner.graph_replays == 0)
        results[graphs] = got
        ku.compare(got, want, dtype, fraction=0.1)
    for key, row in results[True].items():
        torch.testing.assert_close(row, results[False][key], rtol=0, atol=0 if dtype == "float32" else 1e-2)


def test_first_tokens_and_slot_reuse(folders):
    """A request that takes over the state slot of one that ended: its first token has no token before
    it, whatever the slot still holds; requests of one and two tokens."""
    from forge_engine_amd.engine import ModelRunner, StepEntry, load_model
    _, model = load_model(folders["A"], dtype="float32", device=DEV)
    runner = ModelRunner(model, block_size=4, block_capacity=16, num_state_slots=1)
    cfg, weights = ku.folder_weights(folders["A"])
    for tokens in ([5, 90, 17, 3], [44], [7, 7], [90, 5, 17, 3, 3, 3, 8, 1, 2]):
        runner.begin("only")
        rows = []
        for token in tokens:          # token by token: every token's predecessor comes from the slot
            rows.append(runner.step([StepEntry("only", [token], [0])])[0].cpu().clone())
        runner.end("only")
        want = ku.plain.forward(tokens, weights, cfg)
        for got, expected in zip(rows, want):
            assert float((got.double() - expected).abs().max()) <= 1e-5 + 1e-4 * float(expected.abs().max())


def test_generation_through_the_entry_point_and_the_command_line(folders):
    import os
    import subprocess
    import sys
    from conftest import ROOT
    from forge_engine_amd.config import SchedulerConfig
    from forge_engine_amd.engine import engine_from_folder
    from forge_engine_amd.sampling import SamplingParams

    cfg, weights = ku.folder_weights(folders["A"])

    def greedy(prompt, count):
        tokens = list(prompt)
        for _ in range(count):
            tokens.append(int(ku.plain.forward(tokens, weights, cfg)[-1].argmax()))
        return tokens[len(prompt):]

    prompts = list(requests_of("A", 13, (11, 3, 25)).values())
    want = [greedy(prompt, 8) for prompt in prompts]
    engine = engine_from_folder(folders["A"], scheduler_config=SchedulerConfig(block_size=4, block_capacity=128, token_budget=16),
                                dtype="float32", eos_token_ids=[])
    ids = [engine.submit(prompt, sampling_params=SamplingParams(max_new_tokens=8)) for prompt in prompts]
    engine.run_until_idle()
    assert [list(engine.request(i).output_token_ids) for i in ids] == want
    command = [sys.executable, str(ROOT / "bin" / "forge-engine"), "generate", "--model", str(folders["A"]), "--dtype", "float32",
               "--max-new-tokens", "8", "--block-size", "4", "--prompt-ids", ",".join(map(str, prompts[0]))]
    done = subprocess.run(command, capture_output=True, text=True, timeout=300, env=dict(os.environ))
    assert done.returncode == 0, done.stderr[-2000:]
    assert ",".join(map(str, want[0])) in done.stdout.replace(" ", "")
