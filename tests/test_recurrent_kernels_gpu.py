"""The kernels of the output-norm layers, the short-convolution attention path and the linear
recurrences, each alone against its plain reference (tests/kernel_refs.py): sizes that are no
multiple of a tile, sequences of unequal length with empty ones between, state slots in any
order, both dtypes."""

from __future__ import annotations

import pytest
import torch

import kernel_refs as refs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from forge_engine_amd.kernels import ops as real_ops
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    return real_ops


def tol(dtype):
    return dict(atol=2e-2, rtol=2e-2) if dtype == torch.bfloat16 else dict(atol=2e-5, rtol=2e-5)


def rand(gen, *shape, dtype=torch.float32, scale=1.0):
    return (torch.randn(*shape, generator=gen) * scale).to(dtype)


def layout(lengths, slots):
    """cu_q, token_seq, state_slots for sequences of the given lengths (0: an empty one)."""
    cu = [0]
    for n in lengths:
        cu.append(cu[-1] + n)
    seq = [i for i, n in enumerate(lengths) for _ in range(n)]
    return (torch.tensor(cu, dtype=torch.int32), torch.tensor(seq, dtype=torch.int32),
            torch.tensor(slots, dtype=torch.int32))


def dev(*tensors):
    return [None if t is None else t.to(DEV) for t in tensors]


LENGTHS = [(5, 0, 1, 19), (1, 1, 1), (70,), (2, 33, 0, 0)]


@pytest.mark.parametrize("x_dtype,out_dtype", [(torch.float32, torch.float32), (torch.float32, torch.bfloat16),
                                               (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("lengths", LENGTHS)
@pytest.mark.parametrize("width,count", [(24, 1), (200, 5), (1030, 2)])
def test_token_shift(ops, x_dtype, out_dtype, lengths, width, count):
    g = torch.Generator().manual_seed(3)
    cu, seq, slots = layout(lengths, [3, 0, 5, 2][:len(lengths)])
    x = rand(g, cu[-1].item(), width, dtype=x_dtype)
    w = torch.rand(count, width, generator=g)
    state = rand(g, 7, width)
    state_ref = state.clone()
    want = refs.token_shift(x, w, state_ref, cu, seq, slots, num_seqs=len(lengths), out_dtype=out_dtype)
    xd, wd, sd, cud, seqd, slotsd = dev(x, w, state, cu, seq, slots)
    got = ops.token_shift(xd, wd, sd, cud, seqd, slotsd, num_seqs=len(lengths), out_dtype=out_dtype)
    torch.testing.assert_close(got.cpu().float(), want.float(), **tol(out_dtype))
    torch.testing.assert_close(sd.cpu(), state_ref, atol=0, rtol=0)


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("parts", [1, 4, 5])
@pytest.mark.parametrize("rows,width", [(1, 24), (3, 256), (6, 1024), (6, 2048), (7, 2049), (512, 4097), (300, 2048), (2, 8192)])
def test_update_and_shift_in_one_launch(ops, out_dtype, parts, rows, width):
    """Every count of elements a thread holds, tokens in another order than their sequences, and a token without a slot of its own: the
    bits of the norm of the update and the token shift behind it."""
    g = torch.Generator().manual_seed(rows + width)
    h, update, w = rand(g, rows, width).to(DEV), rand(g, parts, rows, width).to(DEV), (1.0 + rand(g, width, scale=0.1)).to(DEV)
    shift, state = torch.rand(1, width, generator=g).to(DEV), rand(g, rows + 3, width).to(DEV)
    seq = torch.arange(rows, dtype=torch.int32, device=DEV)
    slots = (1 + torch.randperm(rows + 1, generator=g)[:rows]).int().to(DEV)      # the first and the last row are nobody's
    if rows > 2:
        slots[1] = rows + 9
    want_h, want_state = h.clone(), state.clone()
    ops.rmsnorm_update(want_h, update, w, 1e-6, None)
    want = ops.token_shift(want_h, shift, want_state, torch.arange(rows + 1, dtype=torch.int32, device=DEV), seq, slots, num_seqs=rows, out_dtype=out_dtype)
    got = ops.rmsnorm_update_shift(h, update, w, 1e-6, shift, state, seq, slots, out_dtype=out_dtype)
    assert torch.equal(got, want) and torch.equal(h, want_h) and torch.equal(state, want_state)
    with pytest.raises(ops.KernelError):
        ops.rmsnorm_update_shift(h[:, :width - 1].contiguous(), update, w, 1e-6, shift, state, seq, slots, out_dtype=out_dtype)


@pytest.mark.parametrize("rows,n,k,launches", [(1, 64, 2048, 1), (6, 64, 2048, 1), (16, 2050, 1024, 1), (17, 64, 2048, 2), (3, 40, 72, 2)])
def test_product_with_its_tanh(ops, rows, n, k, launches, monkeypatch):
    """In the product's launch or behind it: the same bits."""
    g = torch.Generator().manual_seed(rows + n)
    x, w = rand(g, rows, k, dtype=torch.bfloat16).to(DEV), rand(g, n, k, dtype=torch.bfloat16, scale=0.1).to(DEV)
    x[0, :8] = torch.tensor([float("nan"), 3e38, 1.0, -1.0, 0.0, 1e-30, -1e-3, 2.0]).bfloat16().to(DEV) if rows > 1 else x[0, :8]
    want = ops.tanh_rows(ops.linear(x, w))
    calls = []
    real = ops._call
    monkeypatch.setattr(ops, "_call", lambda library, name, *args: (calls.append(name), real(library, name, *args)))
    got = ops.linear_tanh(x, w)
    assert calls == ["fe_gemm_ring"] if launches == 1 else (len(calls) == 2 and calls[0] != "fe_gemm_ring" and calls[1] != "fe_gemm_ring")
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(9.0), want.nan_to_num(9.0))


@pytest.mark.parametrize("out_dtype", [None, torch.float32, torch.bfloat16])
@pytest.mark.parametrize("parts", [0, 3])
@pytest.mark.parametrize("rows,width", [(7, 24), (33, 200), (300, 2050)])
def test_rmsnorm_update(ops, out_dtype, parts, rows, width):
    g = torch.Generator().manual_seed(4)
    h = rand(g, rows, width, scale=2.0)
    update = rand(g, *((parts,) if parts else ()), rows, width, scale=5.0)
    w = 1.0 + rand(g, width, scale=0.1)
    h_ref = h.clone()
    out_ref = None if out_dtype is None else torch.empty(rows, width, dtype=out_dtype)
    refs.rmsnorm_update(h_ref, update, w, 1e-6, out_ref)
    hd, ud, wd = dev(h, update, w)
    out = None if out_dtype is None else torch.empty(rows, width, dtype=out_dtype, device=DEV)
    ops.rmsnorm_update(hd, ud, wd, 1e-6, out)
    torch.testing.assert_close(hd.cpu(), h_ref, atol=2e-5, rtol=2e-5)
    if out is not None:
        torch.testing.assert_close(out.cpu().float(), out_ref.float(), **tol(out_dtype))


@pytest.mark.parametrize("rows,width", [(2, 256), (513, 257), (513, 513), (6, 1024), (6, 1025), (513, 1025), (6, 2049), (6, 4097), (600, 2049), (6, 8192), (6, 8193)])
@pytest.mark.parametrize("parts", [1, 4, 5, 9])
def test_rows_held_in_registers(ops, rows, width, parts):
    """Both sides of every count of elements a thread holds (256 and 1,024 threads a row), parts that fill no round of four; NaN
    beside the last element stays in its row."""
    g = torch.Generator().manual_seed(width + parts)
    h, update, w = rand(g, rows, width, scale=2.0), rand(g, parts, rows, width), 1.0 + rand(g, width, scale=0.1)
    update[0, rows - 1, width - 1] = float("nan")
    h_ref, hd = h.clone(), h.to(DEV)
    refs.rmsnorm_update(h_ref, update, w, 1e-6, None)
    ops.rmsnorm_update(hd, update.to(DEV), w.to(DEV), 1e-6, None)
    torch.testing.assert_close(hd.cpu(), h_ref, atol=2e-5, rtol=2e-5, equal_nan=True)
    if parts > 1:
        many = [update[:, : rows - 1].contiguous(), update[:2, : rows - 1].contiguous()] * 2
        weights = 1.0 + rand(g, 4, width, scale=0.1)
        want = refs.rmsnorm_mean(many, weights, 1e-6, torch.empty(rows - 1, width))
        torch.testing.assert_close(ops.rmsnorm_mean(dev(*many), weights.to(DEV), 1e-6, torch.empty(rows - 1, width, device=DEV)).cpu(), want,
                                   atol=2e-5, rtol=2e-5)
    coeff = torch.tensor([0.7, -0.4, 0.25, 0.1])
    for dtype in (torch.float32, torch.bfloat16):
        z = update[0].to(dtype)
        want = refs.polynorm(z, coeff, 1e-6, torch.empty_like(z))
        torch.testing.assert_close(ops.polynorm(z.to(DEV), coeff.to(DEV), 1e-6, torch.empty_like(z, device=DEV)).cpu().float(), want.float(),
                                   **tol(dtype), equal_nan=True)


@pytest.mark.parametrize("count", [1, 2, 4])
@pytest.mark.parametrize("rows,width", [(5, 40), (129, 1000)])
def test_rmsnorm_mean(ops, count, rows, width):
    g = torch.Generator().manual_seed(5)
    updates = [rand(g, *((2,) if i == 1 else ()), rows, width, scale=float(i + 1)) for i in range(count)]
    w = 1.0 + rand(g, count, width, scale=0.2)
    want = refs.rmsnorm_mean(updates, w, 1e-5, torch.empty(rows, width))
    got = ops.rmsnorm_mean(dev(*updates), w.to(DEV), 1e-5, torch.empty(rows, width, device=DEV))
    torch.testing.assert_close(got.cpu(), want, atol=2e-5, rtol=2e-5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,width", [(3, 20), (65, 320), (10, 5000)])
def test_polynorm(ops, dtype, rows, width):
    g = torch.Generator().manual_seed(6)
    z = rand(g, rows, width, dtype=dtype, scale=1.5)
    coeff = torch.tensor([0.7, -0.4, 0.25, 0.1])
    want = refs.polynorm(z, coeff, 1e-6, torch.empty_like(z))
    got = ops.polynorm(z.to(DEV), coeff.to(DEV), 1e-6, torch.empty_like(z, device=DEV))
    torch.testing.assert_close(got.cpu().float(), want.float(), **tol(dtype))
    for shape in ((9, 40), (3, 9, 40)):
        update, row_bias = rand(g, *shape), rand(g, 40)
        torch.testing.assert_close(ops.add_bias(update.to(DEV), row_bias.to(DEV)).cpu(), refs.add_bias(update.clone(), row_bias))
    x = rand(g, 1000, dtype=dtype, scale=2.0)
    torch.testing.assert_close(ops.tanh_rows(x.to(DEV)).cpu().float(), refs.tanh_rows(x.clone()).float(), **tol(dtype))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads,dim,shared,act,extra", [(4, 32, False, "silu", 0), (3, 64, True, "silu", 0),
                                                        (2, 100, False, "sigmoid", 1), (5, 24, False, "none", 0)])
def test_head_norm_gate(ops, dtype, heads, dim, shared, act, extra):
    g = torch.Generator().manual_seed(7)
    tokens = 37
    o = rand(g, tokens, heads, dim + extra, scale=3.0)
    weight = 1.0 + rand(g, dim if shared else heads * dim, scale=0.2)
    wide = rand(g, tokens, heads * dim + 9, dtype=dtype)
    gate = None if act == "none" else wide[:, 9:]
    floor = torch.rand(tokens, heads, generator=g) * 4.0 if extra else None
    want = refs.head_norm_gate(o, weight, gate, torch.empty(tokens, heads * dim, dtype=dtype), heads=heads, dim=dim, eps=1e-6,
                               act=act, extra=extra, floor=floor)
    wide_d = wide.to(DEV)
    got = ops.head_norm_gate(o.to(DEV), weight.to(DEV), None if gate is None else wide_d[:, 9:],
                             torch.empty(tokens, heads * dim, dtype=dtype, device=DEV), heads=heads, dim=dim, eps=1e-6,
                             act=act, extra=extra, floor=None if floor is None else floor.to(DEV))
    torch.testing.assert_close(got.cpu().float(), want.float(), **tol(dtype))


def attention_case(g, dtype, lengths, before, *, q_heads, kv_heads, head_dim, value_dim, block_size):
    """Pages, tables and lengths for sequences that hold ``before[i]`` tokens and bring ``lengths[i]``."""
    ctx = [b + n for b, n in zip(before, lengths)]
    width = max(1, max(-(-c // block_size) for c in ctx))
    pages = sum(-(-c // block_size) for c in ctx) + 3
    order = torch.randperm(pages, generator=g).tolist()
    table = torch.full((len(lengths), width), -1, dtype=torch.int32)
    for i, c in enumerate(ctx):
        for b in range(-(-c // block_size)):
            table[i, b] = order.pop()
    keys = rand(g, pages, kv_heads, block_size, head_dim, dtype=dtype)
    values = rand(g, pages, kv_heads, value_dim, block_size, dtype=dtype)
    return torch.tensor(ctx, dtype=torch.int32), table, keys, values


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("sizes", [
    dict(q_heads=6, kv_heads=3, head_dim=64, value_dim=64, block_size=16, taps=3, rotary_dim=32),
    dict(q_heads=3, kv_heads=3, head_dim=24, value_dim=40, block_size=4, taps=2, rotary_dim=12),
    dict(q_heads=6, kv_heads=2, head_dim=128, value_dim=32, block_size=8, taps=0, rotary_dim=0),
    dict(q_heads=2, kv_heads=1, head_dim=256, value_dim=72, block_size=16, taps=1, rotary_dim=2),
])
def test_conv_rope_norm_write(ops, dtype, sizes):
    g = torch.Generator().manual_seed(8)
    lengths, before = [5, 0, 1, 2, 30], [0, 7, 9, 14, 3]
    taps, rotary_dim = sizes["taps"], sizes["rotary_dim"]
    geometry = {k: sizes[k] for k in ("q_heads", "kv_heads", "head_dim", "value_dim")}
    cu, seq, slots = layout(lengths, [2, 4, 0, 1, 3])
    ctx, table, keys, values = attention_case(g, dtype, lengths, before, block_size=sizes["block_size"], **geometry)
    tokens = sum(lengths)
    positions = torch.tensor([b + i for b, n in zip(before, lengths) for i in range(n)], dtype=torch.int32)
    channels = (sizes["q_heads"] + sizes["kv_heads"]) * sizes["head_dim"] + sizes["kv_heads"] * sizes["value_dim"]
    wide = rand(g, tokens, channels + 17, dtype=dtype)
    qkv = wide[:, :channels]
    bias = rand(g, channels) if sizes["value_dim"] != 32 else None
    conv_w = rand(g, channels, taps) if taps else None
    state = rand(g, 6, taps - 1, channels) if taps > 1 else None
    inv_freq = (1.0 / 10000.0 ** (torch.arange(0, rotary_dim, 2).float() / rotary_dim)) if rotary_dim else None
    state_ref = None if state is None else state.clone()
    keys_ref, values_ref = keys.clone(), values.clone()
    q_ref = torch.empty(tokens, sizes["q_heads"] * sizes["head_dim"], dtype=dtype)
    refs.conv_rope_norm_write(qkv, bias, conv_w, state_ref, inv_freq, positions, seq, cu, slots, table, keys_ref, values_ref, q_ref,
                              num_seqs=len(lengths), rotary_dim=rotary_dim, unit_norm_eps=1e-6, taps=taps, **geometry)
    wide_d, conv_d, state_d, freq_d, pos_d, seq_d, cu_d, slots_d, table_d, keys_d, values_d = dev(
        wide, conv_w, state, inv_freq, positions, seq, cu, slots, table, keys, values)
    q_d = torch.empty_like(q_ref, device=DEV)
    ops.conv_rope_norm_write(wide_d[:, :channels], None if bias is None else bias.to(DEV), conv_d, state_d, freq_d, pos_d, seq_d, cu_d, slots_d, table_d, keys_d,
                             values_d, q_d, num_seqs=len(lengths), rotary_dim=rotary_dim, unit_norm_eps=1e-6, taps=taps,
                             **geometry)
    torch.testing.assert_close(q_d.cpu().float(), q_ref.float(), **tol(dtype))
    torch.testing.assert_close(keys_d.cpu().float(), keys_ref.float(), **tol(dtype))
    torch.testing.assert_close(values_d.cpu().float(), values_ref.float(), **tol(dtype))
    if taps > 1:
        torch.testing.assert_close(state_d.cpu(), state_ref, atol=0, rtol=0)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("taps", [2, 4, 8])
def test_convolution_state_of_single_tokens(ops, dtype, taps):
    """Moved on by the launch that reads it, or by one of its own: the same bits everywhere; a slot that is no slot stays out of it."""
    g = torch.Generator().manual_seed(taps)
    seqs, geometry = 5, dict(q_heads=6, kv_heads=2, head_dim=72, value_dim=40)
    cu, seq, slots = layout([1] * seqs, [2, 4, 0, 9, 3])
    ctx, table, keys, values = attention_case(g, dtype, [1] * seqs, [0, 7, 9, 14, 3], block_size=8, **geometry)
    channels = 8 * 72 + 2 * 40
    qkv, bias, conv_w, state = rand(g, seqs, channels, dtype=dtype), rand(g, channels), rand(g, channels, taps), rand(g, 6, taps - 1, channels)
    inv_freq = 1.0 / 10000.0 ** (torch.arange(0, 32, 2).float() / 32)
    found = []
    for single in (False, True):
        held = dev(qkv, bias, conv_w, state, inv_freq, torch.tensor([0, 7, 9, 14, 3], dtype=torch.int32), seq, cu, slots, table, keys, values)
        q = torch.empty(seqs, 6 * 72, dtype=dtype, device=DEV)
        ops.conv_rope_norm_write(*held, q, num_seqs=seqs, rotary_dim=32, unit_norm_eps=1e-6, taps=taps, single=single, **geometry)
        found.append((q, held[3], held[10], held[11]))
    assert all(torch.equal(a, b) for a, b in zip(*found))
    with pytest.raises(ops.KernelError):
        ops.conv_rope_norm_write(*held, q, num_seqs=seqs - 1, rotary_dim=32, unit_norm_eps=1e-6, taps=taps, single=True, **geometry)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("sizes", [
    dict(q_heads=8, kv_heads=2, head_dim=64, value_dim=64, block_size=16, chunk=24, window=None, sink=True, gate=True),
    dict(q_heads=6, kv_heads=2, head_dim=128, value_dim=128, block_size=32, chunk=33, window=None, sink=True, gate=True),
    dict(q_heads=3, kv_heads=3, head_dim=24, value_dim=40, block_size=4, chunk=7, window=None, sink=True, gate=False),
    dict(q_heads=6, kv_heads=1, head_dim=128, value_dim=16, block_size=8, chunk=None, window=11, sink=False, gate=True),
    dict(q_heads=2, kv_heads=2, head_dim=200, value_dim=130, block_size=16, chunk=1000, window=None, sink=True, gate=False),
])
def test_masked_attention(ops, dtype, sizes):
    g = torch.Generator().manual_seed(9)
    lengths, before = [5, 0, 1, 1, 40], [0, 7, 48, 23, 30]
    geometry = {k: sizes[k] for k in ("q_heads", "kv_heads", "head_dim", "value_dim")}
    cu, _, _ = layout(lengths, [0] * len(lengths))
    ctx, table, keys, values = attention_case(g, dtype, lengths, before, block_size=sizes["block_size"], **geometry)
    tokens = sum(lengths)
    q = rand(g, tokens, sizes["q_heads"] * sizes["head_dim"], dtype=dtype)
    wide = rand(g, tokens, sizes["q_heads"] * sizes["value_dim"] + 5, dtype=dtype)
    sink = rand(g, sizes["q_heads"], scale=2.0) if sizes["sink"] else None
    options = dict(num_seqs=len(lengths), max_q_len=max(lengths), scale=sizes["head_dim"] ** -0.5 * 3.0,
                   window=sizes["window"], chunk=sizes["chunk"], **geometry)
    want = refs.masked_attention(q, keys, values, torch.zeros(tokens, sizes["q_heads"] * sizes["value_dim"], dtype=dtype), cu, ctx,
                                 table, sink=sink, gate=wide[:, 5:] if sizes["gate"] else None, **options)
    q_d, keys_d, values_d, cu_d, ctx_d, table_d, sink_d, wide_d = dev(q, keys, values, cu, ctx, table, sink, wide)
    got = ops.masked_attention(q_d, keys_d, values_d, torch.zeros_like(want, device=DEV), cu_d, ctx_d, table_d, sink=sink_d,
                               gate=wide_d[:, 5:] if sizes["gate"] else None, **options)
    torch.testing.assert_close(got.cpu().float(), want.float(), **tol(dtype))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("form", ["rwkv", "gla", "mlstm", "plain"])
@pytest.mark.parametrize("heads,key_dim,value_dim", [(5, 32, 32), (2, 48, 80), (3, 20, 50), (1, 128, 16), (2, 200, 24), (3, 64, 40), (2, 136, 9)])
def test_linear_recurrence(ops, dtype, form, heads, key_dim, value_dim):
    g = torch.Generator().manual_seed(10)
    lengths = [5, 0, 1, 37, 2]
    cu, _, slots = layout(lengths, [4, 1, 0, 2, 5])
    tokens = sum(lengths)
    wide = rand(g, tokens, 2 * heads * key_dim + heads * value_dim + 3, dtype=dtype)
    q, k = wide[:, 3:3 + heads * key_dim], wide[:, 3 + heads * key_dim:3 + 2 * heads * key_dim]
    v = wide[:, 3 + 2 * heads * key_dim:]
    ones = form == "mlstm"
    columns = value_dim + (1 if ones else 0)
    state = rand(g, 7, heads, columns, key_dim)
    options = dict(num_seqs=len(lengths), max_q_len=max(lengths), heads=heads, key_dim=key_dim, value_dim=value_dim)
    extra = {}
    if form == "rwkv":
        extra = dict(decay=rand(g, tokens, heads * key_dim), decay_kind="exp_neg_exp", decay_bias=rand(g, heads * key_dim) - 1.0,
                     bonus=rand(g, heads, key_dim))
    elif form == "gla":
        extra = dict(decay=rand(g, tokens, heads * key_dim, scale=2.0), decay_kind="sigmoid_root",
                     decay_bias=rand(g, heads * key_dim), tau=7.0, q_scale=key_dim ** -0.5)
    elif form == "mlstm":
        extra = dict(head_decay=torch.rand(tokens, heads, generator=g), in_scale=torch.rand(tokens, heads, generator=g),
                     q_scale=key_dim ** -0.5, ones_column=True)
    state_ref = state.clone()
    want = refs.linear_recurrence(q, k, v, torch.zeros(tokens, heads, columns), state_ref, cu, slots, **options, **extra)
    wide_d, state_d, cu_d, slots_d = dev(wide, state, cu, slots)
    extra_d = {n: (t.to(DEV) if isinstance(t, torch.Tensor) else t) for n, t in extra.items()}
    got = ops.linear_recurrence(wide_d[:, 3:3 + heads * key_dim], wide_d[:, 3 + heads * key_dim:3 + 2 * heads * key_dim],
                                wide_d[:, 3 + 2 * heads * key_dim:], torch.zeros(tokens, heads, columns, device=DEV), state_d,
                                cu_d, slots_d, **options, **extra_d)
    torch.testing.assert_close(got.cpu(), want, atol=1e-4, rtol=1e-4)
    torch.testing.assert_close(state_d.cpu(), state_ref, atol=1e-4, rtol=1e-4)


# one and several passes of a block's columns, key sizes that leave lanes of a column without channels, the smallest and largest heads
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("form", ["rwkv", "gla", "mlstm", "plain"])
@pytest.mark.parametrize("heads,key_dim,value_dim", [(3, 64, 64), (2, 64, 128), (2, 128, 256), (5, 4, 1), (2, 48, 80), (2, 20, 50), (1, 128, 16),
                                                     (2, 200, 24), (1, 256, 512), (2, 32, 511)])
def test_linear_recurrence_step(ops, dtype, form, heads, key_dim, value_dim):
    g = torch.Generator().manual_seed(12)
    cu, _, slots = layout([1] * 4, [4, 1, 0, 5])
    tokens, keys, values = 4, heads * key_dim, heads * value_dim
    wide = rand(g, tokens, 2 * keys + 2 * values + 3, dtype=dtype)
    cut = lambda t: (t[:, 3:3 + keys], t[:, 3 + keys:3 + 2 * keys], t[:, 3 + 2 * keys:3 + 2 * keys + values], t[:, 3 + 2 * keys + values:])
    columns = value_dim + (1 if form == "mlstm" else 0)
    state, maximum = rand(g, 7, heads, columns, key_dim), rand(g, 7, heads, scale=2.0)
    tensors = {"weight": rand(g, value_dim if form == "gla" else values)}
    numbers = dict(num_seqs=tokens, heads=heads, key_dim=key_dim, value_dim=value_dim, eps=1e-6, act="sigmoid" if form == "mlstm" else "silu")
    if form == "rwkv":
        tensors.update(decay=rand(g, tokens, keys), decay_bias=rand(g, keys) - 1.0, bonus=rand(g, heads, key_dim))
        numbers.update(decay_kind="exp_neg_exp")
    elif form == "gla":
        tensors.update(decay=rand(g, tokens, keys, scale=2.0), decay_bias=rand(g, keys))
        numbers.update(decay_kind="sigmoid_root", tau=7.0, q_scale=key_dim ** -0.5)
    elif form == "mlstm":
        tensors.update(gates=rand(g, tokens, 2 * heads, scale=6.0), gate_bias=rand(g, 2 * heads), maximum=maximum)
        numbers.update(cap=12.0, q_scale=key_dim ** -0.5)
    state_d, wide_d, cu_d, slots_d = dev(state, wide, cu, slots)
    tensors_d = {n: t.to(DEV) for n, t in tensors.items()}
    got = ops.linear_recurrence_step(*cut(wide_d), torch.zeros(tokens, values + 5, dtype=dtype, device=DEV)[:, 5:], state_d, cu_d, slots_d,
                                     **tensors_d, **numbers)
    want = refs.linear_recurrence_step(*cut(wide), torch.zeros(tokens, values, dtype=dtype), state, cu, slots, **tensors, **numbers)
    torch.testing.assert_close(got.cpu().float(), want.float(), **tol(dtype))
    torch.testing.assert_close(state_d.cpu(), state, atol=1e-4, rtol=1e-4)
    if form == "mlstm":
        torch.testing.assert_close(tensors_d["maximum"].cpu(), maximum, atol=1e-5, rtol=1e-5)


# chunks of 16 tokens whole and not, columns that fill no block, columns of 32 lanes and (few of them) of 64
@pytest.mark.parametrize("lengths", [[40] * 10 + [0, 1], [400, 1, 5]])
@pytest.mark.parametrize("form", ["plain", "mlstm", "rwkv"])
@pytest.mark.parametrize("key_dim,value_dim", [(128, 256), (96, 250), (65, 251), (128, 32), (100, 30), (65, 33)])
def test_linear_recurrence_of_many_and_few_walks(ops, lengths, form, key_dim, value_dim):
    g = torch.Generator().manual_seed(13)
    heads, tokens, ones = 2, sum(lengths), form == "mlstm"
    cu, _, slots = layout(lengths, list(range(len(lengths))))
    q, k, v = (rand(g, tokens, heads * n) for n in (key_dim, key_dim, value_dim))
    state = rand(g, len(lengths) + 1, heads, value_dim + ones, key_dim)
    options = dict(num_seqs=len(lengths), max_q_len=max(lengths), heads=heads, key_dim=key_dim, value_dim=value_dim, q_scale=key_dim ** -0.5,
                   ones_column=ones)
    extra = dict(head_decay=torch.rand(tokens, heads, generator=g), in_scale=torch.rand(tokens, heads, generator=g))
    if form == "rwkv":
        extra = dict(decay=rand(g, tokens, heads * key_dim), decay_kind="exp_neg_exp", decay_bias=rand(g, heads * key_dim) - 1.0,
                     bonus=rand(g, heads, key_dim))
    state_d, cu_d, slots_d = dev(state, cu, slots)
    extra_d = {n: (t.to(DEV) if isinstance(t, torch.Tensor) else t) for n, t in extra.items()}
    got = ops.linear_recurrence(q.to(DEV), k.to(DEV), v.to(DEV), torch.zeros(tokens, heads, value_dim + ones, device=DEV), state_d, cu_d, slots_d,
                                **options, **extra_d)
    want = refs.linear_recurrence(q, k, v, torch.zeros(tokens, heads, value_dim + ones), state, cu, slots, **options, **extra)
    torch.testing.assert_close(got.cpu(), want, atol=1e-4, rtol=1e-4)
    torch.testing.assert_close(state_d.cpu(), state, atol=1e-4, rtol=1e-4)


@pytest.mark.parametrize("heads", [1, 2, 5])
def test_mlstm_gate_scan(ops, heads):
    g = torch.Generator().manual_seed(11)
    lengths = [5, 0, 1, 150, 64]
    cu, _, slots = layout(lengths, [4, 1, 0, 2, 5])
    tokens = sum(lengths)
    gates = rand(g, tokens, 2 * heads, scale=6.0)
    bias = rand(g, 2 * heads)
    maximum = rand(g, 6, heads, scale=2.0)
    maximum_ref = maximum.clone()
    want = refs.mlstm_gate_scan(gates, bias, 12.0, maximum_ref, cu, slots, torch.zeros(3, tokens, heads), num_seqs=len(lengths), heads=heads)
    gates_d, bias_d, maximum_d, cu_d, slots_d = dev(gates, bias, maximum, cu, slots)
    got = ops.mlstm_gate_scan(gates_d, bias_d, 12.0, maximum_d, cu_d, slots_d, torch.zeros(3, tokens, heads, device=DEV),
                              num_seqs=len(lengths), heads=heads)
    torch.testing.assert_close(got.cpu(), want, atol=1e-5, rtol=1e-4)
    torch.testing.assert_close(maximum_d.cpu(), maximum_ref, atol=1e-5, rtol=1e-5)


@pytest.mark.parametrize("together", [True, False])
def test_a_requests_states_from_zero(ops, together):
    """Rows of one word, of words that end no 16-byte piece and start on none, of more pieces than a launch has threads; with a row of
    an odd number of bytes among them, one by one."""
    states = [torch.ones(5, device=DEV, dtype=torch.int32), torch.ones(5, 3, 7, device=DEV), torch.ones(5, 8, 129, 128, device=DEV),
              torch.ones(5, 600, 4000, device=DEV), torch.ones(5, 6, device=DEV, dtype=torch.bfloat16)]
    if not together:
        states.append(torch.ones(5, 3, device=DEV, dtype=torch.bfloat16))
    slots = ops.SlotStates(states)
    assert slots.together == together
    for slot in (4, 0):
        slots.zero(slot)
    for state in states:
        assert not state[[0, 4]].any() and bool((state[1:4] == 1).all())
    for slot in (-1, 5):
        with pytest.raises(ops.KernelError):
            slots.zero(slot)
