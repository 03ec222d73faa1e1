"""Mazanex through the engine on the CPU, with the kernels' plain references patched in, against
the plain implementation (tests/plain_mazanex.py): configuration and tensor names, each mixer
alone, and that logits do not depend on how requests are cut into steps, batched, or placed in
pages and state slots.  The kernels themselves run in the GPU tests."""

from __future__ import annotations

import pytest
import torch

import kernel_refs
import mazanex_util as mu
import replay_util as ru
from forge_engine_amd.config import ConfigError, SchedulerConfig, load_model_config
from forge_engine_amd.engine import ModelRunner, StepEntry, build_engine, load_model
from forge_engine_amd.sampling import SamplingParams
from forge_engine_amd.weights.random_init import declared_tensors

CONFIGS = {"A": mu.MIXED_A, "B": mu.MIXED_B}
LENGTHS = {"A": (5, 1, 14, 27), "B": (2, 9, 21, 33)}


@pytest.fixture(scope="module")
def folders(tmp_path_factory):
    made = {name: mu.write_model(raw, 7, tmp_path_factory.mktemp(f"mazanex_{name}")) for name, raw in CONFIGS.items()}
    for name, raw in mu.ALONE.items():
        made[name] = mu.write_model(raw, 8, tmp_path_factory.mktemp(f"alone_{name}"))
    return made


def requests_of(name, seed, lengths):
    return ru.make_requests({"vocab_size": CONFIGS.get(name, mu.ALONE.get(name))["vocab"]}, seed, lengths)


def test_configuration_names_and_shapes():
    config = load_model_config(mu.MIXED_A)
    assert config.architecture == "Mazanex" and load_model_config(config.to_dict()) == config
    tensors = declared_tensors(config)
    for name, shape in {"embed": (96, 48), "head": (96, 48), "final.norm": (48,), "l0.shift": (48,), "l0.norm1": (48,),
                        "l0.norm2": (48,), "l0.mix.left.q": (64, 48), "l0.mix.left.q.b": (64,), "l0.mix.left.k.conv": (32, 3),
                        "l0.mix.left.v": (16, 48), "l0.mix.left.sink": (4,), "l0.mix.left.g": (32, 48), "l0.mix.left.o": (48, 32),
                        "l0.mix.left.o.b": (48,), "l0.mix.left.out": (48,), "l0.mix.right.out": (48,), "l0.mix.right.mu.w": (48,),
                        "l0.mix.right.w1": (5, 48), "l0.mix.right.w2": (48, 5), "l0.mix.right.u": (3, 16), "l0.mix.right.norm": (48,),
                        "l1.mix.a1": (5, 48), "l1.mix.a2.b": (16,), "l1.mix.norm": (24,), "l1.mix.v": (48, 48),
                        "l2.mix.i": (3, 48), "l2.mix.f.b": (3,), "l2.mix.norm": (48,), "l2.mlp.act": (4,), "l2.mlp.up": (56, 48)}.items():
        assert tuple(tensors[name].shape) == shape, name
    assert "l1.norm2" not in tensors and not any(n.startswith("l1.mlp") for n in tensors)     # a layer without a feed-forward
    for broken in ({**mu.MIXED_A, "layers": []}, {**mu.MIXED_A, "layers": [mu.layer("conv", {}, None)]},
                   {**mu.MIXED_A, "layers": [mu.layer("parallel", {"left": mu.attention(3, 2, 8, 8, 2, 4, 8), "right": {"heads": 1, "dim": 8}}, None)]},
                   {k: v for k, v in mu.MIXED_A.items() if k != "norm"}):
        with pytest.raises(ConfigError):
            load_model_config(broken)


def test_decay_ranks_come_from_the_checkpoint(folders, tmp_path, monkeypatch):
    """The inner size of a low-rank decay projection is nowhere in config.json: a folder whose
    config lacks the optional key loads by the tensors' shapes."""
    import json
    import shutil
    kernel_refs.install(monkeypatch)
    folder = shutil.copytree(folders["A"], tmp_path / "copy")
    raw = json.loads((folder / "config.json").read_text())
    del raw["layers"][0]["mixer"]["right"]["rank"], raw["layers"][1]["mixer"]["rank"]
    (folder / "config.json").write_text(json.dumps(raw))
    _, model = load_model(folder, dtype="float32", device="cpu")
    assert model.layers[1].mixer.decay_rank == 5 and model.layers[0].mixer.branches["right"].decay_rank == 5


@pytest.mark.parametrize("name", list(mu.ALONE))
def test_each_mixer_alone(name, folders, tmp_path, monkeypatch):
    kernel_refs.install(monkeypatch)
    requests = requests_of(name, 2, (19, 1))
    got = ru.run_trace(folders[name], "float32", ru.trace_whole(requests), tmp_path, block_size=4, device="cpu", on_cpu=True)
    mu.compare(got, mu.plain_logits(folders[name], requests), "float32")


@pytest.mark.parametrize("name", ["A", "B"])
@pytest.mark.parametrize("mode", ["whole", "tail", "portions", "mixed"])
def test_replay_matches_plain(name, mode, folders, tmp_path, monkeypatch):
    """Whole prompts; a prompt and then token by token (across the edges of chunks and pages);
    portions down to two tokens; up to four live requests, portions beside single tokens."""
    kernel_refs.install(monkeypatch)
    requests = requests_of(name, 3, LENGTHS[name])
    trace = {"whole": ru.trace_whole, "tail": lambda r: ru.trace_tail(r, 16), "portions": ru.trace_portions,
             "mixed": lambda r: ru.trace_mixed(r, 5, max_live=3)}[mode](requests)
    got = ru.run_trace(folders[name], "float32", trace, tmp_path, block_size=mu.BLOCK_SIZE[name], device="cpu", on_cpu=True)
    mu.compare(got, mu.plain_logits(folders[name], requests), "float32")


def test_pages_and_state_slots_are_used_again(folders, tmp_path, monkeypatch):
    """Seven requests through four state slots and a pool smaller than their sum: a slot's state
    starts at zero again for the request that takes it over."""
    kernel_refs.install(monkeypatch)
    requests = requests_of("A", 4, (12, 20, 7, 16, 9, 3, 11))
    trace = ru.trace_mixed(requests, 9, max_live=4)
    assert sum(ru.round64(len(t)) for t in requests.values()) > trace.peak_tokens
    got = ru.run_trace(folders["A"], "float32", trace, tmp_path, block_size=4, device="cpu", on_cpu=True)
    mu.compare(got, mu.plain_logits(folders["A"], requests), "float32")


def test_chunked_groups_give_pages_back(folders, monkeypatch):
    """Keys before the run of positions that the next token lies in are never read again: their
    pages return to the pool while the request lives."""
    kernel_refs.install(monkeypatch)
    _, model = load_model(folders["A"], dtype="float32", device="cpu")
    runner = ModelRunner(model, block_size=2, block_capacity=16, num_state_slots=2)
    tokens = requests_of("A", 5, (40,))["r0"]
    runner.begin("r0")
    for start in range(0, 40, 5):
        runner.step([StepEntry("r0", tokens[start:start + 5], [4])])
        record = runner.cache.request("r0")
        chunk = mu.PARALLEL_P["left"]["mask"]["size"]
        assert record.first_block[0] == (start + 5) // chunk * chunk // 2
        assert sum(1 for page in record.tables[0] if page >= 0) <= 5
    runner.cache.check_invariants()
    runner.end("r0")
    assert runner.cache.allocated_pages == 0


def test_long_decoding_token_by_token(folders, tmp_path, monkeypatch):
    kernel_refs.install(monkeypatch)
    requests = requests_of("B", 6, (70,))
    got = ru.run_trace(folders["B"], "float32", ru.trace_tail(requests, 69), tmp_path, block_size=8, device="cpu", on_cpu=True)
    mu.compare(got, mu.plain_logits(folders["B"], requests), "float32")


def test_greedy_generation_through_the_scheduler(folders, monkeypatch):
    kernel_refs.install(monkeypatch)
    _, model = load_model(folders["A"], dtype="float32", device="cpu")
    engine = build_engine(model, scheduler_config=SchedulerConfig(block_size=4, block_capacity=64, token_budget=8, max_batch_size=3),
                          eos_token_ids=())
    prompts = list(requests_of("A", 11, (13, 4, 9)).values())
    ids = [engine.submit(prompt, sampling_params=SamplingParams(max_new_tokens=6)) for prompt in prompts]
    engine.run_until_idle()
    for request_id, prompt in zip(ids, prompts):
        assert list(engine.request(request_id).output_token_ids) == mu.plain_greedy(folders["A"], prompt, 6)


class _Matrix:
    """A mixer or a feed-forward that is one matrix."""

    takes_stream = leaves_product = False

    def __init__(self, g, width):
        self.matrix = torch.randn(width, width, generator=g)

    def forward(self, x, *step):
        return x @ self.matrix.T


@pytest.mark.parametrize("chosen", [None, [2, 0]])
@pytest.mark.parametrize("last", ["layer_norm", "rms_norm", "own"])
@pytest.mark.parametrize("arrangement", ["shifted", "shifted_alone", "sandwich"])
def test_a_norm_left_pending_reaches_whoever_reads_the_stream(arrangement, last, chosen, monkeypatch):
    """Two layers that leave their last norm pending, and a last norm that applies it, one that knows none, and one of a program's own, for
    whole steps and for chosen rows: the formulas in 64 bits."""
    from types import SimpleNamespace

    from forge_engine_amd.cache.spec import CacheView
    from forge_engine_amd.parts.base import BuildContext, Residual
    from forge_engine_amd.parts.block import OutputNormBlock, SandwichNormBlock
    from forge_engine_amd.parts.norm import LayerNorm, RMSNorm, UpdateRMSNorm
    kernel_refs.install(monkeypatch)
    ctx, width, g = BuildContext(torch.device("cpu"), torch.float32), 6, torch.Generator().manual_seed(5)

    class OwnNorm(RMSNorm):
        leaves_factors = False

        def forward(self, residual, rows=None):
            if residual.pending is not None:
                residual.h += residual.pending
                residual.pending = None
            z = residual.h if rows is None else residual.h[rows.long()]
            return kernel_refs._unit(z, self.eps) * self.weight

    def norm(kind, **how):
        made = kind(ctx, "n", size=width, eps=1e-3, **how)
        for name, spec in made.param_specs().items():
            made.set_param(name, 1.0 + 0.3 * torch.randn(spec.shape, generator=g))
        return made

    def unit(x):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-3)

    x0 = torch.randn(4, width, generator=g)
    residual, want = Residual(x0.clone()), x0.double()
    batch = SimpleNamespace(cu_q=torch.tensor([0, 3, 4], dtype=torch.int32), token_seq=torch.tensor([0, 0, 0, 1], dtype=torch.int32),
                            state_slots=torch.tensor([1, 0], dtype=torch.int32), num_seqs=2, num_decode=1, carry={})
    for _ in range(2):
        mixer, feed_forward = _Matrix(g, width), None if arrangement == "shifted_alone" else _Matrix(g, width)
        if arrangement == "sandwich":
            norms = {role: norm(RMSNorm) for role in SandwichNormBlock.NORMS}
            SandwichNormBlock(ctx, mixer, feed_forward, norms).forward(residual, batch, None)
            w = {role: n.weight.double() for role, n in norms.items()}
            want = want + unit((unit(want) * w["input"]) @ mixer.matrix.T.double()) * w["mixer_out"]
            want = want + unit((unit(want) * w["post_mixer"]) @ feed_forward.matrix.T.double()) * w["ff_out"]
            continue
        norms = {role: norm(UpdateRMSNorm) for role in OutputNormBlock.NORMS}
        block = OutputNormBlock(ctx, mixer, feed_forward, norms, hidden_size=width, token_shift=True)
        block.set_param(block.name("shift"), torch.rand(width, generator=g))
        state = torch.zeros(2, width)
        block.forward(residual, batch, CacheView(states={OutputNormBlock.SHIFT_STATE: state}))
        before = torch.cat([torch.zeros(1, width), want[:2], torch.zeros(1, width)])
        mixed = (want + (before - want) * block.shift.double()) @ mixer.matrix.T.double()
        want = want + unit(mixed) * norms["mixer_out"].weight.double()
        if feed_forward is not None:
            want = want + unit(want @ feed_forward.matrix.T.double()) * norms["ff_out"].weight.double()
    final = norm({"layer_norm": LayerNorm, "rms_norm": RMSNorm, "own": OwnNorm}[last])
    rows = None if chosen is None else torch.tensor(chosen, dtype=torch.int32)
    got = final.forward(residual, rows=rows)
    if last == "layer_norm":
        centred = want - want.mean(-1, keepdim=True)
        expected = unit(centred) * final.weight + final.bias
    else:
        expected = unit(want) * final.weight
    assert torch.allclose(got.double(), expected if rows is None else expected[chosen], atol=2e-5)
    assert torch.allclose(residual.flush().double(), want, atol=2e-5) and residual.pending is None and residual.pending_norm is None


def test_a_norm_of_updates_needs_an_update(monkeypatch):
    """A part that has added its update into the stream itself leaves nothing to norm: refused, with the norm left pending as without."""
    from forge_engine_amd.parts.base import BuildContext, Residual
    from forge_engine_amd.parts.block import OutputNormBlock
    from forge_engine_amd.parts.norm import UpdateRMSNorm
    kernel_refs.install(monkeypatch)
    ctx = BuildContext(torch.device("cpu"), torch.float32)
    for shift in (True, False):
        block = OutputNormBlock(ctx, None, None, {"mixer_out": UpdateRMSNorm(ctx, "n", size=4, eps=1e-3)}, hidden_size=4, token_shift=shift)
        residual = Residual(torch.ones(2, 4))
        residual.add(None)
        with pytest.raises(ValueError, match="pending update"):
            block._last_norm("mixer_out", residual)


@pytest.mark.parametrize("knows_parts", [False, True])
def test_norms_of_their_own_way_are_called_as_before(knows_parts, monkeypatch):
    """A norm that takes over another's ``forward`` is not asked for rows with their parts, nor is its way left out where it norms updates."""
    from forge_engine_amd.parts.base import BuildContext, FeedForward, Residual
    from forge_engine_amd.parts.block import OutputNormBlock, PreNormBlock
    from forge_engine_amd.parts.norm import RMSNorm, UpdateRMSNorm
    kernel_refs.install(monkeypatch)
    ctx, asked = BuildContext(torch.device("cpu"), torch.float32), []

    class Before(RMSNorm):
        if not knows_parts:
            def forward(self, residual, rows=None, unscaled=False):
                asked.append(unscaled)
                return super().forward(residual, rows)

    class Takes(FeedForward):
        def takes_split(self, tokens):
            return True

    monkeypatch.setattr(RMSNorm, "forward", RMSNorm.forward if not knows_parts else lambda self, residual, rows=None, unscaled=False, split=False: asked.append(split))
    norm = Before(ctx, "n", size=4, eps=1e-3)
    norm.weight = torch.ones(4)
    block = PreNormBlock(ctx, None, Takes(ctx, "f"), {"input": norm})
    block._normed("input", Residual(torch.ones(2, 4)), block.feed_forward)
    assert asked == [knows_parts]

    class Doubled(UpdateRMSNorm):
        def forward(self, residual, rows=None):
            residual.pending = residual.pending * 2.0
            residual.flush()

    residual = Residual(torch.ones(2, 4))
    residual.add(torch.ones(2, 4))
    OutputNormBlock(ctx, None, None, {"mixer_out": Doubled(ctx, "n", size=4, eps=1e-3)}, hidden_size=4, token_shift=True)._last_norm("mixer_out", residual)
    assert torch.equal(residual.flush(), torch.full((2, 4), 3.0))
