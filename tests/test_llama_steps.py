"""Whole Llama-family steps against a plain float64 implementation: what one
fused kernel hands the next, the paged cache, and decode inputs that stay on the
device between steps."""
import gc
import math

import pytest
import torch

from rbg_amd import ops
from rbg_amd.engine.config import EngineConfig, ModelConfig
from rbg_amd.engine.engine import LLMEngine
from rbg_amd.engine.kv_cache import BlockTable
from rbg_amd.engine.model_runner import ModelRunner
from rbg_amd.engine.sequence import SamplingParams, Sequence

DEVICES = ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)]

# Three layers round some eight tensors each to bf16, by 2^-9 / sqrt(3) of their
# size on average, and such errors add up as a root: sqrt(24) * 2^-9 * 0.6 = 0.006
# of a row's size.  Products of few tokens' attention add to the worst row: 0.011
# to 0.015 over the cases here.  Twice that; a wrong hand-over shows as 0.1 or more.
NEAR = 3e-2


def config(norms: bool) -> ModelConfig:
    # splits of wo, w_down and wqkv, silu within the GEMM and after it, and the
    # kernels of a few rows all occur at these widths
    return ModelConfig(name="steps", hidden_size=2048, intermediate_size=5632,
                       num_layers=3, num_heads=16, num_kv_heads=4,
                       head_dim=128, vocab_size=512, max_position=4096,
                       rope_theta=1e4, qk_norm=norms)


def engine_config(norms, device, **kw):
    return EngineConfig(model=config(norms), device=device, max_seq_len=1024,
                        kv_pool_tokens=16384, enable_prefix_cache=False, **kw)


def spread_norms(model):
    """Norm weights away from 1."""
    gen = torch.Generator().manual_seed(7)
    with torch.no_grad():
        for name, p in model.named_parameters():
            if name.endswith("norm"):
                p.copy_(1 + 0.2 * torch.randn(p.shape, generator=gen))


def rms(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def oracle(model, tokens):
    """Logits [T, vocab] and every layer's rotated keys and values [layers, 2,
    kv heads, T, 128] of one sequence, in float64."""
    cfg = model.cfg
    w = {k: v.double() for k, v in model.state_dict().items()}
    ids = torch.tensor(tokens, device=model.device)
    at = torch.arange(len(tokens), dtype=torch.float64, device=ids.device)
    angle = at[:, None] * cfg.rope_theta ** (
        -torch.arange(64, dtype=torch.float64, device=ids.device) / 64)
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]

    def rotate(t):
        a, b = t[..., :64], t[..., 64:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    hide = at[None] > at[:, None]
    h, kvh = cfg.num_heads, cfg.num_kv_heads
    x, kept = w["embed"][ids], []
    for i in range(cfg.num_layers):
        lw = {k[len(f"layers.{i}."):]: v for k, v in w.items()
              if k.startswith(f"layers.{i}.")}
        y = rms(x, lw["input_norm"], cfg.rms_eps) @ lw["attn.wqkv"].t()
        q, k, v = y.view(len(tokens), -1, 128).split([h, kvh, kvh], 1)
        if cfg.qk_norm:
            q = rms(q, lw["attn.q_norm"], cfg.rms_eps)
            k = rms(k, lw["attn.k_norm"], cfg.rms_eps)
        q, k = rotate(q), rotate(k)
        heads = []
        for j in range(h):
            g = j // (h // kvh)
            s = q[:, j] @ k[:, g].t().contiguous() / math.sqrt(128)
            heads.append(s.masked_fill(hide, -math.inf).softmax(-1) @ v[:, g])
        x = x + torch.cat(heads, -1) @ lw["attn.wo"].t()
        gate, up = (rms(x, lw["post_norm"], cfg.rms_eps) @
                    lw["mlp.w_gate_up"].t()).chunk(2, -1)
        x = x + (torch.nn.functional.silu(gate) * up) @ lw["mlp.w_down"].t()
        kept.append(torch.stack([k, v]).transpose(1, 2))
    return rms(x, w["final_norm"], cfg.rms_eps) @ w["lm_head"].t(), \
        torch.stack(kept)


def near(got, want):
    """Of every row."""
    err = (got.double() - want).norm(dim=-1) / want.norm(dim=-1)
    assert err.max() < NEAR, err.max()


def held(cache, table, n):
    """Keys and values of a sequence's first n tokens, as oracle's."""
    kv = cache.kv[:, :, table.pages[:(n + 15) // 16]]
    return kv.transpose(2, 3).flatten(3, 4)[:, :, :, :n]


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("norms", [False, True])
@pytest.mark.parametrize("n", [1, 3, 5, 33, 65])
def test_steps(device, norms, n):
    """A prompt, a portion behind it for every other sequence, then single
    tokens: as many rows as each route of a decode step has, of padded
    batches; the first prompt is one token."""
    if device == "cpu" and n != 3:
        pytest.skip("the CPU has one route")
    runner = ModelRunner(engine_config(norms, device,
                                       enforce_eager=device == "cpu"))
    spread_norms(runner.model)
    gen = torch.Generator().manual_seed(n)

    def draw(count):
        return torch.randint(0, 512, (count,), generator=gen).tolist()

    seqs, done, wants = [], [0] * n, []
    for i in range(n):
        seq = Sequence(draw(1 + 37 * i % 50 + 20))
        seq.block_table = BlockTable(runner.cache)
        seq.block_table.ensure(seq.num_prompt_tokens)
        seqs.append(seq)
        wants.append(oracle(runner.model, seq.prompt_tokens))

    def feed(which, count):
        chunks = [(seqs[i], done[i],
                   seqs[i].prompt_tokens[done[i]:done[i] + count(i)])
                  for i in which]
        got = runner.feed(chunks, [[len(c[2]) - 1] for c in chunks])
        for i, c in zip(which, chunks):
            done[i] += len(c[2])
        near(got, torch.stack([wants[i][0][done[i] - 1] for i in which]))

    feed(range(n), lambda i: 1 if i == 0 else 2 + 5 * i % 7)
    feed(range(0, n, 2), lambda i: 3 + i % 10)
    for _ in range(3):
        # the runner takes a decode token as the sequence's last
        rows = []
        for i, seq in enumerate(seqs):
            whole = seq.prompt_tokens
            seq.prompt_tokens = whole[:done[i] + 1]
            rows.append(whole)
        feed(range(n), lambda i: 1)
        for seq, whole in zip(seqs, rows):
            seq.prompt_tokens = whole
    assert bool(runner._graphs) == (device == "cuda")
    for seq, at, (_, want) in zip(seqs, done, wants):
        near(held(runner.cache, seq.block_table, at), want[:, :, :, :at])


@pytest.mark.parametrize("device,eager", [
    ("cpu", True), pytest.param("cuda", True, marks=pytest.mark.gpu),
    pytest.param("cuda", False, marks=pytest.mark.gpu)])
@pytest.mark.parametrize("norms", [False, True])
@pytest.mark.parametrize("first,later", [(1, 0), (1, 2), (3, 2), (5, 4)])
def test_generated_steps(device, eager, norms, first, later):
    """Decode steps one after another, whose inputs stay on the device: padded
    batches, a prompt between them, a batch that grows into another captured
    size and shrinks again.  Every step's logits are those of the tokens so
    far."""
    if device == "cpu" and (first, later) != (1, 2):
        pytest.skip("the CPU has one route")
    eng = LLMEngine(engine_config(norms, device, max_batch_size=16,
                                  enforce_eager=eager))
    runner = eng.runner
    spread_norms(runner.model)
    inner, seen = runner._decode_logits, []

    def keep(seqs):
        out = inner(seqs)
        seen.extend((s, s.num_tokens - 1, row)
                    for s, row in zip(seqs, out.clone()))
        return out
    runner._decode_logits = keep
    gen = torch.Generator().manual_seed(first)

    def add(count, new):
        return [eng.add_request(
            torch.randint(0, 512, (3 + 29 * i % 40,), generator=gen).tolist(),
            SamplingParams(max_new_tokens=new + i)) for i in range(count)]

    seqs = add(first, 14)
    for _ in range(6):
        eng.step()
    seqs += add(later, 4)
    while eng.scheduler.has_work():
        eng.step()
    del runner._decode_logits           # no cycle that keeps the pool
    assert bool(runner._graphs) != eager
    assert len(seen) == sum(len(s.output_tokens) - 1 for s in seqs)
    wants = {s.seq_id: oracle(runner.model, s.prompt_tokens +
                              s.output_tokens)[0] for s in seqs}
    near(torch.stack([row for _, _, row in seen]),
         torch.stack([wants[s.seq_id][at] for s, at, _ in seen]))
    for s in seqs:          # greedy, but for a near tie
        for at, tok in enumerate(s.output_tokens):
            row = wants[s.seq_id][s.num_prompt_tokens + at - 1]
            assert row.max() - row[tok] < NEAR * row.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("collects", [True, False])
def test_nothing_is_collected_in_a_capture(collects):
    """Python's own collection, which may free a dropped engine's pool and
    captured steps, rests while a step is captured."""
    runner = ModelRunner(engine_config(False, "cuda"))
    seq = Sequence([1, 2, 3])
    seq.block_table = BlockTable(runner.cache)
    seq.block_table.ensure(4)
    runner.feed([(seq, 0, [1, 2])], [[1]])
    inner, seen = runner.model.logits, []

    def logits(hidden):
        if torch.cuda.is_current_stream_capturing():
            seen.append(gc.isenabled())
        return inner(hidden)
    runner.model.logits = logits
    try:
        gc.enable() if collects else gc.disable()
        out = runner.feed([(seq, 2, [3])], [[0]])
        assert gc.isenabled() == collects
    finally:
        gc.enable()
        del runner.model.logits
    assert seen == [False] and out.isfinite().all()


class Prompts:
    """Two sequences, of which a step takes a half."""

    def __init__(self, norms, rows):
        self.runner = ModelRunner(engine_config(norms, "cuda"))
        spread_norms(self.runner.model)
        gen = torch.Generator().manual_seed(rows)
        self.seqs = []
        for count in (rows - 2, 2):
            seq = Sequence(torch.randint(0, 512, (2 * count,),
                                         generator=gen).tolist())
            seq.block_table = BlockTable(self.runner.cache)
            seq.block_table.ensure(2 * count)
            self.seqs.append(seq)

    def step(self, half):
        chunks = []
        for s in self.seqs:
            n = len(s.prompt_tokens) // 2
            chunks.append((s, half * n, s.prompt_tokens[half * n:][:n]))
        return self.runner.feed(chunks, [[0, len(c[2]) - 1] for c in chunks])


def count_blocks(monkeypatch):
    """(name, whether it took the call) of every native block."""
    calls = []
    for name in ("prompt_attention_block", "swiglu_block"):
        def counted(*args, name=name, inner=getattr(ops, name)):
            out = inner(*args)
            calls.append((name, out is not None))
            return out
        monkeypatch.setattr(ops, name, counted)
    return calls


@pytest.mark.gpu
@pytest.mark.parametrize("norms", [False, True])
@pytest.mark.parametrize("rows", [5, 37, 65, 300, 1100])
def test_blocks_issued_by_one_call(norms, rows, monkeypatch):
    """The same launches as of a block's parts, so the same bits: prompts, and
    portions behind a past."""
    prompts = Prompts(norms, rows)
    layers = len(prompts.runner.model.layers)
    calls = count_blocks(monkeypatch)
    got = [prompts.step(0), prompts.step(1), prompts.runner.cache.kv.clone()]
    for name in ("prompt_attention_block", "swiglu_block"):
        assert calls.count((name, True)) == 2 * layers
        monkeypatch.setattr(ops, name, lambda *a: None)
    prompts.runner.cache.kv.zero_()
    want = [prompts.step(0), prompts.step(1), prompts.runner.cache.kv]
    assert len(calls) == 4 * layers
    for a, b in zip(got, want):
        assert torch.equal(a, b)


class Delegate(torch.nn.Module):
    """In the place of a module, with its attributes."""

    def __init__(self, inner, seen):
        super().__init__()
        self.inner, self.seen = inner, seen

    def forward(self, *args):
        self.seen.append("other module")
        return self.inner(*args)

    def __getattr__(self, name):
        try:
            return super().__getattr__(name)
        except AttributeError:
            return getattr(self.inner, name)


@pytest.mark.gpu
@pytest.mark.parametrize("part", ["attn", "mlp"])
def test_changed_parts_of_layers_are_called(part, monkeypatch):
    """Prompts go through a part whose forward is replaced or hooked, or that is
    another module, and give the same bits."""
    prompts = Prompts(False, 37)
    model, seen = prompts.runner.model, []
    want = prompts.step(0)

    def noted(name, result=None):
        def note(*args):
            seen.append(name)
            return result(*args) if result else None
        return note
    module = getattr(model.layers[1], part)
    module.forward = noted("instance", module.forward)
    assert torch.equal(prompts.step(0), want)
    del module.forward
    with monkeypatch.context() as m:
        inner = type(module).forward
        m.setattr(type(module), "forward", noted("class", inner))
        assert torch.equal(prompts.step(0), want)
    setattr(model.layers[1], part, Delegate(module, seen))
    assert torch.equal(prompts.step(0), want)
    setattr(model.layers[1], part, module)
    for name, register in (
            ("hook", module.register_forward_hook),
            ("hook before", module.register_forward_pre_hook)):
        handle = register(noted(name))
        assert torch.equal(prompts.step(0), want)
        handle.remove()
    handle = torch.nn.modules.module.register_module_forward_hook(
        lambda m, *a: seen.append("any hook") if m is module else None)
    assert torch.equal(prompts.step(0), want)
    handle.remove()
    assert seen == ["instance"] + ["class"] * len(model.layers) + [
        "other module", "hook", "hook before", "any hook"]


@pytest.mark.gpu
def test_layers_of_other_widths(monkeypatch):
    """A layer's products go by its own weights, not by the first layer's."""
    prompts = Prompts(False, 300)
    mlp = prompts.runner.model.layers[1].mlp
    gate, up = mlp.w_gate_up.chunk(2)
    with torch.inference_mode():        # no multiple that the kernels take
        mlp.w_gate_up = torch.nn.Parameter(
            torch.cat([gate[:1000], up[:1000]]), requires_grad=False)
        mlp.w_down = torch.nn.Parameter(mlp.w_down[:, :1000].contiguous(),
                                        requires_grad=False)
    got = prompts.step(0)
    for name in ("prompt_attention_block", "swiglu_block"):
        monkeypatch.setattr(ops, name, lambda *a: None)
    assert torch.equal(prompts.step(0), got)
