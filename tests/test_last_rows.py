"""Behind the last layer's attention only the rows go on whose logits are asked for: the same logits and the same memory as with all rows."""

import pytest
import torch

from kvmini.engine.engine import EngineConfig, LLMEngine
from kvmini.engine.scheduler import Batch, ScheduledChunk
from kvmini.models import pipilix, registry
from kvmini.models.llama import LlamaConfig

LLAMA = LlamaConfig("few-rows", 512, 256, 512, 3, 4, 2, 64, 500000.0, 1e-5, 512, 1, 2)
BACKENDS = [pytest.param("cpu", torch.float32, False, id="cpu"), pytest.param("cuda:0", torch.float32, False, id="hip-fp32", marks=pytest.mark.gpu),
            pytest.param("cuda:0", torch.bfloat16, False, id="hip-bf16", marks=pytest.mark.gpu), pytest.param("cuda:0", torch.bfloat16, True, id="hip-bf16-graphs", marks=pytest.mark.gpu)]


@pytest.mark.parametrize("design", ["llama", "vodinex-tiny", "pipilix-tiny", "zipelix-tiny", "gebasun-tiny"])
@pytest.mark.parametrize("device,dtype,graphs", BACKENDS)
def test_rows_that_nobody_asks_for_end_at_the_last_layer(design, device, dtype, graphs):
    """A decode row, the end of a prompt and a fresh one, with several rows, one and none asked for.  The selected rows' products are those of fewer rows:
    fp32 sums in another order, within 2e-5 of the logits' spread; in bf16 a last layer rounded otherwise, within 2 % of it."""
    if design == "llama" and device != "cpu" and dtype == torch.float32:
        pytest.skip("this family's kernels are bf16")
    cfg = LLAMA if design == "llama" else registry.resolve_model(design)[0]
    weights = registry.random_weights(cfg, device, dtype, seed=1)
    held, new, want = (40, 30, 0, 3), (1, 25, 70, 20), ([0], [3, 24], [69], [])

    def step(few):
        eng = LLMEngine(EngineConfig(model=cfg.name, device=device, max_num_seqs=4, max_batched_tokens=256, max_model_len=256, num_blocks=80, use_graphs=False), weights=weights)
        eng.runner.few_at_last = few
        seqs = [eng.make_sequence([1 + (i * (j + 3)) % 500 for i in range(h + n)]) for j, (h, n) in enumerate(zip(held, new))]
        batch = eng.scheduler.schedule_given([(s, h, []) for s, h in zip(seqs, held) if h])
        eng.runner.execute(batch)
        eng.scheduler.note_computed(batch)
        if graphs:
            eng.runner.rcfg.use_graphs = True
            eng.runner.capture_graphs([eng.runner.bucket_for(sum(new))])
            assert eng.runner.graphs
        assert (eng.runner.last_rows(eng.runner.bucket_for(sum(new))) is not None) == few
        for _ in range(3 if graphs else 1):
            logits = eng.runner.execute(eng.scheduler.schedule_given([(s, n, w) for s, n, w in zip(seqs, new, want)]))[1].clone()
        memory = [eng.runner.kv_cache] if design == "llama" else [t for run in eng.runner.memory.runs for branch in run for t in branch]
        return logits.double(), memory

    (got, mine), (ref, theirs) = step(True), step(False)
    assert got.shape == ref.shape == (4, cfg.vocab_size)
    assert ((got - ref).pow(2).mean(-1).sqrt() / ref.std(-1)).max().item() < (2e-5 if dtype == torch.float32 else 0.02)
    for a, b in zip(mine, theirs):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


@pytest.mark.gpu
@pytest.mark.parametrize("graphs", [False, True])
@pytest.mark.parametrize("design", ["llama-128", "llama", "vodinex-tiny", "pipilix-tiny", "zipelix-tiny", "gebasun-tiny"])
def test_prompts_alone_leave_out_the_launches_for_single_rows(design, graphs):
    """A step without a row that is the only one of its sequence, and one with such a row: as with those launches, bit for bit."""
    cfg = LlamaConfig("alone", 512, 512, 512, 2, 4, 2, 128, 500000.0, 1e-5, 512, 1, 2) if design == "llama-128" else LLAMA if design == "llama" else registry.resolve_model(design)[0]
    weights = registry.random_weights(cfg, "cuda:0", torch.bfloat16, seed=1)

    def steps(apart):
        eng = LLMEngine(EngineConfig(model=cfg.name, device="cuda:0", max_num_seqs=4, max_batched_tokens=256, max_model_len=256, num_blocks=80, use_graphs=graphs), weights=weights)
        eng.runner.rows_apart = eng.runner.rows_apart and apart
        eng.warmup()
        kinds = []
        launch = eng.runner.launch
        eng.runner.launch = lambda *a, **k: (lambda h: (kinds.append(h.key[1]), h)[1])(launch(*a, **k))
        seqs = [eng.make_sequence([1 + (i * (j + 3)) % 500 for i in range(150)]) for j in range(3)]
        out = []
        for part in ((70, 33, 0), (80, 17, 100), (0, 1, 50), (0, 99, 0)):
            batch = eng.scheduler.schedule_given([(s, n, [0, n - 1]) for s, n in zip(seqs, part) if n > 1] + [(s, n, [0]) for s, n in zip(seqs, part) if n == 1])
            out.append(eng.runner.execute(batch)[1].clone())
            eng.scheduler.note_computed(batch)
        memory = [eng.runner.kv_cache] if "llama" in design else [t for run in eng.runner.memory.runs for branch in run for t in branch]
        return out + memory, kinds

    (got, kinds), (want, old) = steps(True), steps(False)
    assert 4 not in old and (kinds == old if design == "llama" else kinds[0] == 4 and kinds[2] == 0)  # (heads of 64 have one launch for both)
    for a, b in zip(got, want):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


@pytest.mark.parametrize("device,graphs", [pytest.param("cpu", False, id="cpu"), pytest.param("cuda:0", False, id="hip", marks=pytest.mark.gpu), pytest.param("cuda:0", True, id="hip-graphs", marks=pytest.mark.gpu)])
def test_drafts_cut_to_one_token_are_a_single_row(device, graphs):
    """A chunk of drafts of which the step's budget leaves one token, beside longer chunks: a hybrid's kernels take it as a single row, so the step has the launches for
    those, and what the row leaves in memory is that of a step that always has them."""
    cfg = registry.resolve_model("pipilix-tiny")[0]
    weights = registry.random_weights(cfg, device, torch.float32 if device == "cpu" else torch.bfloat16, seed=1)

    def step(apart):
        eng = LLMEngine(EngineConfig(model=cfg.name, device=device, max_num_seqs=4, max_batched_tokens=64, max_model_len=128, num_blocks=40, use_graphs=graphs), weights=weights)
        eng.runner.rows_apart = apart
        eng.warmup()
        seqs = [eng.make_sequence([1 + (i * (j + 3)) % 500 for i in range(30)]) for j in range(2)]
        first = eng.scheduler.schedule_given([(s, 20, [19]) for s in seqs])
        eng.runner.execute(first)
        eng.scheduler.note_computed(first)
        seqs[0].prompt_ids, seqs[0].draft_ids = seqs[0].prompt_ids[:21], [7, 9]  # decoding, two drafts behind its last token
        whole = eng.scheduler.schedule_given([(seqs[1], 10, [9])])
        cut = ScheduledChunk(seqs[0], 20, 1, False)
        missing = eng.scheduler._blocks_needed(seqs[0], 21)
        seqs[0].blocks += eng.scheduler.bm.allocate(missing) if missing else []
        handle = eng.runner.launch(Batch([cut] + whole.chunks, 11))
        eng.runner.collect(handle)
        return handle.key[1], [t.clone() for run in eng.runner.memory.runs for branch in run for t in branch]

    (kind, got), (_, want) = step(True), step(False)
    assert kind == 0  # (4: prompts alone)
    for a, b in zip(got, want):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


@pytest.mark.parametrize("design", ["gebasun-tiny", "sandwich"])
@pytest.mark.parametrize("device,dtype", [pytest.param("cpu", torch.float32, id="cpu"), pytest.param("cuda:0", torch.bfloat16, id="hip", marks=pytest.mark.gpu)])
def test_the_last_layers_experts_have_no_rows_that_nobody_asks_for(design, device, dtype, monkeypatch):
    """The rows behind the last layer's mixer are as many as a step may ask for: those beyond the ones it does ask for are padding, as the others are in warm-up."""
    cfg = pipilix.stack("experts-last", 512, 96, "DM", 3, 24, 40, 48, 20, 112, 6, 2, 40) if design == "sandwich" else registry.resolve_model(design)[0]
    assert cfg.layers[cfg.runs[-1].layer].moe is not None
    eng = LLMEngine(EngineConfig(model=cfg.name, device=device, max_num_seqs=4, max_batched_tokens=256, max_model_len=256, num_blocks=80, use_graphs=False),
                    weights=registry.random_weights(cfg, device, dtype, seed=1))
    calls, experts = [], eng.runner.mixers.experts
    monkeypatch.setattr(eng.runner.mixers, "experts", lambda m, w, h, st, **kw: (calls.append((h.shape[0], st.slots.tolist())), experts(m, w, h, st, **kw))[1])
    seqs = [eng.make_sequence([1 + (i * (j + 3)) % 500 for i in range(60)]) for j in range(2)]
    eng.runner.execute(eng.scheduler.schedule_given([(seqs[0], 60, [59]), (seqs[1], 40, [7, 39])]))
    rows, slots = calls[-1]
    assert rows == len(slots) == eng.runner.sample_rows(eng.runner.bucket_for(100)) > 3
    at = lambda s, pos: s.blocks[pos // eng.runner.block_size] * eng.runner.block_size + pos % eng.runner.block_size
    assert slots == [at(seqs[0], 59), at(seqs[1], 7), at(seqs[1], 39)] + [-1] * (rows - 3)
    eng.runner._stage_dummy()
    calls.clear()
    with torch.no_grad():
        eng.runner.forward(eng.runner.bucket_for(100))
    assert all(s == -1 for _rows, slots in calls for s in slots)
