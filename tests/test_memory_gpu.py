"""The engine's memory figure (GPU): weights, workspace and cache are known when the engine is built, a limit
that they exceed is refused there with the three numbers, the cache is sized from what the limit leaves, and
no later step makes the workspace grow."""
import pytest
import torch

import plain_minicpm as plain
import tiny

pytestmark = pytest.mark.gpu


def total_memory():
    return torch.cuda.get_device_properties(0).total_memory


@pytest.mark.parametrize("name", ["A", "B"])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_no_step_grows_the_workspace_after_the_engine_is_built(model_dirs, name, dtype):
    from cpmcu_amd import Engine, EngineOptions, StepEntry
    eng = Engine.from_dir(model_dirs[name], EngineOptions(dtype=dtype, max_tokens=8192, max_slots=20,
                                                          max_step_tokens=128, hip_graph=True))
    ws, gen = eng.workspace.bytes(), eng.workspace.generation
    mem = eng.memory_report()
    assert mem["weight_bytes"] > 0 and mem["workspace_bytes"] == ws and mem["cache_bytes"] == eng.cache.bytes()
    vocab = eng.vocab_size
    slots = [eng.acquire() for _ in range(20)]
    # prompts of every kind of length, one pass and several; then decode steps of every batch size, up to
    # the model's longest sequence (tiny B's block selection is at work from 64 on, long LongRoPE factors and split keys later)
    limit = eng.max_seq_len
    grow = (limit // 2) // 19
    eng.step([StepEntry(s, tiny.random_tokens(3 + grow * i, vocab, i), [2 + grow * i]) for i, s in enumerate(slots)])
    for b in (20, 17, 16, 9, 3, 2, 1):
        for _ in range(2):
            eng.step([StepEntry(s, [5], [0]) for s in slots[:b]])
    more = limit - eng.length(slots[0]) - 4
    eng.step([StepEntry(slots[0], tiny.random_tokens(more, vocab, 77), [more - 1])])
    eng.step([StepEntry(slots[0], [1], [0]), StepEntry(slots[1], [2], [0])])
    assert eng.workspace.grown == [] and eng.workspace.bytes() == ws and eng.workspace.generation == gen
    for s in slots:
        eng.release(s)


def test_a_limit_that_weights_workspace_and_cache_exceed_is_refused_when_the_engine_is_built(model_dirs):
    from cpmcu_amd import Engine, EngineOptions
    from cpmcu_amd.engine.engine import EngineMemoryError
    ok = Engine.from_dir(model_dirs["B"], EngineOptions(dtype="bfloat16", max_tokens=4096, max_slots=4,
                                                        memory_limit=0.5))
    mem = ok.memory_report()
    need = mem["weight_bytes"] + mem["workspace_bytes"] + mem["cache_bytes"]
    # a limit a little below what the same engine needs: refused with the three numbers
    small = (need - 4096) / total_memory()
    with pytest.raises(EngineMemoryError, match=r"weights .* GiB \+ workspace .* GiB \+ cache .* GiB \(for 4096 tokens\)"
                                                r".*the limit is"):
        Engine.from_dir(model_dirs["B"], EngineOptions(dtype="bfloat16", max_tokens=4096, max_slots=4,
                                                       memory_limit=small))
    # the same limit sizes a cache that fits when max_tokens is left open: fewer tokens, whole pages
    sized = Engine.from_dir(model_dirs["B"], EngineOptions(dtype="bfloat16", max_tokens=None, max_slots=4,
                                                           memory_limit=small))
    m2 = sized.memory_report()
    assert 0 < sized.max_tokens < 4096 and sized.max_tokens % 64 == 0
    assert m2["weight_bytes"] + m2["workspace_bytes"] + m2["cache_bytes"] <= small * total_memory()
    # no room even for a page a slot
    with pytest.raises(EngineMemoryError, match="memory limit exceeded"):
        Engine.from_dir(model_dirs["B"], EngineOptions(dtype="bfloat16", max_tokens=None, max_slots=4,
                                                       memory_limit=(mem["weight_bytes"] + 1000) / total_memory()))
    # no limit given, but a cache that the device cannot hold: said at build too, not by the allocator later
    with pytest.raises(EngineMemoryError, match=r"device memory exceeded: weights .* \+ workspace .* \+ cache .*left for"):
        Engine.from_dir(model_dirs["B"], EngineOptions(dtype="bfloat16", max_tokens=2_000_000_000, max_slots=4))
    with pytest.raises(ValueError, match="max_tokens, or a memory_limit"):
        Engine.from_dir(model_dirs["B"], EngineOptions(dtype="bfloat16", max_tokens=None))


@pytest.mark.parametrize("name,batch,seq", [("A", None, None), ("A", 3, 100), ("B", 2, None)])
def test_llm_sizes_its_cache_from_the_memory_limit_and_generates(model_dirs, name, batch, seq):
    """The command line's default: no max_tokens; the cache takes what memory_limit leaves, capped by the
    sequences it is for (cpmcu/llm.py:115-116)."""
    from cpmcu_amd.llm import LLM
    cfg, w = tiny.read_model(model_dirs[name])
    llm = LLM(model_dirs[name], dtype="float32", memory_limit=0.02, max_batch=batch, max_seq_len=seq)
    with pytest.raises(RuntimeError, match="init_storage"):
        llm.load_from_hf()
    longest = llm.init_storage()
    llm.load_from_hf()
    limit = seq or cfg["max_position_embeddings"]
    slots = batch or 1
    assert longest == limit
    # 2 % of the device holds far more than these sequences: the cap decides, in whole pages
    assert llm.engine.max_tokens == slots * (-(-limit // 64) * 64) and llm.engine.cache.max_slots == slots
    mem = llm.engine.memory_report()
    assert mem["weight_bytes"] + mem["workspace_bytes"] + mem["cache_bytes"] <= 0.02 * total_memory()
    prompts = [tiny.random_tokens(7 + 6 * i, cfg["vocab_size"], 50 + i) for i in range(slots + 1)]   # one batch more
    outs = llm.generate(prompts, generation_length=6)
    assert [c.tokens for c in outs] == [plain.greedy(cfg, w, p, 6) for p in prompts]
    llm.engine.cache.check()
    with pytest.raises(ValueError, match="exceeds maximum supported length"):
        llm.prefill(list(range(limit + 1)))


@pytest.mark.parametrize("name", ["A", "B"])
def test_an_engine_of_short_passes_lets_the_checkpoint_layout_go(model_dirs, name):
    """With forward passes of at most 32 tokens no product reads the weights in the checkpoint's layout: the linear
    layers keep their re-laid copy only (and the fused q/k/v copy), the memory figure shows it, and prompts, cut
    into passes of 32, and decode steps give the logits of the plain implementation."""
    import plain_minicpm as plain
    import schedules
    from cpmcu_amd import Engine, EngineOptions
    from cpmcu_amd.parts.linear import Linear
    cfg, w = tiny.read_model(model_dirs[name])
    full = Engine.from_dir(model_dirs[name], EngineOptions(dtype="bfloat16", max_tokens=1024, max_slots=3))
    short = Engine.from_dir(model_dirs[name], EngineOptions(dtype="bfloat16", max_tokens=1024, max_slots=3,
                                                            max_step_tokens=32, hip_graph=True))
    linears = [p for p in short.model.all_parts() if isinstance(p, Linear)]
    assert linears and all(p.weight is None and p.tiled is not None for p in linears)
    assert all(p.weight is not None for p in full.model.all_parts() if isinstance(p, Linear))
    assert short.memory_report()["weight_bytes"] < 0.8 * full.memory_report()["weight_bytes"]
    reqs = {"x": tiny.random_tokens(150, cfg["vocab_size"], 31), "y": tiny.random_tokens(45, cfg["vocab_size"], 32)}
    refs = {r: plain.forward(cfg, w, t).float() for r, t in reqs.items()}
    for what, got in (("whole", schedules.whole(short, reqs)), ("tail", schedules.tail(short, reqs, 20)),
                      ("batched", schedules.batched(short, reqs, {"x": 100, "y": 7}, [("x", "y")]))):
        for r, ref in refs.items():
            assert float((got[r] - ref).abs().max()) < 0.01 * float(ref.abs().max()), (what, r)
    short.cache.check()


def wide_model(hidden=2048, ff=6144, layers=2):
    """Two layers whose products are large enough for the kernels of many rows."""
    return dict(tiny.tiny_a(), num_hidden_layers=layers, hidden_size=hidden, num_attention_heads=hidden // 128, num_key_value_heads=2, head_dim=128,
                intermediate_size=ff, vocab_size=512, max_position_embeddings=4096,
                rope_scaling={"rope_type": "longrope", "short_factor": [1.0] * 64, "long_factor": [1.0] * 64,
                              "original_max_position_embeddings": 4096})


def wide_engine(ff, **options):
    from cpmcu_amd import Engine, EngineOptions, get_architecture
    from cpmcu_amd.weights import random_tensors
    raw = wide_model(ff=ff)
    cfg = get_architecture(raw["architectures"][0]).config_class.from_dict(raw)
    return Engine.from_tensors(cfg, random_tensors(cfg, 5, device="cuda:0"), EngineOptions(**options))


def prompt(eng, n):
    from cpmcu_amd import StepEntry
    s = eng.acquire()
    out = eng.step([StepEntry(s, [(31 * i) % eng.vocab_size for i in range(n)], [n - 1])])
    eng.release(s)
    return out


@pytest.mark.parametrize("ff,chunk", [(6144, 2048), (16384, 1800)])
def test_products_of_every_number_of_rows_find_their_workspace(ff, chunk):
    """Whether a product is the library's or the kernel's goes up and down with the rows: passes on both sides of the rule, between the rehearsed
    sizes, find the workspace as the engine left it, and the captured decode step stays."""
    from cpmcu_amd import StepEntry, ops
    rows = [65, 100, 300, 512, 700, 705, 769, 900, 1024, 1100, 1280, 1366, 1500, 1536, 1700, 1792, 1800, 2048]
    ways = [ops.product_faster(n, 2 * ff, 2048, True) for n in rows if n <= chunk]
    assert True in ways and False in ways
    eng = wide_engine(ff, dtype="bfloat16", max_tokens=4096, max_slots=8, max_step_tokens=chunk, hip_graph=True)
    held = eng.acquire()
    prompt_of_held = [StepEntry(held, [1, 2, 3], [2])]
    eng.step(prompt_of_held)
    eng.step([StepEntry(held, [5], [0])])
    graphs, ws, gen = dict(eng._graphs), eng.workspace.bytes(), eng.workspace.generation
    assert len(graphs) == 1
    for n in rows:
        if n <= chunk:
            prompt(eng, n)
            assert eng.workspace.grown == [], n
    eng.step([StepEntry(held, [5], [0])])
    assert eng.workspace.bytes() == ws and eng.workspace.generation == gen and eng._graphs == graphs


def test_partial_sums_lie_in_the_workspace():
    """Shares of K leave their sums in room that the engine reserved: a pass that takes them asks the allocator for nothing."""
    from cpmcu_amd import ops
    eng = wide_engine(6144, dtype="bfloat16", max_tokens=4096, max_slots=4, max_step_tokens=1100)
    most = max(ops.product_plan(n, N, K, gated) * n * N * 4 for n in range(65, 1101)
               for N, K, gated in ((12288, 2048, True), (2048, 6144, False))
               if ops.product_plan(n, N, K, gated) > 1 and ops.product_faster(n, N, K, gated))
    assert most > 8 << 20 and eng.workspace.bytes() >= most
    rows = [65, 130, 256, 300, 700, 769, 1025, 1100]
    assert any(ops.product_plan(n, 2048, 6144, False) > 1 and ops.product_faster(n, 2048, 6144) for n in rows if n > 704)
    assert any(ops.product_plan(n, 2048, 6144, False) > 1 and ops.product_faster(n, 2048, 6144) for n in rows if n <= 704)
    out = [prompt(eng, n) for n in rows]                            # (what a pass uploads is allocated by now)
    held, report = torch.cuda.memory_allocated(), eng.memory_report()
    for n, want in zip(rows, out):
        torch.cuda.reset_peak_memory_stats()
        got = prompt(eng, n)
        assert torch.cuda.max_memory_allocated() - held < 1 << 20, n
        assert torch.equal(got, want)
        del got
    assert eng.workspace.grown == [] and eng.memory_report() == report


def test_scratch_that_is_too_small_is_refused():
    from cpmcu_amd import ops
    x, w = torch.zeros(100, 1024, device="cuda:0", dtype=torch.bfloat16), torch.zeros(64, 1024, device="cuda:0", dtype=torch.bfloat16)
    out = torch.empty(100, 64, device="cuda:0", dtype=torch.bfloat16)
    room = torch.empty(2 * 100 * 64 + 1, device="cuda:0")
    ops.product_parts(x, w, out, 2, scratch=room)
    for bad in (room[:-2], room[1:], torch.empty(2 * 100 * 64), room[:2 * 100 * 64].view(64, 200).t()):
        with pytest.raises(ops.KernelError, match="shares"):
            ops.product_parts(x, w, out, 2, scratch=bad)


def test_short_prompts_of_real_widths():
    """Passes of 65 to 1,100 rows through layers whose products take shares of K and the gate's kernel: as far from the float32 engine as the
    same engine's passes of up to 64 rows, which have kernels of their own, within a factor of two (bfloat16 rounds in other places)."""
    from cpmcu_amd import StepEntry
    wide = wide_engine(6144, dtype="bfloat16", max_tokens=4096, max_slots=4, max_step_tokens=2048)
    short = wide_engine(6144, dtype="bfloat16", max_tokens=4096, max_slots=4, max_step_tokens=64)
    exact = wide_engine(6144, dtype="float32", max_tokens=4096, max_slots=4, max_step_tokens=2048)

    def logits(eng, n):
        s = eng.acquire()
        out = eng.step([StepEntry(s, [(31 * i) % eng.vocab_size for i in range(n)], list(range(max(0, n - 40), n)))]).clone()
        eng.release(s)
        return out

    for n in (65, 130, 300, 512, 704, 769, 1100):
        want = logits(exact, n)
        off = [float((logits(eng, n) - want).norm() / want.norm()) for eng in (wide, short)]
        assert off[0] <= 2 * off[1] < 0.04, (n, off)
