"""Generation through the entry points: scheduler, step function, device sampler,
decode graphs, preemption, command line."""
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from helpers import CONFIGS, random_tokens, read_folder
from plain import qwen3_plain as plain

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def plain_generate(cfg, w, prompt, n, number=0, temperature=0.0, top_k=0, top_p=1.0, seed=42):
    from tinyinfer_amd.sampling import uniform, DEFAULT_TOP_K
    toks = list(prompt)
    out = []
    for i in range(n):
        logits = plain.forward(w, cfg, toks)[-1]
        if temperature <= 0:
            t = plain.argmax_lowest(logits)
        else:
            p = plain.sample_distribution(logits, temperature, top_k or DEFAULT_TOP_K, top_p)
            t = plain.draw(p, uniform(seed, number, i))
        toks.append(t)
        out.append(t)
    return out


def test_config_a_greedy_eight_tokens(model_folders):
    """One request, an 8-token prompt, greedy decoding of 8 tokens, in 32-bit."""
    import tinyinfer_amd as ti
    d = model_folders("A", "float32")
    cfg, w = read_folder(d)
    prompt = random_tokens(8, 256, 0)
    llm = ti.LLM(d, dtype="float32", max_seq=64, max_requests=1)
    got = llm.generate([prompt], max_new_tokens=8)[0]
    assert got == plain_generate(cfg, w, prompt, 8)


def test_config_b_mixed_batch_with_temperature(model_folders):
    """Three requests with prompts of 5, 17 and 33 tokens, prefilled in portions of
    7 beside decoding requests, pages of 4 tokens, temperature 0.8, a fixed seed, 6
    tokens each, in 32-bit."""
    import tinyinfer_amd as ti
    d = model_folders("B", "float32")
    cfg, w = read_folder(d)
    prompts = [random_tokens(n, 1000, 10 + n) for n in (5, 17, 33)]
    engine = ti.Engine.from_folder(d, "float32", page_size=4, max_tokens=192, max_requests=3, max_seq=64)
    stats = ti.GenerationStats()
    got = ti.generate_ids(engine, prompts, max_new_tokens=6, temperature=0.8, seed=123, chunk_size=7,
                          max_batched_tokens=12, stats=stats)
    want = [plain_generate(cfg, w, p, 6, number=i, temperature=0.8, seed=123) for i, p in enumerate(prompts)]
    assert got == want
    # every prompt token and all but the last generated token of each request was fed once
    assert stats.prefill_tokens + stats.decode_tokens == 55 + 3 * 5 and stats.steps > 6
    # what a request draws does not depend on its company: alone it gets the same tokens
    engine2 = ti.Engine.from_folder(d, "float32", page_size=16, max_tokens=64, max_requests=1, max_seq=64)
    sched = ti.Scheduler(engine2.cache)
    for i, p in enumerate(prompts):
        sched.set_next_number(i)
        r = sched.add(p, 6, ti.SamplingParams(0.8, 0, 1.0, 123))
        from tinyinfer_amd.api import run_requests
        run_requests(engine2, sched)
        assert r.generated == want[i]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_greedy_generation_with_graphs_equals_eager(model_folders, dtype):
    """Decode steps replayed from captured graphs give the same logits bit for bit
    as eager steps, replay after replay, with eager steps in between (the
    reference checks the same: src/inference.cu:297-341)."""
    import tinyinfer_amd as ti
    d = model_folders("D", "bfloat16", True)
    prompts = [random_tokens(n, 333, 40 + n) for n in (21, 3, 50)]
    outs = {}
    for graph in (False, True):
        engine = ti.Engine.from_folder(d, dtype, page_size=16, max_tokens=384, max_requests=3, max_seq=128)
        outs[graph] = ti.generate_ids(engine, prompts, max_new_tokens=40, use_graph=graph, chunk_size=16,
                                      max_batched_tokens=24)
        if graph:
            assert engine.graph_keys(), "no graph was captured"
    assert outs[True] == outs[False]
    # logits bit for bit, several replays, eager work between them
    e1 = ti.Engine.from_folder(d, dtype, page_size=16, max_tokens=256, max_requests=2, max_seq=128)
    e2 = ti.Engine.from_folder(d, dtype, page_size=16, max_tokens=256, max_requests=2, max_seq=128)
    toks = {"x": random_tokens(70, 333, 1), "y": random_tokens(70, 333, 2)}
    for e in (e1, e2):
        e.step([ti.StepEntry("x", toks["x"][:30], [29]), ti.StepEntry("y", toks["y"][:9], [8])])
    fed = {"x": 30, "y": 9}
    for i in range(30):
        entries = [ti.StepEntry(r, [toks[r][fed[r]]], [0]) for r in ("x", "y")]
        a = e1.step(entries).clone()
        if i % 7 == 3:                         # an eager step through the graph engine as well
            b = e2.step(entries).clone()
        else:
            b = e2.step_graph(entries).clone()
        assert torch.equal(a, b), i
        for r in fed:
            fed[r] += 1


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_steps_of_a_repeated_shape_replay_from_graphs(model_folders, dtype):
    """A prompt that arrives in equal portions beside a decoding request repeats the shape of
    its step: the second time the shape is captured, from then on replayed.  Every step's
    logits equal those of an engine that runs eagerly, bit for bit, replay after replay, with
    eager steps (another shape, and the same one through `step`) in between; and a shape that
    comes once is never captured."""
    import tinyinfer_amd as ti
    d = model_folders("D", "bfloat16", True)
    e1 = ti.Engine.from_folder(d, dtype, page_size=16, max_tokens=512, max_requests=3, max_seq=256)
    e2 = ti.Engine.from_folder(d, dtype, page_size=16, max_tokens=512, max_requests=3, max_seq=256)
    toks = {"x": random_tokens(200, 333, 1), "y": random_tokens(60, 333, 2)}
    for e in (e1, e2):
        e.step([ti.StepEntry("y", toks["y"][:9], [8])])
    fed = {"x": 0, "y": 9}
    shape = None
    for i in range(14):
        entries = [ti.StepEntry("y", [toks["y"][fed["y"]]], [0]),
                   ti.StepEntry("x", toks["x"][fed["x"]:fed["x"] + 12], [0, 11])]
        a = e1.step(entries).clone()
        if i % 5 == 3:
            b = e2.step(entries).clone()               # the same shape, eagerly, between replays
        else:
            b = e2.step_graph(entries).clone()
        assert torch.equal(a, b), i
        fed["x"] += 12
        fed["y"] += 1
        shape = tuple((len(e.tokens), tuple(e.want)) for e in entries)
        if i == 6:                                     # another shape, once: eager, not captured
            odd = [ti.StepEntry("x", toks["x"][fed["x"]:fed["x"] + 5], [4])]
            assert torch.equal(e1.step(odd), e2.step_graph(odd))
            fed["x"] += 5
    assert shape in e2.graph_keys() and len([k for k in e2.graph_keys() if not isinstance(k, int)]) == 1
    assert not e1.graph_keys()
    # the captured shape with other requests in it: a new request takes the portion's place
    for e in (e1, e2):
        e.release("x")
    fed["z"] = 0
    toks["z"] = random_tokens(40, 333, 3)
    for i in range(3):
        entries = [ti.StepEntry("y", [toks["y"][fed["y"]]], [0]),
                   ti.StepEntry("z", toks["z"][fed["z"]:fed["z"] + 12], [0, 11])]
        assert torch.equal(e1.step(entries), e2.step_graph(entries)), i
        fed["z"] += 12
        fed["y"] += 1
    e2.cache.check()


def test_only_the_most_recent_step_shapes_keep_their_graphs(model_folders, monkeypatch):
    """With room for one shape's graph, two shapes in turn push one another out and are captured
    again; the logits stay those of eager steps."""
    import tinyinfer_amd as ti
    d = model_folders("D", "bfloat16", True)
    e1 = ti.Engine.from_folder(d, "bfloat16", page_size=16, max_tokens=512, max_requests=2, max_seq=256)
    e2 = ti.Engine.from_folder(d, "bfloat16", page_size=16, max_tokens=512, max_requests=2, max_seq=256, max_step_graphs=1)
    toks = random_tokens(240, 333, 9)
    fed = 0
    captured = set()
    for i in range(16):
        n = (7, 11)[(i // 2) % 2]                      # two steps of one shape, two of the other, ...
        entries = [ti.StepEntry("x", toks[fed:fed + n], [n - 1])]
        assert torch.equal(e1.step(entries), e2.step_graph(entries)), i
        fed += n
        shapes = [k for k in e2.graph_keys() if not isinstance(k, int)]
        assert len(shapes) <= 1
        captured |= set(shapes)
    assert len(captured) == 2


@pytest.mark.parametrize("graph", [False, True])
def test_a_step_takes_its_tokens_from_the_device(model_folders, graph):
    """A step may name its tokens by rows of the sampler's last call instead of ids: it is then
    launched before those ids are read.  Same logits bit for bit as the step that was given the
    ids, with the rows in another order than the entries, step after step."""
    import tinyinfer_amd as ti
    from tinyinfer_amd.engine import EngineError
    from tinyinfer_amd.sampling import Sampler, SamplingParams
    d = model_folders("D", "bfloat16", True)
    make = lambda: ti.Engine.from_folder(d, "bfloat16", page_size=16, max_tokens=384, max_requests=3, max_seq=128)
    e1, e2 = make(), make()
    assert e2.feedback_rows == 3
    s1, s2 = Sampler(e1.ops), Sampler(e2.ops)
    prompts = {"x": random_tokens(30, 333, 1), "y": random_tokens(9, 333, 2), "z": random_tokens(17, 333, 3)}
    names = ["x", "y", "z"]
    first = [ti.StepEntry(r, prompts[r], [len(prompts[r]) - 1]) for r in names]
    params = [SamplingParams(), SamplingParams(0.9, 5, 0.95, 11), SamplingParams()]
    run = lambda e, entries: e.step_graph(entries) if graph else e.step(entries)
    ids = s1.sample(e1.step(first), params, [0, 1, 2], [0, 0, 0])
    ticket = s2.sample_async(e2.step(first), params, [0, 1, 2], [0, 0, 0], feed=e2)
    history = [ids]
    for i in range(1, 24):
        order = [2, 0, 1] if i % 2 else [1, 2, 0]              # entries in another order than the sampler's rows
        a = run(e1, [ti.StepEntry(names[k], [ids[k]], [0]) for k in order])
        b = run(e2, [ti.StepEntry(names[k], [ti.token_from_feedback(k)], [0]) for k in order])
        back = [order.index(k) for k in range(3)]              # row of request k in this step's logits
        a = a[back].contiguous()
        b_rows = b[back].contiguous()
        ids = s1.sample(a, params, [0, 1, 2], [i] * 3)
        late = s2.collect(ticket)                               # the ids of the step before, read after this step's launch
        assert late == history[-1], i
        assert torch.equal(a, b_rows), i
        ticket = s2.sample_async(b_rows, params, [0, 1, 2], [i] * 3, feed=e2)
        history.append(ids)
    assert s2.collect(ticket) == ids
    with pytest.raises(EngineError, match="feedback"):
        e2.step([ti.StepEntry("x", [ti.token_from_feedback(3)], [0])])
    e2.cache.check()


@pytest.mark.parametrize("dtype,graph", [("float32", False), ("float32", True), ("bfloat16", True)])
def test_steps_launched_ahead_change_no_token(model_folders, dtype, graph):
    """While every running request decodes, `run_requests` launches the next step before it has
    read the last one's ids.  Nothing that is generated changes: requests of different lengths,
    prompts in portions, temperature beside greedy, requests that an end-of-generation id stops in
    the middle (their row in the step launched ahead runs for nothing), a callback per token."""
    import tinyinfer_amd as ti
    from tinyinfer_amd.api import run_requests
    d = model_folders("D", "bfloat16", True)
    prompts = [random_tokens(n, 333, 90 + n) for n in (21, 3, 50, 8)]
    budgets = [40, 17, 28, 40]
    sampling = [ti.SamplingParams(), ti.SamplingParams(0.8, 20, 0.9, 7), ti.SamplingParams(), ti.SamplingParams(1.1, 0, 1.0, 3)]

    def run(ahead, eos):
        engine = ti.Engine.from_folder(d, dtype, page_size=16, max_tokens=512, max_requests=4, max_seq=128)
        sched = ti.Scheduler(engine.cache, max_batched_tokens=24, chunk_size=16)
        reqs = [sched.add(p, n, sp, eos) for p, n, sp in zip(prompts, budgets, sampling)]
        heard = {r.number: [] for r in reqs}
        stats = ti.GenerationStats()
        run_requests(engine, sched, stats=stats, on_token=lambda r, t: heard[r.number].append(t), use_graph=graph,
                     run_ahead=ahead)
        assert all(heard[r.number] == list(r.generated) for r in reqs)
        assert not engine.cache.live_requests()
        engine.cache.check()
        return [list(r.generated) for r in reqs], [r.finish_reason for r in reqs], stats

    plain_run, reasons, st0 = run(False, [])
    ahead_run, reasons1, st1 = run(True, [])
    assert ahead_run == plain_run and reasons1 == reasons == ["length"] * 4
    assert [len(g) for g in plain_run] == budgets
    assert st1.steps == st0.steps and st1.decode_tokens == st0.decode_tokens
    assert st0.steps_ahead == 0 and st1.steps_ahead >= 10
    if dtype == "float32":
        # ids that stop the first and the third request in the middle, at different steps
        eos = [plain_run[0][25], plain_run[2][11]]
        cut, why, st2 = run(False, eos)
        cut1, why1, st3 = run(True, eos)
        assert cut1 == cut and why1 == why and why.count("eos") >= 2
        assert st3.decode_tokens >= st2.decode_tokens           # rows that ran for nothing are counted
        assert st3.steps_ahead >= 10


def test_preemption_recomputes_and_changes_nothing(model_folders):
    """With too few pages the youngest request gives way and is fed again later;
    in 32-bit the tokens are the ones a roomy pool gives."""
    import tinyinfer_amd as ti
    d = model_folders("B", "bfloat16", True)
    prompts = [random_tokens(n, 1000, 70 + n) for n in (12, 12, 9)]
    roomy = ti.Engine.from_folder(d, "float32", page_size=4, max_tokens=256, max_requests=3, max_seq=48)
    want = ti.generate_ids(roomy, prompts, max_new_tokens=20, temperature=0.7, seed=5)
    tight = ti.Engine.from_folder(d, "float32", page_size=4, max_tokens=64, max_requests=3, max_seq=48)
    stats = ti.GenerationStats()
    got = ti.generate_ids(tight, prompts, max_new_tokens=20, temperature=0.7, seed=5, stats=stats)
    assert stats.preemptions > 0
    assert got == want
    assert not tight.cache.live_requests()
    tight.cache.check()


def test_eos_and_length(model_folders):
    import tinyinfer_amd as ti
    d = model_folders("A", "float32")
    prompt = random_tokens(6, 256, 3)
    engine = ti.Engine.from_folder(d, "float32", max_tokens=64, max_requests=1)
    full = ti.generate_ids(engine, [prompt], max_new_tokens=10)[0]
    assert len(full) == 10
    cut = ti.generate_ids(engine, [prompt], max_new_tokens=10, eos_token_ids=[full[4]])[0]
    assert cut == full[:full.index(full[4])]              # the end token itself is not emitted


def test_command_line(model_folders, tmp_path):
    d = model_folders("A", "float32")
    cfg, w = read_folder(d)
    p1, p2 = random_tokens(5, 256, 1), random_tokens(9, 256, 2)
    f = tmp_path / "prompts.txt"
    f.write_text(" ".join(map(str, p2)) + "\r\n\n")
    run = subprocess.run([sys.executable, os.path.join(ROOT, "bin", "tinyinfer"), "-m", d, "-n", "5",
                          "-p", ",".join(map(str, p1)), "-f", str(f), "--dtype", "float32", "--max-seq", "64"],
                         capture_output=True, text=True, timeout=300)
    assert run.returncode == 0, run.stderr
    lines = run.stdout.strip().split("\n")
    assert lines[0] == "==================== prompt 0 ===================="
    assert lines[1] == "[prompt] " + ",".join(map(str, p1))
    assert lines[2] == "[output] " + " ".join(map(str, plain_generate(cfg, w, p1, 5)))
    assert lines[5] == "[output] " + " ".join(map(str, plain_generate(cfg, w, p2, 5)))
    assert "main: prefill:" in run.stderr and "tok/s" in run.stderr
    bad = subprocess.run([sys.executable, os.path.join(ROOT, "bin", "tinyinfer"), "-m", d, "--nonsense"],
                         capture_output=True, text=True, timeout=120)
    assert bad.returncode == 1 and "usage:" in bad.stderr


def test_command_line_options(tmp_path):
    """`--random-weights --seed` from a folder with config.json alone, `--num-pages`, `--cuda-graph`, `-t`, `--top-k`,
    `--verbose`: the tokens are the plain model's on the weights `write_model_folder` writes for that seed, drawn with
    the same temperature, cut and seed; --verbose prints the first five and the five largest logits behind each prompt
    (src/main.cpp:136-158,233-249)."""
    import json
    import tinyinfer_amd as ti
    cfg = CONFIGS["A"]
    bare = tmp_path / "bare"
    bare.mkdir()
    (bare / "config.json").write_text(json.dumps(cfg))
    full = str(tmp_path / "full")
    ti.write_model_folder(full, cfg, seed=9, dtype="float32")
    _, w = read_folder(full)
    p1, p2 = random_tokens(7, 256, 11), random_tokens(21, 256, 12)
    exe = [sys.executable, os.path.join(ROOT, "bin", "tinyinfer")]
    common = ["-m", str(bare), "--random-weights", "--seed", "9", "--dtype", "float32", "--max-seq", "48", "--num-pages", "6",
              "-p", " ".join(map(str, p1)), "-p", " ".join(map(str, p2))]
    greedy = subprocess.run(exe + common + ["-n", "8", "--cuda-graph", "--verbose"], capture_output=True, text=True, timeout=300)
    assert greedy.returncode == 0, greedy.stderr
    lines = greedy.stdout.strip().split("\n")
    assert lines[2] == "[output] " + " ".join(map(str, plain_generate(cfg, w, p1, 8)))
    assert lines[5] == "[output] " + " ".join(map(str, plain_generate(cfg, w, p2, 8)))
    assert "[hip-graph: on]" in greedy.stderr
    for s, p in enumerate((p1, p2)):
        row = plain.forward(w, cfg, p)[-1]
        shown = [ln for ln in greedy.stderr.split("\n") if ln.startswith(f"prefill logits seq {s} (first 5, top 5):")]
        assert len(shown) == 1, greedy.stderr
        first, top = shown[0].split(":", 1)[1].split(" | top5:")
        assert np.allclose([float(v) for v in first.split()], row[:5], atol=2e-3)
        ids = [int(t.split("(")[0]) for t in top.split()]
        assert ids == [int(i) for i in np.lexsort((np.arange(row.size), -row))[:5]], (ids, shown)
    # two pages of 16 tokens instead of six, for requests of 15 and 29 tokens: they cannot both be live; the tokens stay
    tight = subprocess.run(exe + ["-m", str(bare), "--random-weights", "--seed", "9", "--dtype", "float32", "--max-seq", "48",
                                  "--num-pages", "2", "-n", "8", "-p", " ".join(map(str, p1)), "-p", " ".join(map(str, p2))],
                           capture_output=True, text=True, timeout=300)
    assert tight.returncode == 0 and tight.stdout == greedy.stdout, tight.stderr
    drawn = subprocess.run(exe + common + ["-n", "6", "-t", "0.8", "--top-k", "4", "--top-p", "0.9"], capture_output=True, text=True,
                           timeout=300)
    assert drawn.returncode == 0, drawn.stderr
    lines = drawn.stdout.strip().split("\n")
    for s, p in enumerate((p1, p2)):
        want = plain_generate(cfg, w, p, 6, number=s, temperature=0.8, top_k=4, top_p=0.9, seed=9)
        assert lines[3 * s + 2] == "[output] " + " ".join(map(str, want))
    none = subprocess.run(exe + ["-m", str(bare), "-n", "2", "-p", "1 2 3", "--dtype", "float32"], capture_output=True, text=True,
                          timeout=300)
    assert none.returncode == 1 and "safetensors" in none.stderr          # no weights and no --random-weights


def test_smoke_entry():
    sys.path.insert(0, ROOT)
    import __graft_entry__
    __graft_entry__.smoke()


def test_operator_selftest_of_the_command_line():
    """TINY_SELFTEST=1 runs every kernel against a CPU computation; the exit code counts failures."""
    env = dict(os.environ, TINY_SELFTEST="1")
    run = subprocess.run([sys.executable, os.path.join(ROOT, "bin", "tinyinfer")], capture_output=True, text=True,
                         timeout=300, env=env)
    assert run.returncode == 0, run.stdout + run.stderr
    assert "[selftest] all cases passed" in run.stdout
    assert run.stdout.count(" ok") >= 20 and "FAIL" not in run.stdout
