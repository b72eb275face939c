"""The engine against the plain implementation under every way of cutting the work."""

import ctypes
import json
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

import helpers

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# prompt + decoded lengths of the two tiny workloads (5, 17, 31 -> 16 tokens; 1, 9, 40, 64, 100 -> 24),
# as given token sequences, plus one long request each
LENGTHS = {"A": [5 + 16, 17 + 16, 31 + 16, 90, 12, 60, 29], "B": [1 + 24, 9 + 24, 40 + 24, 64 + 24, 100 + 24, 200],
           "C": [5 + 16, 17 + 16, 31 + 16, 90, 12, 60], "D": [25, 33, 64, 88, 124, 150]}


def _requests(which, config):
    return {f"r{i}": helpers.random_tokens(n, config["vocab_size"], 100 + i)
            for i, n in enumerate(LENGTHS[which])}


def _engine(folder, dtype, page_size, pages, max_step_tokens=512):
    from pagedserve_amd.engine import Engine
    from pagedserve_amd.model import load_model

    model, _ = load_model(folder, dtype=dtype, device="cuda")
    return Engine(model, num_pages=pages, page_size=page_size, max_requests=8,
                  max_step_tokens=max_step_tokens)


@pytest.fixture(scope="module")
def folders(tmp_path_factory):
    base = tmp_path_factory.mktemp("models")
    return {which: helpers.tiny_folder(base, which) for which in helpers.TINY}


@pytest.fixture(scope="module")
def references(folders):
    out = {}
    for which, (folder, config, _) in folders.items():
        requests = _requests(which, config)
        for bf16 in (False, True):
            out[(which, bf16)] = {rid: helpers.plain_logits(folder, tokens, bfloat16=bf16)
                                  for rid, tokens in requests.items()}
    return out


CUTS = {
    "whole": helpers.trace_whole,
    "tail_decoded": helpers.trace_tail_decoded,
    "portions": helpers.trace_portions,
    "mixed": helpers.trace_mixed,
}


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("which", list(helpers.TINY))
@pytest.mark.parametrize("cut", list(CUTS))
def test_cuts_match_plain(folders, references, which, dtype, cut):
    """A: heads of 16; B: heads of 48, inverse-layer scaling, erf GELU; C: the sizes of the
    reference's own test (heads of 8) with a head that is not tied; D: heads of 20, widths that
    are no multiple of 8, pages of 12 tokens."""
    folder, config, page_size = folders[which]
    requests = _requests(which, config)
    steps = CUTS[cut](requests)
    # exactly the pages that the live requests hold at their peak, each request's tokens
    # rounded up to whole pages: pages are used again
    budget = helpers.live_token_budget(steps, round_to=page_size)
    engine = _engine(folder, dtype, page_size, pages=budget // page_size)
    holders = {}
    rows = helpers.replay_in_process(engine, steps, page_holders=holders)
    engine.cache.check_invariants()
    assert not engine.cache.requests
    assert engine.cache.pools[0].peak_allocated == budget // page_size
    # some physical page went from one request to another
    assert any(len(owners) > 1 for owners in holders.values())
    assert len(rows) == sum(len(tokens) for tokens in requests.values())
    error, scale, where = helpers.max_error(rows, references[(which, dtype == "bfloat16")])
    print(f"cut {cut} {which} {dtype}: error/scale {error / scale:.2e}")
    assert error <= helpers.TOLERANCE[dtype] * scale, (error, scale, where)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_trace_run_program(folders, references, tmp_path, dtype):
    """bin/trace_run as a user calls it: JSON lines in, <step>.f32 files and 'done' lines out."""
    folder, config, page_size = folders["B"]
    requests = _requests("B", config)
    steps = helpers.trace_mixed(requests, seed=3)
    budget = helpers.live_token_budget(steps)
    out_dir = tmp_path / "out"
    process = subprocess.run(
        [sys.executable, os.path.join(ROOT, "bin", "trace_run"), "--model", folder, "--dtype", dtype,
         "--out", str(out_dir), "--max-tokens", str(budget)],
        input="\n".join(json.dumps(step) for step in steps) + "\n", capture_output=True, text=True,
        timeout=600)
    assert process.returncode == 0, process.stderr[-2000:]
    done = [line for line in process.stdout.splitlines() if line.startswith("done ")]
    assert done == [f"done {step['step']}" for step in steps]
    reference = references[("B", dtype == "bfloat16")]
    held = {}
    worst, scale = 0.0, 0.0
    for step in steps:
        wanted = sum(len(entry["want"]) for entry in step["entries"])
        values = np.fromfile(out_dir / f"{step['step']}.f32", dtype="<f4").reshape(wanted, config["vocab_size"])
        row = 0
        for entry in step["entries"]:
            start = held.get(entry["id"], 0)
            for place in entry["want"]:
                expected = reference[entry["id"]][start + place]
                worst = max(worst, float((torch.from_numpy(values[row]).double() - expected).abs().max()))
                scale = max(scale, float(expected.abs().max()))
                row += 1
            held[entry["id"]] = start + len(entry["tokens"])
    assert worst <= helpers.TOLERANCE[dtype] * scale, (worst, scale)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_graph_replay_matches_direct_launches(folders, references, dtype):
    """Decode steps replayed from a captured HIP graph give the logits of direct launches, on
    every replay, with other work of the engine (a prompt portion, a batch of another size, a
    finished request whose pages go to a new one) between the replays."""
    from pagedserve_amd.engine import StepEntry

    folder, config, page_size = folders["B"]
    requests = _requests("B", config)
    outputs = {}
    for use_graphs in (False, True):
        names = ["r2", "r3", "r4"]
        from pagedserve_amd.engine import Engine
        from pagedserve_amd.model import load_model

        model, _ = load_model(folder, dtype=dtype)
        engine = Engine(model, num_pages=30, page_size=page_size, max_requests=4,
                        max_step_tokens=128, use_graphs=use_graphs)
        rows = {}

        def run(entries):
            out = engine.step(entries)
            values = out.logits.double().cpu()
            for index, key in enumerate(out.rows):
                rows[key] = values[index]

        cursor = {}
        for name in names:
            run([StepEntry(name, requests[name][:20], list(range(20)))])
            cursor[name] = 20
        for turn in range(30):
            live = [name for name in names if cursor[name] < len(requests[name])]
            batch = live if turn % 5 else live[:1]
            run([StepEntry(name, [requests[name][cursor[name]]], [0]) for name in batch])
            for name in batch:
                cursor[name] += 1
            if turn == 7:       # a prompt portion of another request between two replays
                run([StepEntry("r1", requests["r1"][:9], list(range(9)))])
                engine.finish("r1")
            if turn == 15:      # r2 ends; its pages go to a newcomer that joins the decode batch
                engine.finish("r2")
                names[0] = "r0"
                run([StepEntry("r0", requests["r0"][:3], [0, 1, 2])])
                cursor["r0"] = 3
        outputs[use_graphs] = rows
        if use_graphs:
            summary = engine.graph_summary()
            assert summary["captured_graphs"] >= 2 and summary["graph_replays"] >= 15, summary
            assert not summary["capture_failures"], summary
            assert all(nodes > 10 for nodes in summary["graph_nodes"].values())
    reference = references[("B", dtype == "bfloat16")]
    for rows in outputs.values():
        error, scale, where = helpers.max_error(rows, reference)
        assert error <= helpers.TOLERANCE[dtype] * scale, (error, scale, where)
    assert outputs[True].keys() == outputs[False].keys()
    worst = max(float((outputs[True][key] - outputs[False][key]).abs().max()) for key in outputs[True])
    assert worst <= helpers.TOLERANCE[dtype] * 0.2 * float(reference["r4"].abs().max())


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_graph_replay_of_mixed_steps(folders, references, dtype):
    """Steps of one layout that are no pure decode steps (a prompt portion beside a decoded
    token and a two-token portion) are recorded after they have come back a few times; every
    replay gives the logits of the plain computation, with other layouts and a finished
    request's reused pages between the replays."""
    from pagedserve_amd.engine import Engine, StepEntry
    from pagedserve_amd.model import load_model

    folder, config, page_size = folders["B"]
    requests = _requests("B", config)
    model, _ = load_model(folder, dtype=dtype)
    engine = Engine(model, num_pages=30, page_size=page_size, max_requests=4, max_step_tokens=128)
    engine.record_after = 3       # (the default waits for many more returns)
    rows = {}

    def run(entries):
        out = engine.step(entries)
        values = out.logits.double().cpu()
        for index, key in enumerate(out.rows):
            rows[key] = values[index]

    cursor = {"r4": 0, "r3": 0, "r2": 0}
    run([StepEntry("r3", requests["r3"][:11], list(range(11)))])
    cursor["r3"] = 11
    replays_before = 0
    for turn in range(12):
        # the same layout every turn: 7 tokens of r4's prompt, 1 token of r3, 2 tokens of r2
        entries = [StepEntry("r4", requests["r4"][cursor["r4"]:cursor["r4"] + 7], [0, 6]),
                   StepEntry("r3", [requests["r3"][cursor["r3"]]], [0]),
                   StepEntry("r2", requests["r2"][cursor["r2"]:cursor["r2"] + 2], [1])]
        run(entries)
        cursor["r4"] += 7
        cursor["r3"] += 1
        cursor["r2"] += 2
        if turn == 6:    # another layout, and pages that change hands, between two replays
            run([StepEntry("r1", requests["r1"][:9], list(range(9)))])
            engine.finish("r1")
            run([StepEntry("r0", requests["r0"][:1], [0])])
            engine.finish("r0")
    summary = engine.graph_summary()
    assert summary["captured_graphs"] >= 1 and summary["graph_replays"] >= 6, summary
    assert not summary["capture_failures"], summary
    error, scale, where = helpers.max_error(rows, references[("B", dtype == "bfloat16")])
    assert error <= helpers.TOLERANCE[dtype] * scale, (error, scale, where)
    engine.cache.check_invariants()


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_many_live_requests_match_plain(tmp_path, dtype):
    """Up to 24 live requests with portions of 1 to 23 tokens: steps of 17 to 64 tokens and
    more, where the bfloat16 path keeps activations in the skinny products' operand order
    (widths that are multiples of 64, unlike the two tiny configurations), against the plain
    implementation like every other cut."""
    from pagedserve_amd.engine import Engine
    from pagedserve_amd.model import load_model

    config = {"architectures": ["GPT2LMHeadModel"], "model_type": "gpt2", "layer_norm_epsilon": 1e-5,
              "activation_function": "gelu", "tie_word_embeddings": True, "n_layer": 2, "n_embd": 128,
              "n_head": 2, "n_inner": 320, "vocab_size": 1000, "n_positions": 256}
    folder = str(tmp_path / "wide")
    helpers.write_folder(folder, config, helpers.lively_tensors(config, 301))
    g = torch.Generator().manual_seed(11)
    requests = {f"m{i}": helpers.random_tokens(int(torch.randint(3, 90, (1,), generator=g)), 1000, 4000 + i)
                for i in range(30)}
    reference = {rid: helpers.plain_logits(folder, tokens, bfloat16=dtype == "bfloat16")
                 for rid, tokens in requests.items()}
    model, _ = load_model(folder, dtype=dtype)
    steps = helpers.trace_mixed(requests, max_live=24, portion=(5, 23, 1, 9, 17), decode_tail=7, seed=5)
    sizes = {sum(len(e["tokens"]) for e in step["entries"]) for step in steps}
    assert any(17 <= size <= 64 for size in sizes) and any(size <= 16 for size in sizes)
    pages = -(-helpers.live_token_budget(steps) // 16)
    engine = Engine(model, num_pages=pages, page_size=16, max_requests=24, max_step_tokens=512)
    rows = helpers.replay_in_process(engine, steps)
    error, scale, where = helpers.max_error(rows, reference)
    assert error <= helpers.TOLERANCE[dtype] * scale, (dtype, error, scale, where)
    engine.cache.check_invariants()


@pytest.mark.parametrize("num_layers,dtype", [(2, "float32"), (6, "float32"), (2, "bfloat16"),
                                              (6, "bfloat16")])
def test_reference_test_configuration(tmp_path, num_layers, dtype):
    """The configuration and the steps of the reference's own GPT-2 test
    (testing/test_gpt2.py:13-68): vocabulary 41, 16 positions, width 16, two heads of 8, inner
    width 32, 2 and 6 layers, pages of 4; the prompt (4, 8, 15, 16) whole, then token 23
    decoded.  The reference compares with the library's model, in 32-bit; here the plain
    implementation stands in its place.

    Six layers in bfloat16: the 31 bfloat16 stores of activations between kernels (five a layer
    and the final norm, each a relative rounding of up to 2^-9) add up to 4.3e-3 of the largest
    logit here, where wider models with larger vocabularies stay near 2e-3: 41 logits of five
    rows have a largest value of two standard deviations, not of four or five, and the error is
    measured against it.  The tolerance is not widened for that.  This case is compared with the
    plain implementation that rounds the same stores (``plain_gpt2.ACTIVATION_STORAGE``: same
    formulas, the activations a bfloat16 engine writes to memory rounded as it writes them),
    with the tolerance of every other bfloat16 case (measured: 4.5e-8 of the largest logit
    against it, 4.3e-3 against the exact one: the engine's arithmetic is the plain one's, its
    stores are where the difference comes from).  The other configurations are not compared this
    way: a value that lands on the other side of a rounding boundary in one of the two moves a
    logit of a narrow model by a part in a thousand by itself, and the tiled attention also
    rounds its probabilities, so the two agree to 1e-4 ... 2e-3 there, no tighter than with the
    exact implementation."""
    config = {"architectures": ["GPT2LMHeadModel"], "model_type": "gpt2", "vocab_size": 41,
              "n_positions": 16, "n_embd": 16, "n_layer": num_layers, "n_head": 2, "n_inner": 32,
              "activation_function": "gelu_new", "bos_token_id": 0, "eos_token_id": 1}
    folder = str(tmp_path / "reference_config")
    helpers.write_folder(folder, config, helpers.lively_tensors(config, 7))
    prompt, following = [4, 8, 15, 16], 23
    rounds_stores = dtype == "bfloat16" and num_layers > 2
    expected = helpers.plain_logits(folder, prompt + [following], bfloat16=dtype == "bfloat16",
                                    stored_activations=rounds_stores)
    engine = _engine(folder, dtype, 4, pages=2, max_step_tokens=16)
    steps = [{"step": 0, "entries": [{"id": "request", "tokens": prompt, "want": [0, 1, 2, 3]}], "end": []},
             {"step": 1, "entries": [{"id": "request", "tokens": [following], "want": [0]}], "end": ["request"]}]
    rows = helpers.replay_in_process(engine, steps)
    error, scale, where = helpers.max_error(rows, {"request": expected})
    assert len(rows) == 5
    if rounds_stores:
        exact = helpers.plain_logits(folder, prompt + [following], bfloat16=True)
        print("six layers, bfloat16: against the plain implementation with rounded stores",
              f"{error / scale:.2e}, with exact activations {helpers.max_error(rows, {'request': exact})[0] / scale:.2e}")
    assert error <= helpers.TOLERANCE[dtype] * scale, (error, scale, where)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_more_layouts_than_recorded_graphs_are_kept(folders, references, dtype):
    """More step layouts than the engine keeps graphs for, each coming back often enough to be
    recorded, while decode steps replayed from a graph run between them: recorded layouts are
    dropped (their graphs destroyed only once nothing launched before can still be running) and
    every logit still matches the plain implementation."""
    from pagedserve_amd.engine import Engine, StepEntry
    from pagedserve_amd.model import load_model

    folder, config, page_size = folders["B"]
    requests = _requests("B", config)
    model, _ = load_model(folder, dtype=dtype)
    engine = Engine(model, num_pages=40, page_size=page_size, max_requests=4, max_step_tokens=128)
    engine.max_graphs = 3
    engine.record_after = 3
    rows = {}

    def run(entries):
        out = engine.step(entries)
        values = out.logits.double().cpu()
        for index, key in enumerate(out.rows):
            rows[key] = values[index]

    run([StepEntry("r5", requests["r5"][:60], list(range(60)))])
    decoded = 60
    for size in (2, 3, 4, 5, 6, 7):            # six layouts of a prompt portion, each four times
        for repeat in range(4):
            name = f"r{repeat % 4}"
            run([StepEntry(name, requests[name][:size], list(range(size)))])
            engine.finish(name)
            run([StepEntry("r5", [requests["r5"][decoded]], [0])])     # a replayed decode step
            decoded += 1
    summary = engine.graph_summary()
    assert summary["captures"] >= 7 and summary["evicted"] >= 4 and summary["captured_graphs"] <= 3, summary
    assert not summary["capture_failures"], summary
    error, scale, where = helpers.max_error(rows, references[("B", dtype == "bfloat16")])
    assert error <= helpers.TOLERANCE[dtype] * scale, (error, scale, where)
    torch.cuda.synchronize()
    engine.cache.check_invariants()


@pytest.mark.parametrize("live", [3, 20])
def test_greedy_tokens_are_the_argmax_of_the_logits(folders, live):
    """Greedy steps in bfloat16, replayed from a graph: the tokens that the step chooses are the
    columns of the largest logits of the same step.  With 20 requests decoding the head's own
    kernel chooses them (no sampling launch); with 3 the norm is fused into the head's product
    and the sampling kernel does."""
    from pagedserve_amd.engine import Engine, StepEntry
    from pagedserve_amd.model import load_model

    folder, config, page_size = folders["A"]
    model, _ = load_model(folder, dtype="bfloat16")
    engine = Engine(model, num_pages=24 * live, page_size=page_size, max_requests=live, max_step_tokens=64)
    prompts = {f"g{i}": helpers.random_tokens(3 + i % 5, config["vocab_size"], 700 + i) for i in range(live)}
    for name, prompt in prompts.items():
        engine.step([StepEntry(name, prompt, [])])
    last = {name: [prompt[-1]] for name, prompt in prompts.items()}
    for step in range(8):
        entries = [StepEntry(name, last[name], [0]) for name in prompts]
        out = engine.step(entries, greedy=True)
        tokens = out.token_list()
        assert tokens == out.logits.argmax(dim=1).tolist(), step
        for name, token in zip(prompts, tokens):
            last[name] = [token]
    assert (engine.tokens_chosen_by_head > 0) == (live > 16)
    assert engine.graph_summary()["graph_replays"] >= 4
    torch.cuda.synchronize()
    assert int(engine._top_choice.keys.abs().sum()) == 0 and int(engine._top_choice.ticket.abs().sum()) == 0


@pytest.mark.parametrize("count", [0, 1, 3, 4, 1023, 1024, 1025, 70001])
@pytest.mark.parametrize("offset", [0, 1, 2])
def test_words_between_host_memory_and_the_device(count, offset):
    """Whole and ragged pieces, device buffers that do not start at 16 bytes, words behind the last one untouched;
    what the host writes between two copies is seen by the second; ordinary memory is refused."""
    from pagedserve_amd.ops import kernels

    words = kernels.HostWords(70016)
    device = torch.full((70016 + offset,), -7, dtype=torch.int32, device="cuda")[offset:]
    for turn in range(2):
        words.tensor[:] = torch.arange(70016, dtype=torch.int32) * (turn + 3) - 50000
        device.fill_(-7)
        words.to_device(device, count)
        torch.cuda.synchronize()
        assert torch.equal(device[:count].cpu(), words.tensor[:count]) and int((device[count:] != -7).sum()) == 0
        device += 1
        expected = words.tensor.clone()
        expected[:count] += 1
        words.from_device(device, count)
        torch.cuda.synchronize()
        assert torch.equal(words.tensor, expected)
    with pytest.raises(kernels.KernelError):
        words.to_device(device[:3], 4)
    with pytest.raises(kernels.KernelError):
        words.to_device(device.float(), 4)
    # a part of the buffer, on its own
    part = kernels.HostWords(8 + offset, words, 64)
    before = words.tensor.clone()
    device.fill_(11)
    part.from_device(device, 5)
    torch.cuda.synchronize()
    before[64:69] = 11
    assert torch.equal(words.tensor, before) and torch.equal(part.tensor, before[64:72 + offset])
    with pytest.raises(kernels.KernelError):
        kernels.HostWords(17, words, 70000)
    if count == 1 and offset == 0:
        plain = torch.zeros(64, dtype=torch.int32)
        with pytest.raises(kernels.KernelError):
            kernels._call("ps_host_address", plain.data_ptr(),
                          ctypes.cast(ctypes.pointer(ctypes.c_void_p()), ctypes.c_void_p))
        torch.cuda.synchronize()


def _toy_engine():
    from pagedserve_amd.engine import Engine
    from pagedserve_amd.model import random_model

    model, _ = random_model({"architectures": ["GPT2LMHeadModel"], "n_layer": 2, "n_embd": 64, "n_head": 4,
                             "n_inner": 256, "vocab_size": 512, "n_positions": 128, "layer_norm_epsilon": 1e-5,
                             "activation_function": "gelu_new", "eos_token_id": None}, dtype="bfloat16")
    return Engine(model, num_pages=32, page_size=8, max_requests=2, max_step_tokens=64)


def test_an_engine_that_goes_with_work_in_flight_keeps_its_pinned_memory():
    """The pinned buffers of an engine are accessed by kernels.  They are not handed to anyone else while its
    stream still has work, and nobody waits for that."""
    import gc
    import weakref

    from pagedserve_amd.engine import StepEntry

    engine = _toy_engine()
    for step in range(4):
        out = engine.step([StepEntry("a", [5 + step], [0])], greedy=True)
    torch.cuda.synchronize()
    blocks = [words.tensor.untyped_storage() for words in engine._meta_words + engine._tokens_words]
    mine = {(block.data_ptr(), block.nbytes() // 4) for block in blocks}
    stream, gone = engine.stream, weakref.ref(engine)
    # (as many free blocks as are asked for below: memory from the system would wait for the device)
    spare = [torch.empty(count, dtype=torch.int32, pin_memory=True) for _, count in mine]
    del spare
    gc.collect()
    with torch.cuda.stream(stream):
        torch.cuda._sleep(400_000_000)      # (a tenth of a second at least)
        for words in engine._meta_words + engine._tokens_words:
            words.from_device(engine._tokens, 1)
    del engine, out, blocks, words
    assert gone() is None
    others = [torch.empty(count, dtype=torch.int32, pin_memory=True) for _, count in mine]
    assert not stream.query(), "the work was over too soon for this test"
    assert not {b.data_ptr() for b in others} & {address for address, _ in mine}
    stream.synchronize()


def test_an_engine_that_goes_inside_a_capture_leaves_it_whole():
    """The collector may end an engine at any place, also between the launches that another one records."""
    import gc
    import weakref

    from pagedserve_amd.engine import StepEntry
    from pagedserve_amd.ops import kernels

    engine = _toy_engine()
    for step in range(3):
        engine.step([StepEntry("a", [5 + step], [0])], greedy=True)
    engine.ring = engine          # only the collector ends it
    gone = weakref.ref(engine)
    x = torch.randn(4, 64, device="cuda")
    gamma, out = torch.ones(64, device="cuda"), torch.zeros(4, 64, device="cuda")
    side, graph = torch.cuda.Stream(), kernels.StepGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        kernels.StepGraph.begin()
        kernels.norm(x, gamma, None, 1e-5, out)
        del engine
        gc.collect()
        graph.end()
        graph.launch()
    torch.cuda.synchronize()
    assert gone() is None and graph.nodes == 1
    torch.testing.assert_close(out, torch.nn.functional.layer_norm(x, (64,), gamma), atol=1e-5, rtol=1e-5)
    graph.destroy()
