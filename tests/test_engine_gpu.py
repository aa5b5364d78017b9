"""The engine against the plain implementation under every way of cutting the
work, in float32 and in bfloat16, for three tiny configurations and for some drawn at random."""
import pytest
import torch

import cuttings
from engine_helpers import (TOL, first_mismatch, load_runner, make_folder, plain_logits,
                            random_sequences, replay)
from tiny_configs import tiny

pytestmark = pytest.mark.gpu

LENGTHS = {"A": [5, 9, 13, 17, 70, 41], "B": [31, 70, 100, 45, 64, 129], "C": [33, 80, 16, 97, 50]}
DTYPES = [torch.float32, torch.bfloat16]


@pytest.fixture(scope="module")
def cases(tmp_path_factory, gpu_device):
    out = {}
    for name in ("A", "B", "C"):
        folder, page = make_folder(tmp_path_factory, name, seed=11)
        cfg = tiny(name)[0]
        seqs = random_sequences(cfg["vocab_size"], LENGTHS[name], seed=5)
        want = {torch.float32: plain_logits(folder, seqs),
                torch.bfloat16: plain_logits(folder, seqs, torch.bfloat16)}
        out[name] = (folder, page, seqs, want)
    return out


def run_cutting(cases, name, dtype, steps, num_pages=None):
    folder, page, seqs, want = cases[name]
    if num_pages is None:
        num_pages = -(-cuttings.max_live_tokens(steps) // page)
    runner = load_runner(folder, dtype, page, num_pages)
    got = replay(runner, steps, seqs)
    bad = first_mismatch(got, want[dtype], TOL[dtype])
    assert bad is None, f"config {name} {dtype}: first wrong place (request, position, error) = {bad}"
    assert all(g.pool.num_free == g.pool.num_pages for g in runner.manager.paged)


@pytest.mark.parametrize("dtype", DTYPES, ids=["fp32", "bf16"])
@pytest.mark.parametrize("name", ["A", "B", "C"])
def test_whole(cases, name, dtype):
    run_cutting(cases, name, dtype, cuttings.whole(cases[name][2]))


@pytest.mark.parametrize("dtype", DTYPES, ids=["fp32", "bf16"])
@pytest.mark.parametrize("name", ["A", "B", "C"])
def test_last_tokens_one_by_one(cases, name, dtype):
    run_cutting(cases, name, dtype, cuttings.tail_decode(cases[name][2], 32))


@pytest.mark.parametrize("dtype", DTYPES, ids=["fp32", "bf16"])
@pytest.mark.parametrize("name", ["A", "B", "C"])
def test_portions_of_changing_size(cases, name, dtype):
    run_cutting(cases, name, dtype, cuttings.portions(cases[name][2]))


@pytest.mark.parametrize("dtype", DTYPES, ids=["fp32", "bf16"])
@pytest.mark.parametrize("name", ["A", "B", "C"])
def test_mixed_with_page_reuse(cases, name, dtype):
    seqs = cases[name][2]
    steps = cuttings.mixed(seqs, seed=3, max_live=4)
    page = cases[name][1]
    need = cuttings.max_live_tokens(steps, round_to=page) // page
    total = sum(-(-len(t) // page) for t in seqs.values())
    assert need < total, "the pool must be too small to hold all requests at once"
    run_cutting(cases, name, dtype, steps, need)


@pytest.mark.parametrize("dtype", DTYPES, ids=["fp32", "bf16"])
@pytest.mark.parametrize("name", ["A", "B", "C"])
def test_cuttings_replayed_as_graphs(cases, name, dtype):
    """The same cuttings with decode steps and single portions replayed as HIP graphs (their
    padded layouts of a step against the plain model, not against the eager layout): the last
    tokens one by one, portions of changing size, and the mixed trace. A replayed portion has
    one wanted place, so only the last row of every entry is asked for."""
    from engine_helpers import first_wrong_row, load_graph_runner, plain_rows, replay_wanted
    folder, page, seqs, _ = cases[name]
    for steps in (cuttings.tail_decode(seqs, 32), cuttings.portions(seqs), cuttings.mixed(seqs, seed=3)):
        for st in steps:
            for e in st["entries"]:
                e["want"] = e["want"][-1:]
        places = cuttings.wanted_places(steps)
        want = plain_rows(folder, seqs, places, dtype)
        runner = load_graph_runner(folder, dtype, page, -(-cuttings.max_live_tokens(steps) // page),
                                   max_model_len=160, max_num_seqs=4)
        got = replay_wanted(runner, steps)
        bad = first_wrong_row(got, want, places, TOL[dtype])
        assert bad is None, f"config {name} {dtype}: first wrong place (request, position, error) = {bad}"
        assert runner.graphs.buckets and runner.portion_graphs.buckets


@pytest.mark.parametrize("dtype", DTYPES, ids=["fp32", "bf16"])
def test_a_replayed_portion_gives_the_logits_of_any_one_of_its_rows(cases, dtype):
    """A replayed step with a portion computes the logits of one row of the portion: the row the
    entry names, not only its last (first, a middle and the last row of portions of changing
    size, alone and beside decoded tokens of another request), against the plain model."""
    from engine_helpers import first_wrong_row, load_graph_runner, plain_rows, replay_wanted
    folder, page, seqs, _ = cases["B"]
    again = {r + "_again": t for r, t in seqs.items()}        # the same requests under other names
    steps = cuttings.mixed(seqs, seed=11, max_live=3) + cuttings.portions(again, sizes=(9, 40, 2, 17))
    for i, st in enumerate(steps):
        st["step"] = i
        for j, e in enumerate(st["entries"]):
            n = len(e["tokens"])
            e["want"] = [(0, n // 2, n - 1)[(i + j) % 3]] if n > 1 else [0]
    assert any(e["want"] == [0] and len(e["tokens"]) > 2 for st in steps for e in st["entries"])
    both = dict(seqs, **again)
    places = cuttings.wanted_places(steps)
    want = plain_rows(folder, both, places, dtype)
    runner = load_graph_runner(folder, dtype, page, -(-cuttings.max_live_tokens(steps) // page),
                               max_model_len=160, max_num_seqs=4)
    got = replay_wanted(runner, steps)
    bad = first_wrong_row(got, want, places, TOL[dtype])
    assert bad is None, f"{dtype}: first wrong place (request, position, error) = {bad}"
    assert runner.portion_graphs.buckets


@pytest.mark.parametrize("dtype", DTYPES, ids=["fp32", "bf16"])
@pytest.mark.parametrize("name", ["A", "B", "C"])
def test_steps_that_want_few_of_their_rows(cases, name, dtype):
    """Steps of several prompts that want none, one, two (in falling order) or all but one of a prompt's rows: the last
    block gives those rows alone, in the order asked for, and what it keeps of the other rows is read by the next step."""
    from pytriton_llama_amd.engine.batch import StepEntry
    folder, page, seqs, want = cases[name]
    seqs = dict(list(seqs.items())[:4])
    runner = load_runner(folder, dtype, page, sum(-(-len(t) // page) for t in seqs.values()))
    cut = {r: len(t) // 2 for r, t in seqs.items()}
    first = [[], [cut["r1"] - 1], [cut["r2"] - 1, 0], list(range(1, cut["r3"]))]
    got = {r: [] for r in seqs}
    places = {r: [] for r in seqs}
    for step in (0, 1):
        wants = first if step == 0 else [[len(t) - cut[r] - 1] for r, t in seqs.items()]
        entries = [StepEntry(r, t[:cut[r]] if step == 0 else t[cut[r]:], w) for (r, t), w in zip(seqs.items(), wants)]
        logits = runner.step(entries).float().cpu()
        assert logits.shape[0] == sum(len(w) for w in wants)
        for (r, _), w in zip(seqs.items(), wants):
            got[r].append(logits[:len(w)])
            logits = logits[len(w):]
            places[r] += [p + step * cut[r] for p in w]
    for r, g in got.items():
        g, plain = torch.cat(g), want[dtype][r]
        err = float((g - plain[places[r]]).abs().max()) / float(plain.abs().max())
        assert err <= TOL[dtype], f"config {name} {dtype} {r}: off by {err}"


@pytest.mark.parametrize("lengths", [(40, 25), (40, 24), (70, 45, 1), (129, 3, 64, 100), (300, 280, 7), (400, 390, 311)])
def test_steps_of_prompts_in_native_code_give_the_bits_of_the_parts(cases, lengths, monkeypatch):
    """Steps of several prompts: native calls between the attentions (from 65 rows on) launch what the parts launch:
    equal logits, and equal ones in the next step, which reads the pages; rows where the tile products take all, some
    and none of the products, with and without a decoding request."""
    from pytriton_llama_amd.engine.batch import StepEntry
    from pytriton_llama_amd.models import prompt_steps
    folder, page = cases["B"][0], cases["B"][1]
    seqs = random_sequences(tiny("B")[0]["vocab_size"], lengths, seed=9)
    went = []
    native = prompt_steps.run

    def run(how):
        monkeypatch.setattr(prompt_steps, "run", how)
        runner = load_runner(folder, torch.bfloat16, page, sum(-(-len(t) // page) + 1 for t in seqs.values()))
        out = []
        for cut in (slice(0, None), slice(0, 2)):
            out.append(runner.step([StepEntry(r, t[cut], range(len(t[cut]))) for r, t in seqs.items()]).clone())
        return out

    def counted(*args):
        done = native(*args)
        went.append(done is not None)
        return done
    with_native, with_parts = run(counted), run(lambda *args: None)
    assert went == [sum(lengths) >= 65, False]
    assert all(torch.equal(a, b) for a, b in zip(with_native, with_parts))


@pytest.mark.parametrize("heads,kv_heads,head_dim,act", [(16, 4, 64, "silu"), (8, 2, 128, "gelu_tanh"), (16, 4, 80, "silu"),
                                                         (64, 4, 16, "silu")])
def test_native_steps_of_prompts_where_products_come_in_slices(tmp_path, heads, kv_heads, head_dim, act, monkeypatch, gpu_device):
    """As above, at widths whose output and down projections come as several float32 slices, a different number of each, in
    the place that q | k | v and gate | up share with them: numbers of rows with eight, four and two slices, and both sides of
    where a product goes to the library (576, 768 and 1,088 rows); head sizes of the matrix-core and of the vector attention."""
    from pytriton_llama_amd import ops
    from pytriton_llama_amd.engine.batch import StepEntry
    from pytriton_llama_amd.models import prompt_steps
    from pytriton_llama_amd.weights import write_random_model
    H, I = 1024, 4096
    cfg = dict(tiny("B")[0], hidden_size=H, num_attention_heads=heads, num_key_value_heads=kv_heads, head_dim=head_dim,
               intermediate_size=I, vocab_size=512)
    write_random_model(cfg, str(tmp_path), seed=6, dtype=torch.bfloat16, std=0.03)
    runner = load_runner(str(tmp_path), torch.bfloat16, 16, 256)
    assert {prompt_steps._plain(b) for b in runner.model.blocks} == {True}
    for b in runner.model.blocks:
        b.feed_forward.act = ops.GLU_GELU_TANH if act == "gelu_tanh" else ops.GLU_SILU
    native, went = prompt_steps.run, []

    def counted(*args):
        done = native(*args)
        went.append(done is not None)
        return done
    slices = set()
    for rows in (65, 130, 285, 532, 576, 577, 768, 769, 1088, 1089):
        o, down = ops.gemm_tile_splits(rows, H, heads * head_dim), ops.gemm_tile_splits(rows, H, I)
        slices |= {("o", o), ("down", down)} if rows <= 768 else {("down", down)} if rows <= 1088 else set()
        seqs = random_sequences(512, (rows - rows // 3, rows // 3), seed=rows)
        out = []
        for how in (counted, lambda *args: None):
            monkeypatch.setattr(prompt_steps, "run", how)
            out.append([])
            for cut in (slice(0, None), slice(0, 2)):           # the second step reads the pages that the first wrote
                entries = [StepEntry((rows, r), t[cut], range(len(t[cut]))) for r, t in seqs.items()]
                out[-1].append(runner.step(entries).clone())
            for r in seqs:
                runner.end((rows, r))
        assert all(torch.equal(a, b) for a, b in zip(*out)), f"{rows} rows"
        assert bool(torch.isfinite(out[0][0]).all()) and float(out[0][0].std()) > 0.01
    assert went == [True, False] * 10
    assert {("o", 2), ("down", 8), ("down", 4), ("down", 2)} <= slices


@pytest.mark.parametrize("lengths", [(1500, 1571), (400, 301), (200, 40)])
def test_a_native_step_of_prompts_holds_no_more_memory_than_the_parts(tmp_path, lengths, monkeypatch, gpu_device):
    """The most that is allocated during a step of two prompts, launched natively and by the parts (where the activation of
    the block before is held beside the results of the one that runs): rows where the tile products take none, some and all
    of the products. A kept intermediate of the step would be 0.5 to 6 MB; 64 KB are small tensors."""
    from pytriton_llama_amd.engine.batch import StepEntry
    from pytriton_llama_amd.models import prompt_steps
    from pytriton_llama_amd.weights import write_random_model
    cfg = dict(tiny("B")[0], hidden_size=512, num_attention_heads=16, num_key_value_heads=4, head_dim=64,
               intermediate_size=1024, vocab_size=512)
    write_random_model(cfg, str(tmp_path), seed=4, dtype=torch.bfloat16)
    seqs = random_sequences(512, lengths, seed=2)
    native, went, peak, logits = prompt_steps.run, [], [], []

    def counted(*args):
        done = native(*args)
        went.append(done is not None)
        return done
    for how in (counted, lambda *args: None):
        monkeypatch.setattr(prompt_steps, "run", how)
        runner = load_runner(str(tmp_path), torch.bfloat16, 16, 512)
        for turn in range(2):                   # the first step brings what stays: plans, libraries
            torch.cuda.synchronize()
            torch.cuda.reset_peak_memory_stats()
            held = torch.cuda.memory_allocated()
            got = runner.step([StepEntry((turn, r), t, [len(t) - 1]) for r, t in seqs.items()])
            torch.cuda.synchronize()
            most = torch.cuda.max_memory_allocated() - held
        peak.append(most)
        logits.append(got.clone())
        del runner
    assert went == [True, True] and torch.equal(*logits)
    assert peak[0] <= peak[1] + 65536, f"{peak[0]} bytes natively, {peak[1]} by the parts"


@pytest.mark.parametrize("dtype", DTYPES, ids=["fp32", "bf16"])
def test_first_tokens_of_a_sequence(cases, dtype):
    """Positions 0, 1, 2: one token whole, then one by one from an empty cache."""
    folder, page, seqs, want = cases["B"]
    toks = seqs["r0"][:3]
    runner = load_runner(folder, dtype, page, 4)
    from pytriton_llama_amd.engine.batch import StepEntry
    got = []
    for i, t in enumerate(toks):
        got.append(runner.step([StepEntry("x", [t], [0])]).float().cpu()[0])
    runner.end("x")
    ref = want[dtype]["r0"][:3]
    scale = float(ref.abs().max())
    err = (torch.stack(got) - ref).abs().max() / scale
    assert err < TOL[dtype], err
    # the very first token attends only itself
    one = runner.step([StepEntry("y", toks[:1], [0])]).float().cpu()[0]
    assert (one - ref[0]).abs().max() / scale < TOL[dtype]


@pytest.mark.parametrize("dtype", DTYPES, ids=["fp32", "bf16"])
def test_long_decoding(cases, dtype):
    """A short prompt and then 300 tokens one by one across many pages."""
    folder, page, _, _ = cases["A"]
    cfg = tiny("A")[0]
    seqs = random_sequences(cfg["vocab_size"], [308], seed=9)
    want = plain_logits(folder, seqs, dtype)
    steps = cuttings.tail_decode(seqs, tail=300)
    runner = load_runner(folder, dtype, page, -(-320 // page))
    got = replay(runner, steps, seqs)
    bad = first_mismatch(got, want, TOL[dtype])
    assert bad is None, bad


def _drawn_configuration(rng):
    """A Llama configuration with every size drawn: head sizes in steps of 16 up to 256, any
    number of kv heads and of query heads a kv head, widths, feed-forward sizes and
    vocabularies that are no power of two (some no multiple of 8, which the bfloat16 matrix
    kernels refuse and the general ones take), both spellings of the scaling's type key."""
    kv_heads = rng.choice([1, 2, 3, 5])
    scaling = None
    if rng.random() < 0.6:
        scaling = {rng.choice(["rope_type", "type"]): "llama3", "factor": rng.choice([2.0, 8.0, 32.0]),
                   "low_freq_factor": 1.0, "high_freq_factor": rng.choice([2.0, 4.0]),
                   "original_max_position_embeddings": rng.choice([32, 64, 256])}
    return {"architectures": ["LlamaForCausalLM"], "model_type": "llama",
            "num_hidden_layers": rng.randint(1, 3),
            "hidden_size": rng.choice([8 * rng.randint(4, 40), 2 * rng.randint(17, 99)]),
            "num_attention_heads": kv_heads * rng.choice([1, 2, 3, 4, 6, 7, 8, 16]),
            "num_key_value_heads": kv_heads,
            "head_dim": rng.choice([16, 32, 48, 64, 80, 96, 112, 128, 160, 192, 256]),
            "intermediate_size": rng.choice([8 * rng.randint(5, 60), 2 * rng.randint(21, 150)]),
            "vocab_size": rng.choice([rng.randint(100, 2000), rng.randint(2000, 40000) | 1]),
            "rope_theta": rng.choice([1e3, 1e4, 5e5]), "rope_scaling": scaling,
            "rms_norm_eps": rng.choice([1e-3, 1e-5, 1e-6]), "tie_word_embeddings": rng.random() < 0.5,
            "torch_dtype": "float32", "hidden_act": "silu", "max_position_embeddings": 4096}


@pytest.mark.parametrize("seed", [1, 3, 10, 17, 33, 40, 48, 58])
def test_drawn_configurations_mixed_with_page_reuse(tmp_path, gpu_device, seed):
    """Configurations drawn at random (sizes, options, page size), five requests of 2 to 420
    tokens in a mixed batch with so few pages that they are used again, in both dtypes."""
    import random
    from pytriton_llama_amd.weights import write_random_model
    rng = random.Random(seed)
    cfg = _drawn_configuration(rng)
    page = rng.choice([4, 8, 16, 32, 64])
    lengths = [rng.randint(2, 40), rng.randint(40, 140), rng.randint(140, 420), rng.randint(3, 90),
               rng.randint(60, 300)]
    folder = str(tmp_path)
    write_random_model(cfg, folder, seed=seed, dtype=torch.float32, norm_std=0.1,
                       std=0.8 / cfg["hidden_size"] ** 0.5)
    seqs = random_sequences(cfg["vocab_size"], lengths, seed=seed)
    steps = cuttings.mixed(seqs, seed=seed, max_live=rng.choice([2, 3, 4]))
    pages = cuttings.max_live_tokens(steps, round_to=max(64, page)) // page
    for dtype in DTYPES:
        want = plain_logits(folder, seqs, dtype)
        got = replay(load_runner(folder, dtype, page, pages, max_num_seqs=4), steps, seqs)
        bad = first_mismatch(got, want, TOL[dtype])
        assert bad is None, f"{cfg}, page size {page}, {dtype}: first wrong place {bad}"
