"""Steps of few single tokens as one launch (csrc/decode_stack.hip), against the plain implementation: every form of the
kernel, one row to eight with parts of long rows, first tokens, captured steps with padding rows, tokens that the host has not
seen, blocks that arrive too late; and against the same step part by part."""
import gc
import weakref

import numpy as np
import pytest
import torch

import plain_llama
from helpers import random_requests

pytestmark = pytest.mark.gpu

LAST = 3                                    # tokens of every row that are decoded one by one


def _cfg(d, ff, H, Hkv, hd, V=512, L=2, tied=True):
    return dict(architectures=["LlamaForCausalLM"], model_type="llama", hidden_size=d, intermediate_size=ff, num_hidden_layers=L,
                num_attention_heads=H, num_key_value_heads=Hkv, head_dim=hd, vocab_size=V, max_position_embeddings=2048, rms_norm_eps=1e-5,
                rope_theta=500000.0, tie_word_embeddings=tied, hidden_act="silu", eos_token_id=V - 1)


# name -> sizes: each form of the kernel (head size; up to 4096 or 8192 wide; up to 8192 or 14336 between), at the least
# sizes and at ones that leave the waves remainders
CONFIGS = {
    "64": _cfg(512, 512, 8, 2, 64, L=3), "64 uneven": _cfg(2560, 4608, 40, 8, 64, tied=False), "64 wide": _cfg(512, 1024, 72, 9, 64),
    "64 one head": _cfg(512, 1536, 8, 1, 64, V=528), "128": _cfg(1024, 1536, 16, 4, 128, tied=False), "128 long": _cfg(512, 8704, 8, 2, 128),
    "128 wide": _cfg(1024, 1024, 36, 9, 128), "128 longest": _cfg(512, 14336, 8, 2, 128),
    "128 three": _cfg(512, 1024, 24, 8, 128),
}
PAGES = {"128 three": 704}
LONG = [5 + LAST, 40, 100, 513, LAST, 32, 1200, 64]
CASES = [("64", [5 + LAST], "eager", 0), ("64", LONG, "eager", 0), ("64", LONG[4:7], "graph", 0), ("64", LONG, "graph", 0),
         ("64 uneven", LONG[2:7], "graph", 0), ("64 uneven", LONG[:6], "eager", 8), ("64 wide", LONG[3:6], "eager", 0),
         ("64 one head", [1700, 3, 640], "graph", 0), ("128", LONG[1:5], "graph", 0), ("128", [900], "eager", 64),
         ("128 long", [33, 600], "eager", 0), ("128 wide", LONG[:7], "eager", 0),
         ("128 longest", LONG, "graph", 0), ("128 three", [LAST, 40, 1999, 513, 9, 700, 64, 100], "graph", 0),
         ("128 three", [9, 1030, 30, 1999], "eager", 64)]


@pytest.fixture(scope="module")
def engines(tmp_path_factory):
    made = {}

    def get(name):
        if name not in made:
            from rustinfer_amd.config import LlamaConfig
            from rustinfer_amd.engine import build_engine
            from rustinfer_amd.weights import write_random_model
            d = str(tmp_path_factory.mktemp("stack"))
            write_random_model(LlamaConfig.from_dict(CONFIGS[name]), 7 + len(made), d)
            eng = build_engine(d, dtype="bfloat16", page_size=16, num_pages=PAGES.get(name, 256), max_requests=8, max_model_len=2048,
                               max_batch_tokens=2048)
            made[name] = (eng, plain_llama.read_model(d))
        return made[name]
    return get


def _decode(eng, reqs, mode):
    """The rows' last tokens one by one, after the rest: logits [LAST, rows, V].  The rows are released."""
    from rustinfer_amd.engine import StepEntry
    eng.enable_graphs(mode == "graph", capture_sizes=(1, 2, 4, 8))
    for r, t in reqs.items():
        if len(t) > LAST:
            eng.step([StepEntry(r, t[:-LAST], [])])
    out = []
    for s in range(LAST):
        entries = []
        for i, (r, t) in enumerate(reqs.items()):
            token = t[len(t) - LAST + s]
            if s == 1:                      # one that only the device has
                eng.device_tokens[i] = token
                token = -(i + 1)
            entries.append(StepEntry(r, [token], [0]))
        out.append(eng.step(entries).double().cpu().numpy())
    for r in reqs:
        eng.release(r)
    eng.cache.check()
    return np.stack(out)


@pytest.mark.parametrize("name,lengths,mode,grid", CASES, ids=[f"{c[0]}-{len(c[1])}-{c[2]}-{c[3]}" for c in CASES])
def test_steps_in_one_launch(engines, monkeypatch, name, lengths, mode, grid):
    from rustinfer_amd.kernels import ops
    eng, (cfg, w) = engines(name)
    stack = eng.model.stack
    assert stack is not None
    launches = []
    real = ops.decode_stack
    monkeypatch.setattr(ops, "decode_stack", lambda *a, **k: (launches.append(1), real(*a, **k))[1])
    monkeypatch.setattr(ops, "DECODE_STACK_GRID", grid)     # fewer than are waited for: the step goes on without the rest
    reqs = random_requests(cfg["vocab_size"], lengths, seed=3)
    got = _decode(eng, reqs, mode)
    assert len(launches) == (LAST if mode == "eager" else 2)             # (a graph: the pass before its capture, and the capture)
    try:
        eng.model.stack = None
        parts = _decode(eng, reqs, mode)
        assert len(launches) == (LAST if mode == "eager" else 2)
    finally:
        eng.model.stack = stack
        eng.enable_graphs(False)
    want = np.stack([plain_llama.forward(cfg, w, t)[-LAST:] for t in reqs.values()], 1)
    # rounding noise, the same for all rows and the same as part by part: the root of the mean square of a row's error is at most
    # 2 % of the logits' deviation (a wrong key, page or weight tile gives 10 % and more), and in the mean that of the parts' rows but for a tenth
    s = want.std()
    rms, rms_parts = (np.sqrt(np.mean((v - want) ** 2, axis=2)) for v in (got, parts))
    print(f"{name} {mode} {lengths}: {rms.max() / s:.2%}, part by part {rms_parts.max() / s:.2%}")
    assert np.isfinite(got).all() and rms.max() <= 0.02 * s, rms / s
    assert rms.mean() <= 1.1 * rms_parts.mean() + 1e-4 * s, (rms.mean() / s, rms_parts.mean() / s)


DIVIDED = [1203, 611, 1999, 640, 1024, 870, 1611, 770]


@pytest.fixture(scope="module")
def divided(engines):
    _, (cfg, w) = engines("128 three")
    reqs = random_requests(cfg["vocab_size"], DIVIDED, seed=11)
    return reqs, np.stack([plain_llama.forward(cfg, w, t)[-LAST:] for t in reqs.values()], 1)


@pytest.mark.parametrize("rows", range(3, 9))
def test_divided_rows_are_the_same_every_time(engines, divided, monkeypatch, rows):
    """Three query heads a key/value head, keys divided between blocks: what a merge reads is this step's, whatever the scratch held before it (other
    rows' parts, of another number of rows), so a step gives the same bits again; and the error is that of undivided rows."""
    from rustinfer_amd.kernels import ops
    eng, (cfg, _) = engines("128 three")
    reqs, want = dict(list(divided[0].items())[:rows]), divided[1][:, :rows]
    first = _decode(eng, reqs, "eager")
    for other in (rows - 1, rows):
        _decode(eng, random_requests(cfg["vocab_size"], [1300 - 37 * i for i in range(other)], seed=20 + other), "eager")
        assert np.array_equal(_decode(eng, reqs, "eager"), first)
    monkeypatch.setattr(ops, "DECODE_STACK_GRID", 32)       # fewer than two blocks a pair: no row is divided
    whole = _decode(eng, reqs, "eager")
    s = want.std()
    rms, rms_whole = (np.sqrt(np.mean((v - want) ** 2, axis=2)) for v in (first, whole))
    print(f"{rows} divided rows: {rms.max() / s:.2%}, undivided {rms_whole.max() / s:.2%}")
    assert np.isfinite(first).all() and rms.max() <= 0.02 * s, rms / s
    assert rms.mean() <= 1.1 * rms_whole.mean() + 1e-4 * s, (rms.mean() / s, rms_whole.mean() / s)


@pytest.mark.parametrize("mode", ["eager", "graph"])
@pytest.mark.parametrize("times", [dict(LIMIT_US=0.0), dict(GRID=8, CLOSE_US=1e9, JOIN_US=2e3)], ids=["phase", "start"])
def test_a_step_that_gives_up_is_an_error(engines, monkeypatch, mode, times):
    """Blocks that wait too long, for each other's results or for a second block, end the step: NaN, and whatever comes next says so, once; the requests
    have to be released.  The control words are zero again: the same steps then give the same bits as before."""
    from rustinfer_amd.engine import StepEntry, StepLost
    from rustinfer_amd.kernels import ops
    eng, (cfg, _) = engines("64")
    reqs = random_requests(cfg["vocab_size"], [40, 9, 600], seed=8)
    before = _decode(eng, reqs, mode)
    eng.enable_graphs(False)                                   # (drops the graphs)
    eng.enable_graphs(mode == "graph", capture_sizes=(1, 2, 4, 8))
    for r, t in reqs.items():
        eng.step([StepEntry(r, t, [])])
    with monkeypatch.context() as m:
        for name, value in times.items():
            m.setattr(ops, "DECODE_STACK_" + name, value)
        if mode == "graph":                                    # (the pass before the capture gives up too)
            with pytest.raises(StepLost, match="did not run to its end"):
                eng.capture_graphs([3], 700)
                eng.synchronize()
            for r, t in reqs.items():
                with pytest.raises(StepLost, match="released and run again"):
                    eng.step([StepEntry(r, t[:1], [])])
                eng.release(r)
                eng.step([StepEntry(r, t, [])])
        lost = eng.step([StepEntry(r, [5], [0]) for r in reqs])
    with pytest.raises(StepLost, match="did not run to its end"):
        eng.synchronize()
    assert lost.shape == (3, cfg["vocab_size"]) and bool(torch.isnan(lost).all())
    eng.synchronize()                                          # (said once)
    for r in reqs:
        with pytest.raises(StepLost, match="released and run again"):
            eng.step([StepEntry(r, [5], [0])])
        eng.release(r)
    eng.enable_graphs(False)
    eng.cache.check()
    assert np.array_equal(_decode(eng, reqs, mode), before)
    eng.enable_graphs(False)


def test_generate_ends_with_an_error_where_a_step_gives_up(tmp_path, monkeypatch):
    """No token is taken from logits that are none; requests that had started end as errors, and the next ones run."""
    from rustinfer_amd import LLM, SamplingParams
    from rustinfer_amd.config import LlamaConfig
    from rustinfer_amd.engine import StepLost
    from rustinfer_amd.kernels import ops
    from rustinfer_amd.weights import write_random_model
    monkeypatch.setenv("RUSTINFER_DISABLE_GRAPH", "1")
    write_random_model(LlamaConfig.from_dict(CONFIGS["64"]), 5, str(tmp_path))
    llm = LLM(model=str(tmp_path), dtype="bfloat16", paged_block_size=16, num_blocks=64, max_batch_seqs=8, max_model_len=512, max_batch_tokens=512)
    prompts = [[3, 4, 5, 6], [7, 8, 9, 10, 11, 12]]
    params = [SamplingParams(temperature=0.0, max_tokens=n, ignore_eos=True) for n in (2, 6)]      # (the first has ended when the step is missed)
    good = [r.token_ids for r in llm.generate(prompts, params)]
    with monkeypatch.context() as m:
        m.setattr(ops, "DECODE_STACK_LIMIT_US", 0.0)
        with pytest.raises(StepLost):
            llm.generate(prompts, params)
    bad = llm.scheduler.finished[-2:]
    assert {r.finish_reason for r in bad} == {"error"} and all(0 <= t < 512 for r in bad for t in r.output)
    assert not llm.scheduler.has_work() and not llm.engine.cache.live_requests()
    assert [r.token_ids for r in llm.generate(prompts, params)] == good


def test_steps_of_many_keys_go_part_by_part(engines, monkeypatch):
    """The rule goes by the longest row and the number of rows, of a captured step by what its key says of them."""
    from rustinfer_amd.engine import StepEntry
    from rustinfer_amd.kernels import ops
    eng, (cfg, _) = engines("128")
    launches = []
    real = ops.decode_stack
    monkeypatch.setattr(ops, "decode_stack", lambda *a, **k: (launches.append(1), real(*a, **k))[1])
    monkeypatch.setattr(ops, "DECODE_STACK_MOST_KEYS", 4 * 100)
    for r in range(4):
        eng.step([StepEntry(r, [5] * (99 - r), [])])
    eng.step([StepEntry(r, [5], [0]) for r in range(4)])              # 4 x 100
    assert len(launches) == 1
    eng.step([StepEntry(r, [5], [0]) for r in range(4)])              # 4 x 101
    assert len(launches) == 1
    eng.step([StepEntry(r, [5], [0]) for r in range(2)])
    assert len(launches) == 2
    eng.enable_graphs(True, capture_sizes=(1, 2, 4, 8))
    eng.step([StepEntry(r, [5], [0]) for r in range(4)])              # 4 x 1024
    assert len(launches) == 2
    eng.enable_graphs(False)
    for r in range(4):
        eng.release(r)


def test_an_engine_without_a_control_block_steps_part_by_part(engines, monkeypatch):
    """None left for this engine's workspace: the same steps, no launch of the whole stack, the parts' own results."""
    from rustinfer_amd.kernels import ops
    eng, (cfg, _) = engines("64")
    assert eng.workspace._stack_control is not None                  # (taken when the engine was built)
    reqs = random_requests(cfg["vocab_size"], [40, 9, 600], seed=8)
    stack = eng.model.stack
    try:
        eng.model.stack = None
        parts = _decode(eng, reqs, "eager")
    finally:
        eng.model.stack = stack
    monkeypatch.setattr(ops, "decode_stack_control", lambda workspace: None)
    monkeypatch.setattr(ops, "decode_stack", None)
    assert np.array_equal(_decode(eng, reqs, "eager"), parts)


@pytest.mark.parametrize("mode", ["eager", "graph"])
def test_two_engines_step_on_two_streams(engines, mode):
    """Launches that overlap, each with a control block of its own: what one holds of the chip the other waits for or goes on without, and the results
    are those of steps by themselves (rows that are not divided: no bit depends on how many blocks took part)."""
    from rustinfer_amd.engine import StepEntry
    both = [(engines("64")[0], [40, 9, 300]), (engines("128")[0], [100, 480, 17, 3])]
    steps = 12
    rng = np.random.default_rng(5)
    tokens = rng.integers(0, 512, (2, 8, 512))

    def run(streams):
        out = [[], []]
        for k, (eng, lens) in enumerate(both):
            eng.enable_graphs(mode == "graph", capture_sizes=(1, 2, 4, 8))
            for r, n in enumerate(lens):
                eng.step([StepEntry(r, tokens[k, r, :n].tolist(), [])])
            if mode == "graph":
                eng.capture_graphs([len(lens)], 512)
        torch.cuda.synchronize()
        for s in range(steps):
            for k, (eng, lens) in enumerate(both):
                with torch.cuda.stream(streams[k]):
                    out[k].append(eng.step([StepEntry(r, [int(tokens[k, r, (n + s) % 512])], [0]) for r, n in enumerate(lens)]).clone())
        torch.cuda.synchronize()
        for eng, lens in both:
            eng.check_steps()
            for r in range(len(lens)):
                eng.release(r)
            eng.enable_graphs(False)
        return [torch.stack(o).cpu().numpy() for o in out]

    alone = run([torch.cuda.current_stream()] * 2)
    beside = run([torch.cuda.Stream(), torch.cuda.Stream()])
    for a, b in zip(alone, beside):
        assert np.isfinite(a).all() and np.array_equal(a, b)


def test_a_replaced_weight_is_read(tmp_path):
    """A part that takes another weight after the model was loaded: no step reads the old one, of few rows or of many; once the model is loaded again, steps
    go in one launch again."""
    from rustinfer_amd.config import LlamaConfig
    from rustinfer_amd.engine import build_engine
    from rustinfer_amd.weights import write_random_model
    write_random_model(LlamaConfig.from_dict(CONFIGS["64"]), 5, str(tmp_path))
    eng = build_engine(str(tmp_path), dtype="bfloat16", page_size=16, num_pages=64, max_requests=8, max_model_len=512, max_batch_tokens=512)
    reqs = random_requests(512, [9, 40], seed=4)
    before = _decode(eng, reqs, "eager")
    down = eng.model.layers[1].ffn.down
    down.set_weight(-down.weight, eng.rt)
    after = _decode(eng, reqs, "eager")
    eng.model.stack = None
    assert np.array_equal(_decode(eng, reqs, "eager"), after) and np.abs(after - before).max() > 0.1 * before.std()
    from rustinfer_amd.models.stack import decode_stack
    eng.model.stack = decode_stack(eng.model, eng.rt)
    again = _decode(eng, reqs, "eager")
    assert not np.array_equal(again, after) and np.abs(again - after).max() < 0.1 * after.std()      # (the launch, with the new weight)


def test_control_blocks_are_given_back():
    """A block belongs to one workspace; one that is gone leaves its block to the next, and when all are taken there is none."""
    from rustinfer_amd.engine.context import Workspace
    from rustinfer_amd.kernels import ops
    held, blocks = [], []
    while True:
        held.append(Workspace(torch.device("cuda")))
        b = ops.decode_stack_control(held[-1])
        if b is None:
            break
        assert b not in blocks and b == ops.decode_stack_control(held[-1])
        blocks.append(b)
    assert 0 < len(blocks) <= 64
    freed = blocks[3 % len(blocks)]
    del held[3 % len(blocks)]
    gc.collect()
    assert ops.decode_stack_control(held[-1]) == freed


def test_an_engine_is_freed_with_its_last_reference(tmp_path):
    """Weights and cache go when the engine does, and not when Python next looks for cycles."""
    from rustinfer_amd.config import LlamaConfig
    from rustinfer_amd.engine import build_engine
    from rustinfer_amd.weights import write_random_model
    write_random_model(LlamaConfig.from_dict(CONFIGS["64"]), 5, str(tmp_path))
    gc.collect()
    gc.disable()
    try:
        eng = build_engine(str(tmp_path), dtype="bfloat16", page_size=16, num_pages=64, max_requests=8, max_model_len=512, max_batch_tokens=512)
        _decode(eng, random_requests(512, [9, 40], seed=4), "eager")
        assert eng.model.stack is not None
        seen = [weakref.ref(eng.model), weakref.ref(eng.model.embed.weight)]
        del eng
        assert [r() for r in seen] == [None, None]
    finally:
        gc.enable()
