"""GPU parity at the named configurations' shapes (C1-C5), on the default decode path (the
captured graph of the bench) and the prompt/verify paths.

C1: one layer, hidden 2048, 16/4 heads of 128, MLP 8192, KV
pre-filled with 512 (then 254) rows of raw K/V ~ N(0,1) (rotations rebuilt by
the first step on both sides); then decode steps and a prompt.
C2 in full: 16 layers, vocab 100000, a 32-token prompt and 64
greedy steps; the greedy ids must match the oracle's except after a step whose
oracle top-2 logit gap is below 1e-3 (a tie, in FP32), and every
step's logits pass the reference gate.
C3 shapes with 2 of its 24 layers (one local, one global YaRN
layer): attention width 2048 under hidden 2560, the 10240-column down
projection; the engine's flow of a 12-token prefix restored from the prompt
cache, then the 116- and 443-token suffixes of the 128- and 455-token prompts,
then decode steps.
C4 shapes with 4 of its 32 layers and the full 100000-token
head: the 16K-column down projection and the fused attention at group 4.
C5 shapes with 2 of its 60 layers and the tied head: six query
heads per KV head, O and down at 6144 and 24576 columns; decode over a
455-row prefix, then verify of 1-5 candidates (the token GEMV) and 6-16
(the skinny GEMM) committed against sequential oracle forwards
(tests/metal_decode.c:309-365 at this width).
"""

import numpy as np
import pytest

import prompt_cache
from parity import compare, gate, oracle_lib, plamo_hip, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def threads():
    oracle_lib.load().oracle_set_threads(16)


def run_pair(syn, steps, prompt, fill=0, pinned=False):
    gpu, cpu = syn.instance(pinned=pinned), syn.instance()
    be = plamo_hip.Backend(syn)
    try:
        if fill:
            gpu.fill_kv(fill, 7)
            cpu.fill_kv(fill, 7)
        if prompt:
            assert be.prefill(gpu, prompt) == 1
            assert oracle_lib.prefill(cpu, prompt)
            compare(gpu, cpu)
        token = int(np.argmax(cpu.logits())) if prompt else 3
        for step in range(steps):
            say(f"step {step}")
            assert be.forward(gpu, token) == 1
            assert oracle_lib.forward(cpu, token)
            compare(gpu, cpu)
            token = int(np.argmax(cpu.logits()))
        info = be.info()
        assert info.errors == 0 and info.cpu_fallbacks == 0, info.note.decode()
    finally:
        be.close()
        gpu.close()
        cpu.close()


def test_c1_single_layer_prefilled_kv():
    cfg = plamo_hip.CONFIGS["c1"]
    syn = plamo_hip.Synthetic(**cfg, embedding_std=1.0, seed=101)
    try:
        run_pair(syn, steps=6, prompt=None, fill=512)
        # 255 -> 257 rows: four splits per KV head merged by the O projection,
        # then five merged by the last attention block.
        run_pair(syn, steps=3, prompt=None, fill=254)
        run_pair(syn, steps=3, prompt=[3, 9, 1, 15, 0, 7, 2, 11, 4, 5, 13, 6, 8], fill=0)
    finally:
        syn.close()


def test_c4_shapes_four_layers():
    # Pinned host arrays: the decode graph writes logits, state, normalized
    # state and the new K/V rows into them in place (the bench's setup). The
    # 100000-row head of the headline config, then pageable host arrays (the
    # graph stages the step's outputs in a device outbox).
    say("c4 four layers, vocab 100000")
    cfg = dict(plamo_hip.CONFIGS["c4"], layers=4)
    syn = plamo_hip.Synthetic(**cfg, pattern=4, seed=202)
    try:
        run_pair(syn, steps=4, prompt=list(range(5, 5 + 69 * 7, 7)), pinned=True)
        run_pair(syn, steps=2, prompt=list(range(3, 3 + 20 * 5, 5)))
    finally:
        syn.close()


def test_c3_prefix_restore_and_prompts():
    # runtime/engine.c:358-381: the 12-token template prefix is prefilled once
    # and captured (runtime/prompt_cache.c); each request resets the model,
    # restores the prefix rows and prefills the rest of its prompt. The oracle
    # prefills the whole prompt from a reset model.
    cfg = dict(plamo_hip.CONFIGS["c3"], layers=2, vocab=1000)
    syn = plamo_hip.Synthetic(**cfg, pattern=2, seed=606)
    gpu, cpu = syn.instance(pinned=True), syn.instance()
    be = plamo_hip.Backend(syn)
    try:
        rng = np.random.default_rng(128)
        prefix = rng.integers(0, cfg["vocab"], size=12).tolist()
        assert be.prefill(gpu, prefix) == 1
        snap = prompt_cache.capture(gpu, prefix)
        assert snap is not None
        for total in (128, 455):
            say(f"c3 prompt {total} ({total - 12} after the restored prefix)")
            ids = prefix + rng.integers(0, cfg["vocab"], size=total - 12).tolist()
            gpu.reset()
            cpu.reset()
            assert prompt_cache.restore(snap, gpu, ids) == 12
            assert be.prefill(gpu, ids[12:]) == 1
            assert oracle_lib.prefill(cpu, ids)
            compare(gpu, cpu)
            token = prompt_cache.greedy(cpu)
            for step in range(3):
                assert be.forward(gpu, token) == 1
                assert oracle_lib.forward(cpu, token)
                compare(gpu, cpu)
                token = prompt_cache.greedy(cpu)
        info = be.info()
        assert info.errors == 0 and info.cpu_fallbacks == 0, info.note.decode()
    finally:
        be.close()
        gpu.close()
        cpu.close()
        syn.close()


def test_c5_decode_and_verify_over_455_rows():
    cfg = dict(plamo_hip.CONFIGS["c5"], layers=2, vocab=500)
    syn = plamo_hip.Synthetic(**cfg, pattern=2, embedding_std=1.0, seed=707)
    gpu, cpu = syn.instance(pinned=True), syn.instance()
    be = plamo_hip.Backend(syn)
    try:
        # 455 prefix rows of raw K/V ~ N(0,1); the first step rebuilds the
        # rotations (eager), the next ones run the captured graph.
        gpu.fill_kv(455, 9)
        cpu.fill_kv(455, 9)
        token = 7
        for step in range(3):
            say(f"c5 decode step {step}")
            assert be.forward(gpu, token) == 1
            assert oracle_lib.forward(cpu, token)
            compare(gpu, cpu)
            token = prompt_cache.greedy(cpu)
        base = cpu.snapshot()
        ids = [(i * 37 + 11) % cfg["vocab"] for i in range(16)]
        for count in (1, 2, 3, 4, 5, 6, 8, 16):
            say(f"c5 verify {count} candidates over {base['layers'][0][3]} rows")
            cpu.restore(base)
            states, logits, gold = [], [], []
            for i in range(count):
                assert oracle_lib.forward(cpu, ids[i])
                states.append(cpu.state().copy())
                logits.append(cpu.logits().copy())
                gold.append(int(np.argmax(cpu.logits())))
            # The oracle's rows replace the GPU's at unchanged counters: an
            # edit the backend is told about (include/plamo_draft.h).
            gpu.restore(base)
            be.invalidate()
            r, nxt = be.verify(gpu, ids[:count])
            assert r == 1
            for i in range(count):
                top2 = np.sort(logits[i])[-2:]
                if top2[1] - top2[0] >= 1e-3:
                    assert nxt[i] == gold[i], f"candidate {i}"
                assert be.commit(gpu, i) == 1
                gate(gpu.state().copy(), states[i], f"verified state {i}")
                gate(gpu.logits().copy(), logits[i], f"verified logits {i}")
            compare(gpu, cpu)
            assert be.commit(gpu, count) == 0
            if count == 5:
                # A rejected suffix: three commits, then an ordinary step.
                cpu.restore(base)
                for i in range(3):
                    assert oracle_lib.forward(cpu, ids[i])
                assert oracle_lib.forward(cpu, 12)
                gpu.restore(base)
                be.invalidate()
                assert be.verify(gpu, ids[:count])[0] == 1
                for i in range(3):
                    assert be.commit(gpu, i) == 1
                assert be.forward(gpu, 12) == 1
                assert be.commit(gpu, 3) == 0
                compare(gpu, cpu)
        info = be.info()
        assert info.errors == 0 and info.cpu_fallbacks == 0, info.note.decode()
        assert info.verification_batches >= 9
    finally:
        be.close()
        gpu.close()
        cpu.close()
        syn.close()


def test_c2_greedy_64_steps():
    cfg = plamo_hip.CONFIGS["c2"]
    syn = plamo_hip.Synthetic(**cfg, seed=303)
    gpu, cpu = syn.instance(), syn.instance()
    be = plamo_hip.Backend(syn)
    try:
        rng = np.random.default_rng(32)
        prompt = rng.integers(0, cfg["vocab"], size=32).tolist()
        assert be.prefill(gpu, prompt) == 1
        assert oracle_lib.prefill(cpu, prompt)
        compare(gpu, cpu, kv=False)
        token = int(np.argmax(cpu.logits()))
        diverged = False
        for step in range(64):
            lg = cpu.logits().copy()
            top2 = np.sort(lg)[-2:]
            g_tok = int(np.argmax(gpu.logits()))
            if not diverged:
                if g_tok != token:
                    # Allowed only where the oracle's own top-2 gap is tiny.
                    assert top2[1] - top2[0] < 1e-3, f"step {step}: {g_tok} vs {token}"
                    diverged = True
                    break
            assert be.forward(gpu, token) == 1
            assert oracle_lib.forward(cpu, token)
            gate(gpu.logits().copy(), cpu.logits().copy(), f"step {step} logits")
            gate(gpu.state().copy(), cpu.state().copy(), f"step {step} state")
            token = int(np.argmax(cpu.logits()))
            if step % 8 == 0:
                say(f"greedy step {step}: token {token}")
        info = be.info()
        assert info.errors == 0 and info.cpu_fallbacks == 0
    finally:
        be.close()
        gpu.close()
        cpu.close()
        syn.close()


def test_long_context_split_attention():
    # Contexts past 1024 rows split a KV head over several blocks whose
    # partials are merged by the last one; 1023 -> 1025 crosses the boundary.
    syn = plamo_hip.Synthetic(512, 2, 8, 2, 128, 1024, 500, window=4096, global_capacity=8192,
                              pattern=2, embedding_std=1.0, seed=404)
    try:
        run_pair(syn, steps=3, prompt=None, fill=1023)
        run_pair(syn, steps=3, prompt=None, fill=3000)
    finally:
        syn.close()


@pytest.mark.parametrize("pinned", [False, True])
def test_short_context_graph_boundary(pinned):
    # Below 256 rows in every layer a decode step runs the short-context graph
    # (32-row attention blocks over at most 256 allocated rows); the step whose
    # count reaches 256 switches to the general graph. 250 -> 262 crosses it,
    # with the allocation grown to 512 rows first (a longer prompt earlier in
    # the request), as the bench's decode runs after its 455-token prompts.
    syn = plamo_hip.Synthetic(512, 2, 8, 2, 128, 1024, 500, window=4096, global_capacity=8192,
                              pattern=2, embedding_std=1.0, seed=405)
    try:
        run_pair(syn, steps=12, prompt=None, fill=250, pinned=pinned)
        gpu, cpu = syn.instance(pinned=pinned), syn.instance()
        be = plamo_hip.Backend(syn)
        try:
            prompt = [(j * 13 + 5) % 500 for j in range(300)]
            assert be.prefill(gpu, prompt) == 1  # allocation grows past 256 rows
            gpu.reset()
            cpu.reset()
            assert be.prefill(gpu, prompt[:200]) == 1
            assert oracle_lib.prefill(cpu, prompt[:200])
            token = int(np.argmax(cpu.logits()))
            for step in range(60):
                assert be.forward(gpu, token) == 1
                assert oracle_lib.forward(cpu, token)
                compare(gpu, cpu)
                token = int(np.argmax(cpu.logits()))
            info = be.info()
            assert info.errors == 0 and info.cpu_fallbacks == 0, info.note.decode()
        finally:
            be.close()
            gpu.close()
            cpu.close()
    finally:
        syn.close()


def test_eager_decode_matches_graph(monkeypatch):
    """PLAMO_HIP_EAGER_DECODE=1 (read when the backend opens) launches the
    decode step's kernels one by one instead of replaying the captured graph:
    the same kernels with the same arguments, so logits, states and the
    appended KV rows are bit-identical to the graph's, in the short-context
    graph's range and past it."""
    cfg = dict(plamo_hip.CONFIGS["c4"], layers=2, vocab=1000)
    syn = plamo_hip.Synthetic(**cfg, pattern=2, seed=808)
    runs = []
    try:
        for eager in ("", "1"):
            say(f"eager={eager!r}")
            monkeypatch.setenv("PLAMO_HIP_EAGER_DECODE", eager)
            gpu = syn.instance(pinned=True)
            be = plamo_hip.Backend(syn)
            monkeypatch.delenv("PLAMO_HIP_EAGER_DECODE")
            try:
                gpu.fill_kv(250, 5)
                token, out = 3, []
                for step in range(10):  # rows 251..260 cross the 256-row boundary
                    assert be.forward(gpu, token) == 1
                    out.append((gpu.logits().copy(), gpu.state().copy(), gpu.normalized().copy()))
                    token = int(np.argmax(out[-1][0]))
                kv = [gpu.kv(i, w).copy() for i in range(cfg["layers"])
                      for w in ("k", "v", "rot")]
                info = be.info()
                assert info.errors == 0 and info.cpu_fallbacks == 0, info.note.decode()
                runs.append((out, kv))
            finally:
                be.close()
                gpu.close()
    finally:
        syn.close()
    (graph_out, graph_kv), (eager_out, eager_kv) = runs
    for a, b in zip(graph_out, eager_out):
        for x, y in zip(a, b):
            assert np.array_equal(x, y)
    for x, y in zip(graph_kv, eager_kv):
        assert np.array_equal(x, y)


# The fp16-pair prompt attention without a window: groups whose (query tile,
# head) units leave waves of a block idle, prompts of one tile and a row, of
# whole tiles, a prefix of four prompts (its limit) and one past it, and grids
# of more than one block per CU (one group of waves per block instead of two).
# Few query rows (tokens x heads below 5120) take the FP32 form at the groups it
# covers: the first rows stand on its side, the others on that of the pairs.
@pytest.mark.parametrize("qh,kh,dim,prefix,tokens", [
    (6, 3, 128, 0, 33), (6, 1, 64, 0, 65), (4, 4, 64, 160, 40), (4, 4, 64, 161, 40),
    (3, 3, 64, 5, 129), (16, 1, 128, 7, 96), (32, 32, 64, 0, 1030), (16, 4, 128, 3, 2050),
    (5, 1, 64, 0, 33), (3, 1, 128, 0, 65), (128, 64, 64, 160, 40), (128, 64, 64, 161, 40),
    (102, 51, 64, 0, 51), (60, 60, 64, 5, 129), (64, 4, 128, 7, 96), (102, 17, 64, 0, 64),
])
def test_prompt_pair_attention(qh, kh, dim, prefix, tokens):
    say(f"pair attention {qh}/{kh}x{dim} prefix={prefix} tokens={tokens}")
    syn = plamo_hip.Synthetic(256, 2, qh, kh, dim, 96, 300, window=2304, global_capacity=2304,
                              pattern=2, embedding_std=1.0, seed=77)
    gpu, cpu = syn.instance(), syn.instance()
    be = plamo_hip.Backend(syn)
    try:
        ids = [(j * 13 + 5) % 300 for j in range(prefix + tokens)]
        for part in (ids[:prefix], ids[prefix:]):
            if not part:
                continue
            actual = np.zeros((len(part), 256), np.float32)
            expected = np.zeros((len(part), 256), np.float32)
            assert be.prefill(gpu, part, actual) == 1
            assert oracle_lib.prefill(cpu, part, expected)
            gate(actual, expected, "all prompt states")
            compare(gpu, cpu)
        info = be.info()
        assert info.errors == 0 and info.cpu_fallbacks == 0, info.note.decode()
    finally:
        be.close()
        gpu.close()
        cpu.close()
        syn.close()


# The copies of a prompt's ids in and of its results out, at vocabularies that
# leave the host blocks at every word alignment.
@pytest.mark.parametrize("vocab", [200, 201, 202, 203])
@pytest.mark.parametrize("pinned", [False, True])
def test_result_copies(vocab, pinned):
    say(f"result copies vocab={vocab} pinned={pinned}")
    syn = plamo_hip.Synthetic(256, 2, 4, 2, 64, 96, vocab, window=64, global_capacity=128,
                              pattern=2, embedding_std=1.0, seed=vocab)
    gpu, cpu = syn.instance(pinned=pinned), syn.instance()
    be = plamo_hip.Backend(syn)
    try:
        for tokens in (1, 2, 7, 19):
            ids = [(7 * j + 3) % vocab for j in range(tokens)]
            assert be.prefill(gpu, ids) == 1
            assert oracle_lib.prefill(cpu, ids)
            compare(gpu, cpu)
        for tokens in (1, 3, 16):
            ids = [(5 * j + 2) % vocab for j in range(tokens)]
            assert be.verify(gpu, ids)[0] == 1
            for i in range(min(tokens, 2)):
                assert oracle_lib.forward(cpu, ids[i])
                assert be.commit(gpu, i) == 1
                compare(gpu, cpu)
    finally:
        be.close()
        gpu.close()
        cpu.close()
        syn.close()


# Decode steps whose contexts take 16, 17, 32 and 33 splits, at the edges of the
# merging block's batches (16 partials, 32 maxima).
@pytest.mark.parametrize("rows", [1022, 1086, 2046, 2110])
def test_decode_split_merge(rows):
    say(f"split merge rows={rows}")
    syn = plamo_hip.Synthetic(256, 1, 16, 4, 128, 96, 300, window=2304, global_capacity=2304,
                              pattern=1, embedding_std=1.0, seed=31)
    gpu, cpu = syn.instance(), syn.instance()
    be = plamo_hip.Backend(syn)
    try:
        ids = [(j * 13 + 5) % 300 for j in range(rows)]
        states = np.zeros((rows, 256), np.float32)
        assert be.prefill(gpu, ids, states) == 1
        assert oracle_lib.prefill(cpu, ids, states)
        for token in (7, 11, 2, 290):
            assert be.forward(gpu, token) == 1
            assert oracle_lib.forward(cpu, token)
            compare(gpu, cpu)
        info = be.info()
        assert info.errors == 0 and info.cpu_fallbacks == 0, info.note.decode()
    finally:
        be.close()
        gpu.close()
        cpu.close()
        syn.close()


# Prompts, decode steps and candidates past a sliding window at the head dims
# and groups of the matrix-core prompt attention and the fused decode
# attention: windows of less and more than a key tile (32) and an attention
# block (64), prompts that start before, at and past the window's end, and a
# window of which no prompt row sees the prefix.
@pytest.mark.parametrize("qh,kh,dim,window,prefix,tokens", [
    (8, 2, 128, 40, 0, 100), (8, 2, 128, 40, 12, 45), (4, 4, 64, 17, 18, 33),
    (12, 2, 128, 32, 33, 2), (16, 1, 64, 300, 3, 700), (8, 4, 128, 64, 50, 17),
    (16, 2, 64, 5, 6, 300), (16, 2, 128, 70, 12, 75),
    # On the fp16 pairs (enough query rows).
    (64, 16, 128, 40, 0, 100), (52, 26, 64, 17, 18, 130), (36, 6, 128, 5, 6, 150),
    (64, 4, 64, 64, 50, 97),
])
@pytest.mark.parametrize("pinned", [False, True])
def test_past_the_window(qh, kh, dim, window, prefix, tokens, pinned):
    say(f"past the window {qh}/{kh}x{dim} window={window} prefix={prefix} tokens={tokens}")
    syn = plamo_hip.Synthetic(512, 2, qh, kh, dim, 768, 300, window=window, global_capacity=1200,
                              pattern=2, embedding_std=1.0, seed=909)
    gpu, cpu = syn.instance(pinned=pinned), syn.instance()
    be = plamo_hip.Backend(syn)
    try:
        ids = [(j * 13 + 5) % 300 for j in range(prefix + tokens)]
        for part in (ids[:prefix], ids[prefix:]):
            if not part:
                continue
            actual = np.zeros((len(part), 512), np.float32)
            expected = np.zeros((len(part), 512), np.float32)
            assert be.prefill(gpu, part, actual) == 1
            assert oracle_lib.prefill(cpu, part, expected)
            gate(actual, expected, "all prompt states")
            compare(gpu, cpu)
        for token in (7, 11, 2, 290):
            assert be.forward(gpu, token) == 1
            assert oracle_lib.forward(cpu, token)
            compare(gpu, cpu)
        candidates = [9, 4, 250, 31, 8, 77, 6]
        assert be.verify(gpu, candidates)[0] == 1
        for i, token in enumerate(candidates[:5]):
            assert oracle_lib.forward(cpu, token)
            assert be.commit(gpu, i) == 1
            compare(gpu, cpu)
        # Past the slack rows a full window moves through (128 steps).
        for step in range(135):
            assert be.forward(gpu, step) == 1
            assert oracle_lib.forward(cpu, step)
        compare(gpu, cpu)
        if qh * dim == 2048:
            # A step on full windows whose O blocks give up their wait: -1, and
            # the host rows as they were, so that the step can be taken again.
            before = [gpu.kv(0, which).copy() for which in ("k", "v")]
            be.debug_waits(1, 16)
            assert be.forward(gpu, 21) == -1
            be.debug_waits(0, 0)
            for which, rows in zip(("k", "v"), before):
                assert np.array_equal(gpu.kv(0, which), rows)
            assert be.info().errors == 1
            assert be.forward(gpu, 21) == 1
            assert oracle_lib.forward(cpu, 21)
            compare(gpu, cpu)
        # A new request on the moved buffers.
        gpu.reset()
        cpu.reset()
        assert be.prefill(gpu, ids[:9]) == 1
        assert oracle_lib.prefill(cpu, ids[:9])
        for token in (3, 5):
            assert be.forward(gpu, token) == 1
            assert oracle_lib.forward(cpu, token)
            compare(gpu, cpu)
        info = be.info()
        assert info.errors == (qh * dim == 2048) and info.cpu_fallbacks == 0, info.note.decode()
    finally:
        be.close()
        gpu.close()
        cpu.close()
        syn.close()


# Steps on full 2049-row windows whose rows the host has just changed (other
# rows, stale and current rotations; a CPU step; an announced edit), with every
# table and buffer grown by an earlier step: 17 MB cross the bus while the step
# moves the host's rows by one.
@pytest.mark.parametrize("pinned", [False, True])
def test_edited_full_windows(pinned):
    say(f"edited full windows pinned={pinned}")
    syn = plamo_hip.Synthetic(256, 2, 16, 8, 128, 96, 300, window=2048, global_capacity=4096,
                              pattern=0, embedding_std=1.0, seed=12)
    gpu, cpu = syn.instance(pinned=pinned), syn.instance()
    be = plamo_hip.Backend(syn)
    try:
        def step(token):
            assert be.forward(gpu, token) == 1
            assert oracle_lib.forward(cpu, token)
            compare(gpu, cpu)

        for seed in (1, 2):
            say(f"fill {seed}")
            for inst in (gpu, cpu):
                inst.fill_kv(2049, seed)
            step(7)
            step(8)
        say("CPU step")
        assert oracle_lib.forward(gpu, 9) and oracle_lib.forward(cpu, 9)
        step(10)
        say("announced edit")
        for inst in (gpu, cpu):
            inst.kv(1, "v")[5:1500] *= 0.5
            inst.kv(0, "k")[5:1500] *= 0.5
            inst.rotation(0).processed_count = 0
        be.invalidate()
        step(11)
        step(12)
        info = be.info()
        assert info.errors == 0 and info.cpu_fallbacks == 0, info.note.decode()
    finally:
        be.close()
        gpu.close()
        cpu.close()
        syn.close()


# A prompt without its states (only the last row feeds the logits) at groups
# the fp16-pair attention takes and the FP32 matrix-core form does not, and at
# groups both take.
@pytest.mark.parametrize("qh,kh,dim", [(3, 1, 128), (6, 2, 64), (5, 1, 64), (14, 2, 128),
                                       (64, 16, 128), (60, 10, 128)])
@pytest.mark.parametrize("prefix,tokens,window", [(0, 33, 2304), (9, 90, 2304), (12, 300, 2304),
                                                  (9, 90, 40)])
def test_prompt_last_row(qh, kh, dim, prefix, tokens, window):
    say(f"last row {qh}/{kh}x{dim} prefix={prefix} tokens={tokens} window={window}")
    syn = plamo_hip.Synthetic(256, 3, qh, kh, dim, 96, 300, window=window, global_capacity=2304,
                              pattern=2, embedding_std=1.0, seed=5)
    gpu, cpu = syn.instance(), syn.instance()
    be = plamo_hip.Backend(syn)
    try:
        for turn in range(2):  # the buffers then hold another prompt's rows
            gpu.reset()
            cpu.reset()
            ids = [(j * 13 + 5 * turn) % 300 for j in range(prefix + tokens)]
            for part in (ids[:prefix], ids[prefix:]):
                if part:
                    assert be.prefill(gpu, part) == 1
                    assert oracle_lib.prefill(cpu, part)
                    compare(gpu, cpu)
                    gate(gpu.normalized().copy(), cpu.normalized().copy(), "normalized")
        info = be.info()
        assert info.errors == 0 and info.cpu_fallbacks == 0, info.note.decode()
    finally:
        be.close()
        gpu.close()
        cpu.close()
        syn.close()


# A prompt in which a run of tokens has V rows some 2^24 times the others' (their
# embedding alone reaches a column of the V projection): the tokens before them,
# in their key tiles and in earlier ones, are as close to the oracle as without
# them, and those after them, which see them, agree with the oracle as well.
# Runs of one, of part of a tile, and of whole tiles.
@pytest.mark.parametrize("qh,kh,dim,prefix,tokens,at,run", [
    (52, 26, 64, 0, 100, 80, 1), (24, 6, 128, 12, 300, 290, 1), (9, 3, 64, 5, 60, 59, 1),
    (16, 16, 64, 0, 1030, 700, 1), (32, 8, 128, 12, 200, 84, 70), (42, 7, 64, 7, 130, 25, 105),
    (16, 16, 64, 5, 1030, 707, 300), (5, 1, 128, 0, 90, 40, 20),
])
def test_prompt_attention_large_value_rows(qh, kh, dim, prefix, tokens, at, run):
    say(f"large V rows {qh}/{kh}x{dim} prefix={prefix} tokens={tokens} at={at} run={run}")
    hidden, vocab, special = 256, 300, 299
    syn = plamo_hip.Synthetic(hidden, 2, qh, kh, dim, 96, vocab, window=2304, global_capacity=2304,
                              pattern=2, embedding_std=1.0, seed=qh)
    gpu, cpu = syn.instance(), syn.instance()
    emb = np.ctypeslib.as_array(gpu.model.embedding, shape=(vocab, hidden))
    emb[:, 0] = 0
    emb[special] = 0
    emb[special, 0] = 0x3f80  # 1.0
    qkv = np.ctypeslib.as_array(gpu.layer(0).mixer.contents.qkv.contents.weight,
                                shape=((qh + 2 * kh) * dim, hidden))
    v = qkv[(qh + kh) * dim:]
    v[:, 0] = np.where(v[:, 0] & 0x7fff, v[:, 0] + np.uint16(22 << 7), 0)  # 2^4 from the norm
    be = plamo_hip.Backend(syn)
    try:
        ids = [(j * 13 + 5) % 290 for j in range(prefix + tokens)]
        ids[prefix + at:prefix + at + run] = [special] * run
        for part in (ids[:prefix], ids[prefix:]):
            if not part:
                continue
            actual = np.zeros((len(part), hidden), np.float32)
            expected = np.zeros((len(part), hidden), np.float32)
            assert be.prefill(gpu, part, actual) == 1
            assert oracle_lib.prefill(cpu, part, expected)
            gate(actual, expected, "all prompt states")
        before, _ = gate(actual[:at], expected[:at], "states before the rows")
        say(f"before them {before:.3g}")
        # Without them 2e-7 to 3.5e-7 (sums of up to 1030 terms in FP32).
        assert before <= 1e-6
        compare(gpu, cpu)
    finally:
        be.close()
        gpu.close()
        cpu.close()
        syn.close()
