"""Host code of the decode session without a device: libnerva_hip.so on a stand-in for the HIP runtime (tests/host/hip_double.cpp), in a process of
its own."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = os.path.join(ROOT, "tests", "host", "hip_double.cpp")

PRELUDE = """
import ctypes, sys, threading, time
double = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
double.double_launches.restype = double.double_copies.restype = ctypes.c_long
double.double_waits.restype = ctypes.c_long
double.double_hold.argtypes = [ctypes.c_long]
double.double_log.restype = ctypes.c_char_p
double.double_fail_copy.argtypes = [ctypes.c_long]
sys.path[:0] = [%r, %r]
import numpy as np
import nerva_amd as N
from test_gpu_session import BF16, F16, random_model
NARROW = (BF16, 256, 4, 2, 64, 512, 64, 4, 5)   # (dtype, hidden, heads, kv, hd, inter, vocab, layers, seed)

def model(shape=NARROW):
    return random_model(*shape)[0]

def step(session):
    assert session.start(np.arange(5, dtype=np.uint32))[0] == 0
    return session.advance(2)[1]

def log():
    return double.double_log().decode().splitlines()

# Makes the call in a thread, up to where it waits for that stream; what is returned lets it end.
def while_held(stream, call):
    double.double_hold(stream)
    thread = threading.Thread(target=call)
    thread.start()
    while not double.double_waits():
        time.sleep(0.001)
    def over():
        double.double_hold(0)
        thread.join()
    return over
""" % (ROOT, os.path.join(ROOT, "tests"))


@pytest.fixture(scope="module")
def double(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    out = str(tmp_path_factory.mktemp("double") / "libhip_double.so")
    res = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-shared", "-fPIC", "-I/opt/rocm/include", SOURCE, "-o", out], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    return out


def run(double, body):
    res = subprocess.run([sys.executable, "-c", PRELUDE + body, double], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stdout + res.stderr


def test_chains_only_where_the_device_holds_all_their_workgroups(double):
    """A chain's workgroups wait for each other: a device (or a partition of one) with places for fewer of them takes the step's launches."""
    run(double, """
for cus, each, chained in ((256, 2, True), (16, 2, True), (16, 1, False), (8, 3, False), (32, 0, False)):   # 32 workgroups at this width
    double.double_device(cus, each)
    s = N.DecodeSession.create(model(), 64)
    assert step(s).graph_nodes == (3 if chained else 3 + 5 * 4), (cus, each)
    s.destroy()
""")


def test_the_models_that_a_chain_takes(double):
    """Either side of every line: layers, width, feed-forward, key heads, weights a layer."""
    run(double, """
double.double_device(256, 2)
base = dict(dtype=BF16, hidden=256, heads=4, kv_heads=2, head_dim=64, intermediate=512, vocab=64, layers=4, rms_eps=1e-6, rope_theta=1e4)
for change, chained in (({}, True), (dict(layers=3), False), (dict(layers=254, hidden=128, intermediate=256), True), (dict(layers=255, hidden=128, intermediate=256), False),
                        (dict(hidden=128), True), (dict(hidden=120), False), (dict(hidden=1024), True), (dict(hidden=1032), False), (dict(hidden=260), False),
                        (dict(intermediate=256), True), (dict(intermediate=248), False), (dict(intermediate=4096), True), (dict(intermediate=4104), False), (dict(intermediate=516), False),
                        (dict(heads=32, kv_heads=32), True), (dict(heads=33, kv_heads=33), False), (dict(heads=64, kv_heads=8), True), (dict(heads=65, kv_heads=13), False),
                        (dict(heads=9, kv_heads=1), False), (dict(heads=32, kv_heads=16, head_dim=128), True), (dict(heads=17, kv_heads=17, head_dim=128), True),
                        (dict(heads=22, kv_heads=22, head_dim=128), False), (dict(head_dim=96), False),
                        (dict(hidden=1024, heads=1, kv_heads=1, intermediate=1536), True), (dict(hidden=1024, heads=1, kv_heads=1, intermediate=1544), False)):
    s = N.DecodeSession.create_synthetic(dict(base, **change), 64)
    nodes = step(s).graph_nodes
    assert (nodes == 3) == chained, (change, nodes)
    s.destroy()
""")


def test_the_contexts_that_a_chain_takes(double):
    """A step at the last position of a chain's and at the first behind it: blocks a wave by the splits there are, the length of its walks, the heads."""
    run(double, """
double.double_device(256, 2)
base = dict(dtype=BF16, vocab=64, layers=4, rms_eps=1e-6, rope_theta=1e4)
for hidden, heads, kv, hd, ff, context in ((512, 8, 4, 64, 1376, 4096), (512, 16, 2, 128, 1280, 2048), (1024, 8, 2, 128, 768, 2048), (624, 3, 1, 128, 1808, 2048),
                                           (176, 8, 1, 128, 864, 2048), (128, 64, 8, 64, 1024, 4096), (768, 16, 16, 64, 768, 2048), (512, 32, 32, 64, 512, 1024),
                                           (312, 5, 5, 128, 504, 3072), (264, 20, 20, 64, 4096, 1536)):
    s = N.DecodeSession.create_synthetic(dict(base, hidden=hidden, heads=heads, kv_heads=kv, head_dim=hd, intermediate=ff), 4200)
    for tokens, nodes in ((context - 1, 3), (context, 3 + 5 * 4)):
        assert s.start(np.zeros(tokens, np.uint32))[0] == 0
        assert s.advance(2)[1].graph_nodes == nodes, (hidden, heads, kv, hd, ff, tokens)
    s.destroy()
""")


def test_the_models_that_a_launch_of_the_whole_device_takes(double):
    """Either side of every line of the wider models: layers, weights a layer, widths, heads, what fits the LDS; a device that does not hold 256 workgroups; contexts."""
    run(double, """
double.double_device(256, 1)
base = dict(dtype=BF16, hidden=1024, heads=8, kv_heads=2, head_dim=128, intermediate=4096, vocab=64, layers=4, rms_eps=1e-6, rope_theta=1e4)
for change, wide in (({}, True), (dict(layers=3), False), (dict(layers=254, intermediate=2048), True), (dict(layers=255, intermediate=2048), False),
                     (dict(intermediate=1096), False), (dict(intermediate=1104), True), (dict(intermediate=4100), False), (dict(hidden=1036), False), (dict(hidden=1032), True),
                     (dict(hidden=256, intermediate=16384), True), (dict(hidden=248, intermediate=16384), False), (dict(hidden=8192, intermediate=512), True),
                     (dict(hidden=8200, intermediate=512), False), (dict(hidden=8192, intermediate=504), False), (dict(hidden=512, intermediate=30720), True),
                     (dict(heads=9, kv_heads=1), False), (dict(heads=32, kv_heads=32), True), (dict(heads=33, kv_heads=33), False),
                     (dict(heads=64, kv_heads=8, head_dim=64), True), (dict(head_dim=96), False),
                     (dict(layers=3, hidden=2048, intermediate=4352), False), (dict(layers=3, hidden=2048, intermediate=4360), True),    # (32 M weights)
                     (dict(layers=2, hidden=2048, intermediate=4360), True), (dict(layers=1, hidden=2048, intermediate=4360), False),
                     (dict(layers=1, hidden=4096, intermediate=9560), False), (dict(layers=1, hidden=4096, intermediate=9568), True)):   # (128 M)
    s = N.DecodeSession.create_synthetic(dict(base, **change), 64)
    nodes = step(s).graph_nodes
    assert (nodes == 3) == wide, (change, nodes)
    s.destroy()
for cus, each, wide in ((256, 1, True), (255, 1, False), (128, 2, True), (304, 0, False)):
    double.double_device(cus, each)
    s = N.DecodeSession.create_synthetic(base, 64)
    assert step(s).graph_nodes == (3 if wide else 3 + 5 * 4), (cus, each)
    s.destroy()
double.double_device(256, 1)
for kv, context in ((2, 8192), (8, 32768)):
    s = N.DecodeSession.create_synthetic(dict(base, kv_heads=kv), context + 8)
    for tokens, nodes in ((context - 1, 3), (context, 3 + 5 * 4)):
        assert s.start(np.zeros(tokens, np.uint32))[0] == 0
        assert s.advance(2)[1].graph_nodes == nodes, (kv, tokens)
    s.destroy()
""")


def test_steps_come_behind_those_that_they_must_not_meet(double):
    """A launch that needs the whole device comes behind those of other sessions that are under way, and they behind it: an event of that stream, waited for ahead of the launch. Narrow models' steps
    meet each other, sessions that have nothing under way nobody; and captured steps are the same whoever else is there."""
    run(double, """
double.double_device(256, 2)
wide = dict(dtype=BF16, hidden=1024, heads=8, kv_heads=2, head_dim=128, intermediate=4096, vocab=64, layers=4, rms_eps=1e-6, rope_theta=1e4)
a = N.DecodeSession.create(model(), 64)
b = a.fork_shared_weights()
c = N.DecodeSession.create_synthetic(wide, 64)
d = c.fork_shared_weights()
sessions = (a, b, c, d)
stream = {}
for s in sessions:
    assert s.start(np.arange(5, dtype=np.uint32))[0] == 0
    double.double_clear_log()
    assert s.advance(2)[1].graph_nodes == 3
    assert not any(line.startswith("wait") for line in log()), log()
    stream[s], = (int(line.split()[1]) for line in log() if line.startswith("graph"))
for held, meets in ((a, (b,)), (c, ())):
    for other in sessions:
        if other is held:
            continue
        assert held.start(np.arange(5, dtype=np.uint32))[0] == other.start(np.arange(5, dtype=np.uint32))[0] == 0
        under_way = while_held(stream[held], lambda: held.advance(2))
        double.double_clear_log()
        assert other.advance(2)[1].graph_nodes == 3
        lines = log()
        launch = lines.index("graph %d 3" % stream[other])
        waits = [line.split()[2] for line in lines[:launch] if line.startswith("wait %d " % stream[other])]
        records = [line.split()[2] for line in lines[:launch] if line.startswith("record %d " % stream[held])]
        assert waits == records and len(waits) == (0 if other in meets else 1), (lines, stream)
        under_way()
        other.start(np.arange(5, dtype=np.uint32))
        double.double_clear_log()
        other.advance(2)
        assert not any(line.startswith("wait") for line in log())
for s in (b, a, d, c):
    s.destroy()
""")


def test_whatever_follows_a_start_comes_behind_the_steps_of_its_prompt(double):
    """A start returns while its prompt is under way: one that is walked, or whose last token takes a step, has attention launches there that must not meet a step of any other session. Every call
    that brings one comes behind it - walked and lone tokens of starts and extensions, advance and run in launches and in one, a batch, a profile -; prompts in blocks neither wait nor are waited for."""
    run(double, """
double.double_device(256, 2)
tokens = np.arange(9, dtype=np.uint32)
few = dict(dtype=BF16, hidden=512, heads=8, kv_heads=2, head_dim=64, intermediate=1024, vocab=64, layers=2, rms_eps=1e-6, rope_theta=1e4)
wide = dict(dtype=BF16, hidden=1024, heads=8, kv_heads=2, head_dim=128, intermediate=4096, vocab=64, layers=4, rms_eps=1e-6, rope_theta=1e4)
narrow = dict(few, layers=4, hidden=256, intermediate=512)
N.Device.set_tuning("prefill_walk", 1)
walked = [N.DecodeSession.create_synthetic(cfg, 64, weight_hash=7) for cfg in (few, wide, narrow)]
N.Device.reset_tuning()
blocks = [N.DecodeSession.create_synthetic(cfg, 64, weight_hash=7) for cfg in (few, wide, narrow)]
stream = {}
for s in walked + blocks:
    double.double_clear_log()
    step(s)
    stream[s], = {int(line.split()[1]) for line in log() if line.startswith("graph")}
    s.profile_step(1)                                      # (every graph is there)

def waits_behind(first, start, other, call):
    assert other.start(tokens)[0] == 0 and first.start(tokens)[0] == 0
    other.release_sequence(), first.release_sequence()
    if call not in (extended, extended_one, ran, started, started_one):
        assert other.start(tokens)[0] == 0
    double.double_clear_log()
    assert first.start(start)[0] == 0
    begun = len(log())
    call(other)
    lines = log()
    steps = [i for i, line in enumerate(lines) if line.split()[:2] in (["graph", "%d" % stream[other]], ["kernel", "%d" % stream[other]]) and "sequence_kernel" not in line and i >= begun]
    events = [line.split()[2] for line in lines[begun:] if line.startswith("record %d " % stream[first])]
    assert steps, (call, lines)
    for i, line in enumerate(lines[begun:steps[-1]]):
        if line.split()[0] == "wait" and line.split()[1] == "%d" % stream[other] and line.split()[2] in events:
            return begun + i < steps[0]
    return False

def started(s): s.start(tokens)
def started_one(s): s.start(tokens[:1])
def extended(s): s.extend(tokens)
def extended_one(s): s.extend(tokens[:1])
def advanced(s): s.advance(3)
def ran(s): s.run(tokens, 2)
def profiled(s): s.profile_step(1)
def batched(s): N.DecodeSession.batch_advance_one([s], 1, 1)
for first in walked + blocks:
    for other in walked + blocks:
        if other is first:
            continue
        for start in (tokens, tokens[:1]):
            steps = first in walked or len(start) == 1
            for call in (advanced, ran, extended_one, started_one, profiled):
                assert waits_behind(first, start, other, call) == steps, (first in walked, other in walked, len(start), call, log())
            for call in (started, extended):
                assert waits_behind(first, start, other, call) == (steps and other in walked), (first in walked, other in walked, len(start), call, log())
for s in walked + blocks:
    s.destroy()
""")


@pytest.mark.parametrize("stack", [False, True])
def test_starts_that_follow_each_other_wait_on_the_device(double, stack):
    """No more than four prompts of a set of weights are under way: the fifth's stream comes behind the first's event, ahead of everything but what brings its tokens. The host waits for the
    session's own stream and for nothing else."""
    run(double, """
if %r:
    from nerva_amd import stackbench
    stackbench.VOCAB = 64
    first = N.DecodeSession.create_stack_synthetic(stackbench.expert_stack_config(1024, 8, 4, 2, 256, 256, 256, 128, 1, 64), 64)
else:
    first = N.DecodeSession.create(model(), 64)
sessions = [first] + [first.fork_shared_weights() for _ in range(6)]
streams, events = [], []
for i, s in enumerate(sessions + sessions[:2]):
    double.double_clear_log()
    assert s.start(np.arange(20, dtype=np.uint32))[0] == 0
    lines = log()
    assert [line.split()[0] for line in lines[:2]] == ["sync", "kernel"] and "sequence_kernel" in lines[1], lines
    streams.append(lines[0].split()[1])
    waits = [line.split() for line in lines if line.startswith("wait")]
    assert len(waits) == 1 and lines[2] == " ".join(waits[0]) and waits[0][1] == streams[-1], lines
    assert sum(line.startswith("sync") for line in lines) == 1
    assert lines[-1].startswith("record %%s " %% streams[-1])
    events.append(lines[-1].split()[2])
    assert i < 4 or waits[0][2] == events[i - 4]
assert len(set(events)) == 4
for s in sessions[::-1]:
    s.destroy()
""" % stack)


def test_long_calls_beside_other_sessions_do_not_run_far_ahead(double):
    """Steps that nobody looks at: some 4 ms of them are under way at the most where a device has other sessions, so that these come in between, and fewer than give up in a row before the
    device ends a sequence where it has not; of steps in launches any number."""
    run(double, """
def looks(s):
    assert s.start(np.arange(5, dtype=np.uint32))[0] == 0
    double.double_clear_log()
    assert s.advance(301)[0] == -1                          # (the stand-in publishes no tokens)
    sent = done = most = 0
    at = {}
    for words in (line.split() for line in log()):
        if words[0] == "graph":
            sent += int(words[2]) // 3
            most = max(most, sent - done)
        elif words[0] == "record":
            at[words[2]] = sent
        elif words[:2] == ["sync", "event"]:
            done = at[words[2]]
    return most, sum(line.startswith("sync event") for line in log())
def lone(s):
    most, times = looks(s)
    return times >= 1 and 150 <= most < 256
s = N.DecodeSession.create(model(), 400)
assert lone(s)
other = s.fork_shared_weights()
most, times = looks(s)
assert times >= 2 and 50 <= most <= 2 * 56, (most, times)
other.destroy()
assert lone(s)
s.destroy()
N.Device.set_tuning("step_chain", 2)
s = N.DecodeSession.create(model(), 400)
assert looks(s)[1] == 0
s.destroy()
N.Device.reset_tuning()
large = dict(dtype=BF16, hidden=4096, heads=32, kv_heads=8, head_dim=128, intermediate=12288, vocab=64, layers=8, rms_eps=1e-6, rope_theta=1e4)   # (steps of .6 ms)
s = N.DecodeSession.create_synthetic(large, 400)
other = s.fork_shared_weights()
double.double_clear_log()
step(other)
stream, = {line.split()[1] for line in log() if line.startswith("graph")}
for held in (False, True, False):
    assert other.start(np.arange(5, dtype=np.uint32))[0] == 0
    looks(s)                                                # (the graph of six is there)
    over = while_held(int(stream), lambda: other.advance(2)) if held else lambda: None
    most, _ = looks(s)
    assert most <= (6 if held else 18) and {line.split()[2] for line in log() if line.startswith("graph")} == {"3" if held else "18"}, (held, most)
    over()
other.destroy()
s.destroy()
""")


def test_the_feed_forwards_that_ride_with_the_attention(double):
    """Up to 80 MiB of a token's experts and shared expert: on either side of the line, by the middle launch's two forms."""
    run(double, """
from nerva_amd import stackbench, stacks
stackbench.VOCAB = 64
for hidden, experts, top, ff, shared, rides in ((2048, 8, 6, 768, 1536, True), (4096, 4, 4, 512, 512, True), (4096, 8, 6, 768, 1536, False), (3584, 8, 6, 768, 1536, False),
                                                (2048, 2, 2, 2048, 2728, True), (2048, 2, 2, 2048, 2736, False), (1024, 20, 20, 1024, 64, False)):
    s = N.DecodeSession.create_stack_synthetic(stackbench.expert_stack_config(hidden, 8, experts, top, ff, shared, 256, 128, 1, 64), 64)
    before = [double.double_launches(b"layer_middle_kernelILj1ELb%d" % i) for i in (0, 1)]
    step(s)
    after = [double.double_launches(b"layer_middle_kernelILj1ELb%d" % i) for i in (0, 1)]
    assert [b - a for a, b in zip(before, after)] == ([0, 1] if rides else [1, 0]), (hidden, top, ff, shared, before, after)
    s.destroy()
""")


@pytest.mark.parametrize("source", ["tensors", "plan", "synthetic", "fork"])
def test_a_copy_that_fails_fails_the_creation(double, source):
    """Whichever of the copies of a session's creation or of a fork fails - tables, weights, what a chain's launch reads -, the call does."""
    run(double, """
weights = model()
plan = N.WeightPlan.from_weights(weights) if %(source)r == "plan" else None
cfg = dict(dtype=BF16, hidden=256, heads=4, kv_heads=2, head_dim=64, intermediate=512, vocab=64, layers=4, rms_eps=1e-6, rope_theta=1e6)
parent = N.DecodeSession.create(weights, 64)

def make():
    if %(source)r == "fork":
        return parent.fork_shared_weights()
    if %(source)r == "synthetic":
        return N.DecodeSession.create_synthetic(cfg, 64)
    return N.DecodeSession.create(weights, 64, plan=plan, tensor_pointers=plan is None)

double.double_fail_copy(-1)
s = make()
copies = double.double_copies()
assert copies >= 3 and step(s).graph_nodes == 3
s.destroy()
for i in range(copies):
    double.double_fail_copy(i)
    try:
        make().destroy()
    except RuntimeError as e:
        assert "hip_error=999" in str(e) and ("stage=0" not in str(e)), e
    else:
        raise SystemExit("copy %%d of %%d failed and nobody said so" %% (i, copies))
double.double_fail_copy(-1)
""" % dict(source=source))


def test_steps_that_go_out_together(double):
    """Steps of few launches share graphs once a session has taken 64, in calls of six and more without a stop token and short of the context where other steps begin:
    as many replays as steps, as many launches as sixes and single ones. (The stand-in publishes no tokens, so every call starts anew.)"""
    run(double, """
def go(s, n, prompt=5, eos=None):
    assert s.start(np.zeros(prompt, np.uint32), eos=eos)[0] == 0
    res = s.advance(n + 1)[1]                             # (the first token is the prompt's)
    return res.graph_replays, res.graph_launches, res.kernel_launches, res.graph_captures

s = N.DecodeSession.create(model(), 4200)
assert go(s, 40) == (40, 40, 120, 1)
assert go(s, 23) == (23, 23, 69, 0)
assert go(s, 5) == (5, 5, 15, 0)
assert go(s, 24) == (24, 4, 72, 0)
assert go(s, 5) == (5, 5, 15, 0)
assert go(s, 23) == (23, 3 + 5, 69, 0)
assert go(s, 23, eos=63)[1:] == (23, 69, 0)
context = next(p for p in range(1024, 4200, 1024) if go(s, 1, p)[2] != 3)
assert go(s, 24, context - 15) == (24, 2 + 12, 15 * 3 + 9 * (3 + 5 * 4), 0)
wide = dict(dtype=BF16, hidden=1024, heads=8, kv_heads=2, head_dim=128, intermediate=4096, vocab=64, layers=4, rms_eps=1e-6, rope_theta=1e4)
c = N.DecodeSession.create_synthetic(wide, 64)            # (nothing of it under way)
assert go(s, 12) == (12, 2, 36, 0)
c.destroy()
assert go(s, 12) == (12, 2, 36, 0)
s.destroy()
launches = N.DecodeSession.create_synthetic(dict(wide, layers=2), 512)
assert go(launches, 100)[:2] == (100, 100)
launches.destroy()
""")
