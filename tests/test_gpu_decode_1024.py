"""Decode batches at D = 1024 (prefill kernels in their FULL form, which keeps
the group sums in fp32): values whose 32-column sums pass fp16's range, a
resident mask (flags 1 and 2, pruning counters), each F, and the direct form's
independence of the batch a token is in.  Outputs against the oracle."""
import sys

import numpy as np
import pytest

import oracle as O
import test_gpu_prefill as P
from nebula_amd import qg, synth

pytestmark = pytest.mark.gpu

LAYERS = {
    "256-iq4": dict(seed=601, width=1024, ff=256, down_type=20, shared=True, sh_types=(12, 12, 20)),
    "256-q4k": dict(seed=602, width=1024, ff=256, down_type=12, shared=False),
    "512-q4k": dict(seed=603, width=1024, ff=512, down_type=12, shared=True, sh_types=(12, 12, 12)),
    "512-iq4": dict(seed=604, width=1024, ff=512, down_type=20, shared=False),
    "640-iq4": dict(seed=605, width=1024, ff=640, down_type=20, shared=True, sh_types=(12, 12, 20)),
}
REL = 3e-6  # fp32 sums of 22-bit activations, as the layer's timed cases


def make(name):
    spec = synth.LayerSpec(**LAYERS[name])
    return synth.build_layer(spec), P.host_layer(spec)


def rel_error(got, want):
    want = want.astype(np.float64)
    return float(np.linalg.norm(got.astype(np.float64) - want) / np.linalg.norm(want))


@pytest.mark.parametrize("nt", [1, 4, 17])
@pytest.mark.parametrize("name", ["256-iq4", "256-q4k"])
def test_input_group_sum_past_fp16(qgl, name, nt):
    """32 inputs of one sign, each within fp16's range and their sum past it."""
    L, H = make(name)
    s = L.spec
    for buf, tensor in (("gate", synth.GATE), ("up", synth.UP)):  # small weights: mid stays within fp16
        qg.call("synth_experts", L.bufs[buf].p, 12, s.seed, tensor, 512, s.ff, s.width, qg.F(0.001))
    L.desc.sh_gate = L.desc.sh_up = L.desc.sh_down = L.desc.sh_gate_inp = None
    H.shared = False
    x = synth.inputs(610 + nt, nt, s.width)
    for t in range(nt):
        g = (5 * t + 3) % 32
        x[t, 32 * g:32 * g + 32] = np.float32(2300 + 100 * t)
    print(f"group sum past fp16 {name} nt={nt}", flush=True, file=sys.stderr)
    fw = P.forward(L, x)
    want, ids, *_ = H.forward(x, fetch=P.fetcher(L))
    np.testing.assert_array_equal(fw.ids.get()[:nt], ids)
    got = fw.out.get()[:nt]
    # products and min term are each about 20 times their difference: 20 x a few 2^-24
    assert np.isfinite(got).all() and rel_error(got, want) < 1e-5


@pytest.mark.parametrize("nt", [1, 5, 17])
@pytest.mark.parametrize("name", ["256-q4k", "512-q4k"])
def test_mid_group_sum_past_fp16(qgl, name, nt):
    """Every gate and up row alike, so the mid values of a group are equal:
    3600 each, their sum 115200."""
    L, H = make(name)
    s = L.spec
    row = np.empty(qg.row_bytes(12, s.width), np.uint8)
    qg.call("read", row.ctypes.data, L.bufs["gate"].p, row.size)
    w = np.array([O.lib().nbo_weight_at(row.ctypes.data, 12, k) for k in range(s.width)], np.float64)
    tiled = np.tile(row, 512 * s.ff)
    for buf in ("gate", "up"):
        qg.call("write", L.bufs[buf].p, tiled.ctypes.data, tiled.size)
    L.desc.sh_gate = L.desc.sh_up = L.desc.sh_down = L.desc.sh_gate_inp = None
    H.shared = False
    x = (60 * w / (w @ w))[None, :] + 0.01 * np.random.default_rng(nt).standard_normal((nt, s.width))
    x = x.astype(np.float32)
    print(f"mid sum past fp16 {name} nt={nt}", flush=True, file=sys.stderr)
    fw = P.forward(L, x)
    want, ids, *_ = H.forward(x, fetch=P.fetcher(L))
    np.testing.assert_array_equal(fw.ids.get()[:nt], ids)
    got = fw.out.get()[:nt]
    # equal mid values: products and min term are each about 50 times their
    # difference (3 sigma x 256 against sigma x 16): 50 x a few 2^-24, in both
    assert np.isfinite(got).all() and rel_error(got, want) < 4e-5


@pytest.mark.parametrize("nt", [1, 3, 4, 17])
@pytest.mark.parametrize("name", sorted(LAYERS))
def test_decode_resident(qgl, name, nt):
    """With and without 60 resident experts: routing, flags and pruning
    counters as the oracle's, outputs within the layer's error."""
    L, H = make(name)
    x = synth.inputs(620 + nt, nt, 1024, correlated=True)
    fw = P.forward(L, x)
    P.check_routing(fw, H, x)
    want = H.forward(x, fetch=P.fetcher(L))[0]
    assert rel_error(fw.out.get()[:nt], want) < REL
    ids, w = O.route(H.logits(x))
    score = np.zeros(512)
    np.add.at(score, ids.ravel(), w.ravel().astype(np.float64))
    resident = np.zeros(512, np.uint8)
    resident[np.lexsort((np.arange(512), -score))[:12]] = 1
    rdev = qg.Device(resident)
    L.desc.resident, L.desc.threshold = rdev.p, 0.10
    fw = synth.Forward(1024, L.spec.ff, nt)
    fw.x.set(x)
    fw.stats.set(np.zeros(qg.C.sizeof(qg.PruneStats), np.uint8))
    print(f"decode resident {name} nt={nt}", flush=True, file=sys.stderr)
    fw.run(L, nt)
    qg.call("sync")
    P.check_routing(fw, H, x, resident)
    P.check_outputs(fw, L, H, x, np.arange(nt), f"{name} resident nt={nt}", resident=resident)
    _, _, want_stats = O.prune(ids, w, resident)
    got = qg.PruneStats.from_buffer_copy(fw.stats.get().tobytes())
    for k in ("token_layers", "missing_selections", "skipped_selections", "avoided_token_handoffs"):
        assert getattr(got, k) == getattr(want_stats, k), k
    assert got.skipped_mass == pytest.approx(want_stats.skipped_mass, rel=1e-12)  # doubles, another order of at most 17


@pytest.mark.parametrize("name", ["256-q4k", "640-iq4"])
def test_decode_batch_independent(qgl, name):
    """A token's output has the same bits alone and in every decode batch."""
    L, _ = make(name)
    x = synth.inputs(630, 17, 1024, correlated=True)
    whole = P.forward(L, x).out.get()[:17]
    for nt in (1, 2, 3, 4, 9):
        got = P.forward(L, x[:nt]).out.get()[:nt]
        np.testing.assert_array_equal(got.view('u4'), whole[:nt].view('u4'), err_msg=f"{name} nt={nt}")


@pytest.mark.parametrize("nt", [1, 2, 17])
def test_decode_phase_events(qgl, nt):
    """Every phase event is recorded, in order."""
    L, _ = make("256-q4k")
    events = [qgl.qg_event_create() for _ in range(6)]
    try:
        qg.call("moe_phase_events", (qg.C.c_void_p * 6)(*events), 6)
        P.forward(L, synth.inputs(640, nt, 1024))
        qg.call("moe_phase_events", None, 0)
        for a, b in zip(events, events[1:]):
            ms = qg.C.c_float(-1)
            qg.call("event_elapsed", qg.C.byref(ms), a, b)
            assert ms.value >= 0
    finally:
        qg.call("moe_phase_events", None, 0)
        for e in events:
            qgl.qg_event_destroy(e)


@pytest.mark.parametrize("nt", [1, 17])
def test_decode_in_a_replayed_graph(qgl, nt):
    """Direct and residual form in one graph, replayed on other inputs, against the eager calls' bits."""
    L, _ = make("512-q4k")
    fw = synth.Forward(1024, 512, nt)
    h, xn, out = (qg.Device(shape=(nt, 1024), dtype=np.float32) for _ in range(3))

    def calls():
        fw.run(L, nt)
        qg.call("moe_forward_residual", h.p, fw.ids.p, fw.w.p, fw.flags.p, None, xn.p, out.p, nt, qg.C.byref(L.desc), fw.ws.p, fw.ws_bytes)

    def results():
        qg.call("sync")
        return [d.get()[:nt].view('u4') for d in (fw.out, h, xn, out)]

    xs = [synth.inputs(650 + k, nt, 1024, correlated=k == 1) for k in range(3)]
    want = []
    for x in xs:
        fw.x.set(x)
        h.set(3 * x)
        calls()
        want.append(results())
    graph = qg.C.c_void_p()
    qg.call("graph_begin", qg.C.byref(graph))
    calls()
    qg.call("graph_end", graph)
    try:
        for k in (0, 1, 2, 0):
            fw.x.set(xs[k])
            h.set(3 * xs[k])
            qg.call("graph_launch", graph)
            for a, b in zip(results(), want[k]):
                np.testing.assert_array_equal(a, b, err_msg=f"nt={nt} input {k}")
    finally:
        qg.lib().qg_graph_destroy(graph)
