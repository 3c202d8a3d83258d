"""Which kernels run a prefill batch's expert products: the short-list kernels
where experts have few rows, the 64-row tiles where tokens of one context share
them, chosen on the device from the lists.  Outputs agree with the oracle
either way, at the smallest and largest batches at which there is a choice; and
tokens of one context take no longer at a batch limit than one token above it,
where the 64-row tiles alone remain."""
import sys

import numpy as np
import pytest

import test_gpu_prefill as P
import test_gpu_sparse_groups as S
from nebula_amd import qg, synth

pytestmark = pytest.mark.gpu

# smallest batch with a choice for down and for gate/up, largest with one for gate/up and for down
LIMITS = {"1024-iq4": (65, 385, 896, 640), "1024-q4k": (65, 385, 896, 768), "2048-iq4": (65, 129, 1280, 448),
          "2048-q4k": (65, 129, 1280, 1280), "2560-iq4": (65, 129, 640, 448)}
GATE_SLOTS, DOWN_SLOTS = (4, 5), (6, 7)


@pytest.fixture(scope="module", params=sorted(LIMITS))
def case(request, qgl):
    spec = synth.LayerSpec(**S.LAYERS[request.param])
    return request.param, synth.build_layer(spec), P.host_layer(spec)


def kernel_us(L, x, slots):
    """Time of the kernels in the given event slots, the least of 9 calls."""
    lib = qg.lib()
    events = [lib.qg_event_create() for _ in range(22)]
    fw = P.forward(L, x)
    best = float("inf")
    try:
        qg.call("moe_kernel_events", (qg.C.c_void_p * 22)(*events), 22)
        for _ in range(9):
            fw.run(L, x.shape[0])
            qg.call("sync")
            us = 0.0
            for k in slots:
                ms = qg.C.c_float()
                if not lib.qg_event_elapsed(qg.C.byref(ms), events[2 * k], events[2 * k + 1]):  # recorded
                    us += ms.value * 1e3
            best = min(best, us)
    finally:
        qg.call("moe_kernel_events", None, 0)
        for e in events:
            lib.qg_event_destroy(e)
    return best


@pytest.mark.parametrize("size", [0, 1, 2, 3])
@pytest.mark.parametrize("routing", ["context", "uniform"])
def test_choice_outputs(case, routing, size):
    name, L, H = case
    nt = LIMITS[name][size]
    if routing == "context":  # about ten groups of nt rows each
        x = S.one_context(700 + nt, nt, L.spec.width)
    else:
        x = synth.inputs(700 + nt, nt, L.spec.width)
    print(f"choice {name} {routing} nt={nt}", flush=True, file=sys.stderr)
    fw = P.forward(L, x)
    P.check_routing(fw, H, x)
    P.check_outputs(fw, L, H, x, np.unique(np.r_[0, 7, 8, 63, 64, nt - 1]), f"{name} {routing} nt={nt}")


@pytest.mark.parametrize("which", ["gate", "down"])
def test_one_context_costs_no_more_below_the_limit(case, which):
    name, L, _ = case
    nt = LIMITS[name][2 if which == "gate" else 3]
    slots = GATE_SLOTS if which == "gate" else DOWN_SLOTS
    x = S.one_context(720, nt + 1, L.spec.width)
    # the short-list kernels would take 1.2 to 2.2 times as long; an idle launch is up to 4 us; three tries on a busy box
    for _ in range(3):
        below, above = kernel_us(L, x[:nt], slots), kernel_us(L, x, slots)
        print(f"limit {name} {which} nt={nt}: {below:.1f} us, one token more {above:.1f}", flush=True, file=sys.stderr)
        if below < 1.12 * above + 4:
            break
    assert below < 1.12 * above + 4


def test_choice_in_a_replayed_graph(case):
    """The choice is made at each replay: a graph captured on independent tokens and replayed on tokens of one context, and
    back, gives the eager calls' bits."""
    name, L, _ = case
    nt = LIMITS[name][3]
    xs = [synth.inputs(740, nt, L.spec.width), S.one_context(741, nt, L.spec.width)]
    want = [P.forward(L, x).out.get()[:nt] for x in xs]
    fw, graph = synth.Forward(L.spec.width, L.spec.ff, nt), qg.C.c_void_p()
    fw.x.set(xs[0])
    fw.run(L, nt)
    qg.call("graph_begin", qg.C.byref(graph))
    fw.run(L, nt)
    qg.call("graph_end", graph)
    try:
        for k in (0, 1, 1, 0):
            fw.x.set(xs[k])
            qg.call("graph_launch", graph)
            qg.call("sync")
            np.testing.assert_array_equal(fw.out.get()[:nt].view('u4'), want[k].view('u4'), err_msg=f"{name} input {k}")
    finally:
        qg.lib().qg_graph_destroy(graph)
