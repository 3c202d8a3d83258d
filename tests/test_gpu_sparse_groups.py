"""The prefill's kernels for short row lists (qg_sparse.h) where they can go
wrong: groups of 1 row, of exactly and just over one tile and one run, few long
groups among empty experts, with and without the shared expert, each width and
down format; and the batch limits, where both kernels see the same rows.
Outputs against the oracle at the layer's tolerance, routing bit for bit."""
import sys

import numpy as np
import pytest

import test_gpu_prefill as P
from nebula_amd import synth

pytestmark = pytest.mark.gpu

LAYERS = {
    "1024-iq4": dict(seed=501, width=1024, ff=256, down_type=20, shared=True, sh_types=(12, 12, 20)),
    "1024-q4k": dict(seed=502, width=1024, ff=256, down_type=12, shared=False),
    "2048-iq4": dict(seed=503, width=2048, ff=512, down_type=20, shared=True, sh_types=(12, 12, 20)),
    "2048-q4k": dict(seed=504, width=2048, ff=512, down_type=12, shared=True, sh_types=(12, 12, 12)),
    "2560-iq4": dict(seed=505, width=2560, ff=640, down_type=20, shared=True, sh_types=(12, 12, 20)),
}


@pytest.fixture(scope="module", params=sorted(LAYERS))
def layer(request, qgl):
    spec = synth.LayerSpec(**LAYERS[request.param])
    return synth.build_layer(spec), P.host_layer(spec)


def one_context(seed, nt, width):
    """Rows so alike that nearly every token selects the same experts: about
    ten groups of nt rows."""
    rng = np.random.default_rng(seed)
    return synth.rmsnorm(rng.standard_normal(width)[None, :] + 0.01 * rng.standard_normal((nt, width)))


@pytest.mark.parametrize("nt", [18, 24, 25, 33, 200])
def test_sparse_long_groups(layer, nt):
    L, H = layer
    x = one_context(510 + nt, nt, L.spec.width)
    fw = P.forward(L, x)
    P.check_routing(fw, H, x)
    P.check_outputs(fw, L, H, x, np.unique(np.r_[0, 7, 8, 15, 16, 17, nt - 1]), f"long groups D={L.spec.width} nt={nt}")


@pytest.mark.parametrize("nt", [18, 61])
def test_sparse_short_groups(layer, nt):
    L, H = layer
    x = synth.inputs(520 + nt, nt, L.spec.width)
    fw = P.forward(L, x)
    P.check_routing(fw, H, x)
    P.check_outputs(fw, L, H, x, P.sample_rows(nt, 8, nt), f"short groups D={L.spec.width} nt={nt}")


@pytest.mark.parametrize("nt", [1, 2, 4, 17])
@pytest.mark.parametrize("name", ["1024-iq4", "1024-q4k"])
def test_sparse_decode_widths(qgl, name, nt):
    """Decode batches of a width without decode kernels, direct and residual
    form: routing, outputs, and the workspace of the batch's own size."""
    from nebula_amd import qg
    spec = synth.LayerSpec(**LAYERS[name])
    L, H = synth.build_layer(spec), P.host_layer(spec)
    x = synth.inputs(550 + nt, nt, spec.width, correlated=True)
    fw = P.forward(L, x)
    P.check_routing(fw, H, x)
    P.check_outputs(fw, L, H, x, np.arange(nt), f"{name} nt={nt}")
    h = qg.Device(x)
    xn, out = qg.Device(np.zeros_like(x)), qg.Device(np.zeros_like(x))
    qg.call("moe_forward_residual", h.p, fw.ids.p, fw.w.p, fw.flags.p, None, xn.p, out.p, nt, qg.C.byref(L.desc), fw.ws.p, fw.ws_bytes)
    qg.call("sync")
    np.testing.assert_array_equal(h.get().view('u4'), (x + out.get()).view('u4'))
    P.assert_close(out.get(), H.forward(xn.get(), fetch=P.fetcher(L))[0], "residual form")


@pytest.mark.parametrize("nt", [9, 10, 14, 17])
@pytest.mark.parametrize("name", ["2048-iq4", "2048-q4k"])
def test_decode_shares_span_experts(qgl, name, nt):
    """Verify batches of independent tokens touch so many experts that a
    gate/up workgroup's share may end one and begin the next; a second call
    with one context's tokens goes back to whole workgroups per expert."""
    spec = synth.LayerSpec(**LAYERS[name])
    L, H = synth.build_layer(spec), P.host_layer(spec)
    for corr in (False, True):
        x = synth.inputs(560 + nt, nt, spec.width, correlated=corr)
        fw = P.forward(L, x)
        P.check_routing(fw, H, x)
        P.check_outputs(fw, L, H, x, np.arange(nt), f"{name} nt={nt} corr={corr}")


@pytest.mark.parametrize("limit", [256, 448, 640, 768, 896, 1280])
def test_sparse_limits_agree(layer, limit):
    """A batch at a limit and one token above it: the shared rows agree (the
    kernels differ in the order of their fp32 sums only)."""
    L, _ = layer
    x = synth.inputs(530, limit + 1, L.spec.width)
    a, b = P.forward(L, x[:limit]), P.forward(L, x)
    np.testing.assert_array_equal(a.ids.get()[:limit], b.ids.get()[:limit])
    u, v = a.out.get()[:limit].astype(np.float64), b.out.get()[:limit].astype(np.float64)
    rel = np.linalg.norm(u - v) / np.linalg.norm(v)
    print(f"limit {limit} D={L.spec.width}: rel {rel:.2e}", flush=True, file=sys.stderr)
    assert rel < 3e-6  # each within 7e-7 of the 64-bit result


def test_sparse_all_tokens_handed_off(layer):
    """No expert resident and a zero threshold: every token is flagged, so the
    routed groups are all empty and only the shared expert (or nothing) runs."""
    from nebula_amd import qg
    L, H = layer
    nt = 40
    desc = qg.MoeLayer.from_buffer_copy(L.desc)
    mask = qg.Device(np.zeros(512, np.uint8))
    desc.resident, desc.threshold = mask.p, 0.10
    saved, L.desc = L.desc, desc
    try:
        x = synth.inputs(540, nt, L.spec.width)
        fw = P.forward(L, x)
        flags = fw.flags.get()[:nt]
        assert np.all(flags == 2)
        got = fw.out.get()[:nt]
        if H.shared:
            P.assert_close(got, H.shared_part(x), "shared part alone")
        else:
            assert np.all(got == 0)
    finally:
        L.desc = saved


def test_whole_workgroups_where_they_fit(qgl):
    """9 independent tokens on 84 experts and the shared one, each a fifth of a percent short of three gate/up
    workgroups: all of them get three, and the layer takes no longer than on 83 experts (within 0.5 %; 4 % if its shares span
    two experts)."""
    from nebula_amd import qg
    spec = synth.LayerSpec(**LAYERS["2048-iq4"])
    L, H = synth.build_layer(spec), P.host_layer(spec)
    import oracle as O
    found = {83: [], 84: []}
    for seed in range(600, 1400):
        x = synth.inputs(seed, 9, spec.width)
        rows = np.bincount(O.route(H.logits(x))[0].ravel(), minlength=512)
        if rows.max() <= 8 and (rows > 0).sum() in found:
            found[int((rows > 0).sum())].append(x)
    lib = qg.lib()
    begin, end = lib.qg_event_create(), lib.qg_event_create()

    def layer_us(x):
        fw, graph = P.forward(L, x), qg.C.c_void_p()
        qg.call("graph_begin", qg.C.byref(graph))
        for _ in range(10):
            fw.run(L, 9)
        qg.call("graph_end", graph)
        best = float("inf")
        for _ in range(10):
            qg.call("event_record", begin)
            qg.call("graph_launch", graph)
            qg.call("event_record", end)
            qg.call("sync")
            ms = qg.C.c_float()
            qg.call("event_elapsed", qg.C.byref(ms), begin, end)
            best = min(best, ms.value * 100)
        lib.qg_graph_destroy(graph)
        return best

    try:
        # in pairs, so that both sides see the same clocks; a slow box gets three tries (the slower form never passes)
        for _ in range(3):
            ratio = float(np.median([layer_us(b) / layer_us(a) for a, b in list(zip(found[83], found[84]))[:9]]))
            print(f"9 tokens: 84 experts / 83 experts {ratio:.3f}", flush=True, file=sys.stderr)
            if ratio < 1.02:
                break
    finally:
        lib.qg_event_destroy(begin)
        lib.qg_event_destroy(end)
    assert ratio < 1.02
