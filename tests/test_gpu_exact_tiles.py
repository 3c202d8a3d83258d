"""qg_matmul's matrix-core tiles (fp32 MFMA, one k per step) at the sizes where
they can go wrong: the edges of the 16- and 32-row tiles, of the 16-, 20- and
32-token tiles and of the superblock ring, both tile choices, and values whose
chains are subnormal, infinite or NaN.  The contract is the reference's
summation order, so every result equals the oracle's bit for bit (NaN results
compare as NaN: their payload is no part of the contract)."""
import sys

import numpy as np
import pytest

import oracle as O
from nebula_amd.qg import Device, call
from test_oracle_cpu import legal_blocks

pytestmark = pytest.mark.gpu


def run(typ, w, rows, cols, x):
    nt = x.shape[0]
    dw, dx, out = Device(w), Device(x), Device(shape=(nt, rows), dtype=np.float32)
    call("matmul", out.p, dw.p, typ, rows, cols, dx.p, nt)
    return out.get()


@pytest.mark.parametrize("typ,widths", [(0, (128, 384, 2048)), (8, (256, 1280)), (12, (256, 768, 2560)), (20, (256, 768, 2560))])
@pytest.mark.parametrize("rows", [1, 15, 33, 64])
def test_exact_tile_edges(qgl, typ, widths, rows):
    rng = np.random.default_rng(1000 * typ + rows)
    for cols in widths:
        w = np.ascontiguousarray(legal_blocks(rng, typ, rows, cols))
        for nt in (1, 4, 5, 15, 16, 17, 20, 21, 33, 64, 65):
            print(f"exact tiles type={typ} {rows}x{cols} nt={nt}", flush=True, file=sys.stderr)
            x = rng.normal(0, .5, (nt, cols)).astype(np.float32)
            np.testing.assert_array_equal(run(typ, w, rows, cols, x).view('u4'), O.matmul(w, typ, rows, cols, x).view('u4'),
                                          err_msg=f"type {typ} {rows}x{cols} nt {nt}")


@pytest.mark.parametrize("typ,nt", [(12, 300), (20, 300), (0, 300), (0, 2049)])
def test_exact_large_tiles(qgl, typ, nt):
    """Enough tiles for the 32 x 32 choice, with a ragged last tile both ways."""
    rng = np.random.default_rng(nt + typ)
    rows, cols = 1031 if typ else 512, 512
    w = np.ascontiguousarray(legal_blocks(rng, typ, rows, cols))
    x = rng.normal(0, .5, (nt, cols)).astype(np.float32)
    print(f"exact large tiles type={typ} {rows}x{cols} nt={nt}", flush=True, file=sys.stderr)
    np.testing.assert_array_equal(run(typ, w, rows, cols, x).view('u4'), O.matmul(w, typ, rows, cols, x).view('u4'))


@pytest.mark.parametrize("nt", [17, 40])
@pytest.mark.parametrize("typ", [0, 12, 20])
def test_exact_special_values(qgl, typ, nt):
    """Rows of subnormal products and sums, zeros of both signs, infinities
    and NaN: what they do to their own outputs, and nothing to the others."""
    rng = np.random.default_rng(5 + typ + nt)
    rows, cols = 19, 512
    w = np.ascontiguousarray(legal_blocks(rng, typ, rows, cols))
    x = rng.normal(0, .5, (nt, cols)).astype(np.float32)
    x[0] *= np.float32(1e-38)
    x[1] *= np.float32(1e-42)
    x[2] = np.where(rng.random(cols) < .5, np.float32(0), np.float32(-0.0))
    x[3, 7], x[4, 300], x[5, 41] = np.inf, -np.inf, np.nan
    x[6, 3], x[6, 35] = np.inf, -np.inf
    x[7] *= np.float32(1e38)
    print(f"exact special values type={typ} nt={nt}", flush=True, file=sys.stderr)
    with np.errstate(all="ignore"):
        want = O.matmul(w, typ, rows, cols, x)
    got = run(typ, w, rows, cols, x)
    nan = np.isnan(want)
    np.testing.assert_array_equal(np.isnan(got), nan)
    np.testing.assert_array_equal(got[~nan].view('u4'), want[~nan].view('u4'))


@pytest.mark.parametrize("nt", [18, 500, 4101])
def test_prefill_router_tiles(qgl, nt):
    """The prefill router's three tile choices, each with a ragged last tile:
    ids and weights of every token bit for bit, and the outputs (with the
    shared expert, whose gate logit the routing kernel forms) on sampled rows."""
    import test_gpu_prefill as P
    from nebula_amd import synth
    spec = synth.LayerSpec(seed=470, width=512, ff=128, gate_type=12, up_type=12, down_type=20, shared=True, sh_types=(12, 12, 20))
    L, H = synth.build_layer(spec), P.host_layer(spec)
    x = synth.inputs(480 + nt, nt, 512)
    fw = P.forward(L, x)
    P.check_routing(fw, H, x)
    P.check_outputs(fw, L, H, x, P.sample_rows(nt, 10, nt), f"512/128 B={nt}")
