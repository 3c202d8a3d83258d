"""qg_matmul's choice of kernels by size.  Each form gives the reference's bits,
so the batches on both sides of every limit are compared with the oracle bit
for bit; and where a size had been sent to the slower form, its time is held
against that of a size that has always been on the faster one."""
import sys

import numpy as np
import pytest

import oracle as O
from nebula_amd import qg
from nebula_amd.qg import Device, call
from test_gpu_exact_tiles import run
from test_oracle_cpu import legal_blocks

pytestmark = pytest.mark.gpu


def check(typ, rows, cols, tokens):
    rng = np.random.default_rng(100 * typ + rows + cols)
    w = np.ascontiguousarray(legal_blocks(rng, typ, rows, cols))
    for nt in tokens:
        print(f"matmul route type={typ} {rows}x{cols} nt={nt}", flush=True, file=sys.stderr)
        x = rng.normal(0, .5, (nt, cols)).astype(np.float32)
        np.testing.assert_array_equal(run(typ, w, rows, cols, x).view('u4'), O.matmul(w, typ, rows, cols, x).view('u4'),
                                      err_msg=f"type {typ} {rows}x{cols} nt {nt}")


def graph_us(typ, rows, cols, nt):
    """Time of one call in a graph of 20, the least of 15 replays."""
    lib = qg.lib()
    w, x, out = Device(nbytes=rows * qg.row_bytes(typ, cols)), Device(nbytes=nt * cols * 4), Device(nbytes=nt * rows * 4)
    begin, end, graph = lib.qg_event_create(), lib.qg_event_create(), qg.C.c_void_p()
    best = float("inf")
    call("matmul", out.p, w.p, typ, rows, cols, x.p, nt)
    call("graph_begin", qg.C.byref(graph))
    for _ in range(20):
        call("matmul", out.p, w.p, typ, rows, cols, x.p, nt)
    call("graph_end", graph)
    try:
        for _ in range(15):
            call("event_record", begin)
            call("graph_launch", graph)
            call("event_record", end)
            call("sync")
            ms = qg.C.c_float()
            call("event_elapsed", qg.C.byref(ms), begin, end)
            best = min(best, ms.value * 1e3 / 20)
    finally:
        lib.qg_graph_destroy(graph)
        lib.qg_event_destroy(begin)
        lib.qg_event_destroy(end)
    print(f"matmul type={typ} {rows}x{cols} nt={nt}: {best:.2f} us", flush=True, file=sys.stderr)
    return best


def time_ratio(a, b, limit):
    """Time of call a over call b: the least of up to three tries (a box may be busy), each with both sides in turn."""
    ratio = float("inf")
    for _ in range(3):
        ratio = min(ratio, graph_us(*a) / graph_us(*b))
        if ratio < limit:
            break
    return ratio


@pytest.mark.parametrize("rows,tokens", [(1, (33, 64, 65)), (48, (64, 65)), (512, (17, 24, 25)), (1100, (11, 12)), (6200, (1, 2))])
def test_f32_limits(qgl, rows, tokens):
    check(0, rows, 256, tokens)


def test_f32_few_rows_stay_on_the_vector_chains(qgl):
    """48 x 6144 takes no longer at 33 tokens than at 32 (the matrix-core tiles take 1.8 times as long)."""
    assert time_ratio((0, 48, 6144, 33), (0, 48, 6144, 32), 1.3) < 1.3


@pytest.mark.parametrize("typ", [12, 20])
@pytest.mark.parametrize("rows,cols", [(7, 256), (2048, 768), (2057, 512), (2057, 768), (2457, 2560), (2458, 2560)])
def test_quantised_5_to_8_tokens(qgl, typ, rows, cols):
    check(typ, rows, cols, (5, 7, 8, 9))


@pytest.mark.parametrize("typ,rows,cols", [(12, 512, 512), (12, 6144, 256), (20, 6144, 256)])
def test_quantised_5_tokens_against_the_tiles(qgl, typ, rows, cols):
    """5 tokens of a small matrix take less time than 9, which the matrix-core tiles serve (their time is the same
    at 5..16 tokens: 5.3 us against 4.1, 5.9 against 4.8, 5.6 against 5.1)."""
    assert time_ratio((typ, rows, cols, 5), (typ, rows, cols, 9), 0.97) < 0.97


@pytest.mark.parametrize("rows,tokens", [(512, (21, 65)), (2560, (70,)), (6144, (33, 130)), (10240, (21, 32, 33, 65))])
def test_iq4nl_tile_choices(qgl, rows, tokens):
    check(20, rows, 256, tokens)


@pytest.mark.parametrize("rows,nt", [(10240, 24), (10240, 70), (6144, 130)])
def test_iq4nl_tiles_as_q4k(qgl, rows, nt):
    """IQ4_NL, whose weights take somewhat more to decode, stays near Q4_K of the same sizes (at most 13 % behind over
    17..1024 tokens where both take the same tile) where 64-token tiles would be mostly padding (1.45 to 1.6 times)."""
    assert time_ratio((20, rows, 2560, nt), (12, rows, 2560, nt), 1.25) < 1.25


def test_output_past_one_launch(qgl):
    """Q8_0, 1048592 rows x 2064 tokens: 65537 row tiles x 129 token tiles are more workgroups than one launch holds
    (2^23 - 1 of 512 threads); the output has 2.2e9 elements.  Sampled rows of the tokens around the cut (127 token
    tiles, 2032 tokens) and at both ends, bit for bit."""
    rows, cols, nt = 65537 * 16, 256, 2064
    rng = np.random.default_rng(8)
    w = np.ascontiguousarray(legal_blocks(rng, 8, 4096, cols))
    w = np.ascontiguousarray(np.resize(w, (rows, w.shape[1])))   # the 4096 rows, repeated
    w[-16:] = legal_blocks(rng, 8, 16, cols)
    x = rng.normal(0, .5, (nt, cols)).astype(np.float32)
    dw, dx = Device(w), Device(x)
    out = qg.lib().qg_alloc(rows * nt * 4)
    assert out
    try:
        print(f"matmul past one launch {rows}x{cols} nt={nt}", flush=True, file=sys.stderr)
        call("matmul", out, dw.p, 8, rows, cols, dx.p, nt)
        call("sync")
        pick = np.r_[0:40, 4080:4112, rows // 2:rows // 2 + 16, rows - 32:rows]
        for t in (0, 1000, 2031, 2032, 2047, 2048, nt - 1):
            got = np.empty(rows, np.float32)
            call("read", got.ctypes.data, out + t * rows * 4, got.nbytes)
            want = O.matmul(np.ascontiguousarray(w[pick]), 8, len(pick), cols, x[t:t + 1])[0]
            np.testing.assert_array_equal(got[pick].view('u4'), want.view('u4'), err_msg=f"token {t}")
    finally:
        qg.lib().qg_free(out)
