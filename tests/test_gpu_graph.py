"""GPU: op calls captured into a HIP graph (sile_hip_graph_begin / end) and
replayed.

A graph of GEMMs (one that splits K' when run eagerly, one with N below a tile,
one plain), a row softmax and a causal flash attention is replayed three times,
with eager split GEMMs on another stream and device synchronisations in between.
Every replay is checked: the ops whose captured form equals the eager one bit for
bit against the eager result, two GEMMs against the oracle (|g - r| <= 2e-2 +
1e-2 |r|, fp32 out 1e-4) and against the first replay bit for bit.  Another graph
holds the forms that this one leaves out: a GEMM that takes the transposed form
eagerly, a few-rows one, one with unaligned C rows, and an fp32 attention with
key ranges eagerly.
"""
import os
import subprocess
import sys

import numpy as np
import pytest

from oracle import cpuref
from tests.helpers import assert_close, bf16_round, rng, say

pytestmark = pytest.mark.gpu


def _bf16_operands(seed, m, n, k):
    a = (rng(seed).normal(size=(m, k)) / np.sqrt(k)).astype(np.float32)
    bt = (rng(seed + 1).normal(size=(n, k)) / np.sqrt(k)).astype(np.float32)
    (qa, a_f), (qb, b_f) = bf16_round(a), bf16_round(bt)
    return qa, qb, cpuref.gemm_nt(a_f, b_f)


def test_graph_replays_op_calls(hip):
    say("graph: capture gemm x3 + softmax + flash attention, replay x3")
    st, other = hip.Stream(), hip.Stream()
    gemms = []
    # (m, n, k, out): split K' eagerly; N < 128; plain 128 tiles
    for idx, (m, n, k, out) in enumerate([(256, 256, 8192, hip.F32), (512, 64, 256, hip.BF16),
                                          (512, 512, 512, hip.BF16)]):
        qa, qb, ref = _bf16_operands(70 + 2 * idx, m, n, k)
        cb = 4 if out == hip.F32 else 2
        bufs = (hip.DeviceBuffer.from_array(qa), hip.DeviceBuffer.from_array(qb),
                hip.DeviceBuffer(m * n * cb))
        gemms.append((m, n, k, out, cb, ref, bufs))
    rows, cols = 64, 4096
    x = (rng(80).normal(size=(rows, cols)) * 2.0).astype(np.float16)
    dx, dy = hip.DeviceBuffer.from_array(x), hip.DeviceBuffer(rows * cols * 2)
    b, h, s, d = 1, 2, 512, 128
    qkv = [rng(81 + i).normal(size=(b, h, s, d)).astype(np.float16) for i in range(3)]
    dq, dk, dv = (hip.DeviceBuffer.from_array(t) for t in qkv)
    do = hip.DeviceBuffer(b * h * s * d * 2)
    scale = 1.0 / np.sqrt(d)

    def calls(stream):
        for m, n, k, out, cb, ref, (da, db, dc) in gemms:
            hip.gemm(hip.BF16, hip.BF16, out, m, n, k, da.ptr, k, hip.ROW_MAJOR, db.ptr, k,
                     hip.COL_MAJOR, dc.ptr, n, 1.0, 1.0, 0, stream)
        hip.softmax_rows(hip.F16, hip.F16, rows, cols, dx.ptr, cols, dy.ptr, cols, stream)
        hip.flash_attn_fwd(hip.F16, b, h, s, d, dq.ptr, dk.ptr, dv.ptr, do.ptr, scale, True,
                           stream)

    def outputs():
        res = [dc.download(np.uint32 if cb == 4 else np.uint16, (m, n))
               for m, n, k, out, cb, ref, (da, db, dc) in gemms]
        return res + [dy.download(np.uint16, (rows, cols)), do.download(np.uint16, (b, h, s, d))]

    def clear():
        for *_, (da, db, dc) in gemms:
            dc.fill_bytes(0xFF)
        dy.fill_bytes(0xFF)
        do.fill_bytes(0xFF)
        hip.synchronize()

    clear()
    calls(st)
    st.synchronize()
    eager = outputs()

    # eager work that uses the device scratch, queued between the replays
    qa, qb, ref_o = _bf16_operands(90, 256, 512, 8192)
    ea, eb = hip.DeviceBuffer.from_array(qa), hip.DeviceBuffer.from_array(qb)
    ec = hip.DeviceBuffer(256 * 512 * 4)

    with hip.Graph(st) as graph:
        calls(st)
    first = None
    for rep in range(3):
        clear()
        graph.launch()
        hip.gemm(hip.BF16, hip.BF16, hip.F32, 256, 512, 8192, ea.ptr, 8192, hip.ROW_MAJOR,
                 eb.ptr, 8192, hip.COL_MAJOR, ec.ptr, 512, 1.0, 1.0, 0, other)
        st.synchronize()
        other.synchronize()
        got = outputs()
        say(f"graph replay {rep}")
        # plain GEMM, softmax and attention: the captured launches are the eager ones
        for i in (2, 3, 4):
            assert (got[i] == eager[i]).all(), f"replay {rep}: output {i} differs from eager"
        # the two others (the first runs without the scratch under capture): the oracle
        for i in (0, 1):
            m, n, k, out, cb, ref, _ = gemms[i]
            val = (got[i].view(np.float32) if cb == 4
                   else cpuref.f32_from_bf16(got[i]))
            tol = (1e-4, 1e-4) if cb == 4 else (2e-2, 1e-2)
            assert_close(val, ref, atol=tol[0], rtol=tol[1], what=f"replay {rep} gemm {i}")
        if first is None:
            first = got
        else:
            for i in range(5):
                assert (got[i] == first[i]).all(), f"replay {rep}: output {i} changed"
        assert_close(ec.download(np.float32, (256, 512)), ref_o, atol=1e-4, rtol=1e-4,
                     what=f"eager split GEMM beside replay {rep}")
    graph.close()
    for buf in [x for *_, bufs in gemms for x in bufs] + [dx, dy, dq, dk, dv, do, ea, eb, ec]:
        buf.close()
    st.close()
    other.close()


def test_graph_replays_other_forms(hip):
    say("graph: C^T shape, few rows, unaligned C, fp32 attention, replay x3")
    st, other = hip.Stream(), hip.Stream()
    # (m, n, k, ldc, same launches under capture)
    gemms = []
    for idx, (m, n, k, ldc, same) in enumerate([(512, 96, 4096, 96, False), (16, 2048, 2048, 2048, True),
                                                (300, 258, 256, 259, True)]):
        qa, qb, ref = _bf16_operands(30 + 2 * idx, m, n, k)
        gemms.append((m, n, k, ldc, same, ref, (hip.DeviceBuffer.from_array(qa), hip.DeviceBuffer.from_array(qb),
                                                hip.DeviceBuffer(m * ldc * 4))))
    n_q, n_k, d = 100, 2000, 64
    q, kt, v = (rng(50 + i).normal(size=z).astype(np.float32) for i, z in enumerate([(n_q, d), (d, n_k), (n_k, d)]))
    att = [hip.DeviceBuffer.from_array(x) for x in (q, kt, v)]
    do = hip.DeviceBuffer(n_q * d * 4)
    aref = cpuref.dsl_attention_f32(q, kt, v, n_k, 0.125, -1e30, d=d, n_q=n_q, s_k=n_k)

    def calls(stream, outs):
        for (m, n, k, ldc, _, _, (da, db, _)), out in zip(gemms, outs):
            hip.gemm(hip.BF16, hip.BF16, hip.F32, m, n, k, da.ptr, k, hip.ROW_MAJOR, db.ptr, k,
                     hip.COL_MAJOR, out.ptr, ldc, 1.0, 1.0, 0, stream)
        hip.attention_f32_kt(n_q, n_k, d, att[0].ptr, d, att[1].ptr, n_k, att[2].ptr, d, outs[-1].ptr, d, 0.125,
                             -1e30, stream)

    outs = [g[-1][2] for g in gemms] + [do]
    beside = [hip.DeviceBuffer(g[0] * g[3] * 4) for g in gemms] + [hip.DeviceBuffer(n_q * d * 4)]

    def results(bufs):
        return [b.download(np.float32, (g[0], g[3]))[:, :g[1]] for g, b in zip(gemms, bufs)] + [
            bufs[-1].download(np.float32, (n_q, d))]

    def check(res, what):
        for g, got in zip(gemms, res):
            assert_close(got, g[5], atol=1e-4, rtol=1e-4, what=f"{what} gemm {g[:3]}")
        assert_close(res[-1], aref, atol=1e-5, rtol=1e-4, what=f"{what} attention")

    calls(st, outs)
    st.synchronize()
    eager = results(outs)
    check(eager, "eager")
    with hip.Graph(st) as graph:
        calls(st, outs)
    first = None
    for rep in range(3):
        for b in outs + beside:
            b.fill_bytes(0xFF)
        hip.synchronize()
        graph.launch()
        calls(other, beside)     # the scratch forms, eagerly beside the replay
        st.synchronize()
        other.synchronize()
        say(f"graph replay {rep}")
        got, near = results(outs), results(beside)
        check(got, f"replay {rep}")
        for i, g in enumerate(gemms):
            assert not g[4] or (got[i] == eager[i]).all(), f"replay {rep}: gemm {i} differs from eager"
        for i, x in enumerate(near):
            assert (x == eager[i]).all(), f"beside replay {rep}: output {i} differs"
        first = first or got
        assert all((x == y).all() for x, y in zip(got, first)), f"replay {rep} changed"
    graph.close()
    for b in [x for g in gemms for x in g[-1][:2]] + att + outs + beside:
        b.close()
    st.close()
    other.close()


# First use and growth of every scratch slot by eager calls, from the thread that
# is capturing another stream (in a process of its own: the slots are empty).
_CAPTURE_CODE = r"""
import numpy as np
from sile_amd import _abi as hip
hip.init(0)
st, other = hip.Stream(), hip.Stream()
r = np.random.default_rng(1)
x = r.normal(size=(64, 1000)).astype(np.float32)
dx, dy = hip.DeviceBuffer.from_array(x), hip.DeviceBuffer(x.nbytes)
nq, nk, d = 64, 2000, 64
att = [r.normal(size=z).astype(np.float32) for z in ((nq, d), (d, nk), (nk, d))]
da = [hip.DeviceBuffer.from_array(t) for t in att]
do, do2 = hip.DeviceBuffer(nq * d * 4), hip.DeviceBuffer(nq * d * 4)
m = 256
ab = r.integers(0x3f00, 0x3f80, size=(2, 512, 4096)).astype(np.uint16)   # bf16 in [0.5, 1)
dab = [hip.DeviceBuffer.from_array(t) for t in ab]
dbt = hip.DeviceBuffer.from_array(np.ascontiguousarray(ab[1][:100].T))
outs = [hip.DeviceBuffer(512 * 512 * 4) for _ in range(6)]
def attention(out, s):
    hip.attention_f32_kt(nq, nk, d, da[0].ptr, d, da[1].ptr, nk, da[2].ptr, d, out.ptr, d, 0.125, -1e30, s)
def gemm(n, splits, out, s):
    hip.gemm(hip.BF16, hip.BF16, hip.F32, n, n, 4096, dab[0].ptr, 4096, hip.ROW_MAJOR, dab[1].ptr, 4096,
             hip.COL_MAJOR, out.ptr, n, 1.0, 1.0, 0, s, tile=128, splits=splits)
def brow(out, s):   # B row-major of 100 columns: transposed into the scratch first
    hip.gemm(hip.BF16, hip.BF16, hip.F32, 512, 100, 4096, dab[0].ptr, 4096, hip.ROW_MAJOR, dbt.ptr, 100,
             hip.ROW_MAJOR, out.ptr, 100, 1.0, 1.0, 0, s)
def eager(o, g, s):
    attention(o, s)
    gemm(256, 2, g[0], s)
    gemm(512, 8, g[1], s)    # a larger scratch: the first one is freed
    brow(g[2], s)
with hip.Graph(st) as graph:
    hip.softmax_rows(hip.F32, hip.F32, 64, 1000, dx.ptr, 1000, dy.ptr, 1000, st)
    eager(do, outs[:3], other)
graph.launch()
st.synchronize()
other.synchronize()
eager(do2, outs[3:], st)
st.synchronize()
e = np.exp(x.astype(np.float64) - x.max(1, keepdims=True))
assert np.abs(dy.download(np.float32, x.shape) - e / e.sum(1, keepdims=True)).max() < 1e-5
assert (do.download(np.uint32, (nq, d)) == do2.download(np.uint32, (nq, d))).all()
assert np.isfinite(do.download(np.float32, (nq, d))).all()
for i, n in enumerate((256 * 256, 512 * 512, 512 * 100)):
    a, b = outs[i].download(np.float32, (n,)), outs[3 + i].download(np.float32, (n,))
    assert (a == b).all() and a.min() > 500
print("CAPTURE_OK", flush=True)
"""


def test_scratch_allocated_beside_a_capture(hip):
    """Eager calls on one stream, by the thread that captures another: their
    scratch is allocated, grown and freed without ending the capture."""
    say("graph: scratch allocated while another stream is captured")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    run = subprocess.run([sys.executable, "-c", _CAPTURE_CODE], cwd=root, capture_output=True, text=True,
                         timeout=100)
    assert run.returncode == 0 and "CAPTURE_OK" in run.stdout, run.stdout + run.stderr
