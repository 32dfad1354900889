"""Chunk attention of calls too small to fill the chip: their page walks are cut into ranges whose partial
results a second kernel puts together.  Against the CPU oracle at the bars of test_gpu_prefill.py, over the
places where the cut can go wrong: ranges that end inside a page pair, ranges wholly past some rows' positions,
uncut blocks beside cut ones, empty chunks, one row to several row blocks."""
import numpy as np
import pytest

from breccia_amd import lib as L
from breccia_amd.kv import DeviceBuffer, Graph, Stream, device_sync
from gpu_common import REF_BAR_MAX_REL, Twin, check_attn
from test_gpu_attn import fill
from test_gpu_prefill import prefill

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", [L.LAYOUT_F16, L.LAYOUT_Q8V, L.LAYOUT_I8H])
@pytest.mark.parametrize("n_q, cases", [
    (16, [(517, 41)]),
    (16, [(2999, 1)]),                                   # one row block, one live wave
    (24, [(0, 239), (4081, 3)]),                         # blocks of one entry uncut beside cut ones
    (6, [(700, 77), (0, 0), (0, 9), (1535, 33)]),        # groups of 3 rows, an empty chunk, a chunk too short to cut
    (2, [(0, 600)]),                                     # ranges past the positions of their block's first rows
])
def test_cut_chunks_match_the_oracle(n_q, cases, layout):
    rng = np.random.Generator(np.random.PCG64(77 + n_q))
    with Twin(n_pages=500, max_seqs=4, layout=layout) as tw:
        tw.pool.fill(0xFF)
        for img in tw.images:
            img.k[:] = 0xFF
            img.v[:] = 0xFF
        tw.pool.set_free_order(rng.permutation(500).astype(np.int32))
        seqs = [tw.pool.seq_create() for _ in cases]
        for s, (before, t) in zip(seqs, cases):
            if before + t:
                fill(tw, s, before + t, rng, chunk=1024)
        qs = [rng.standard_normal((t, n_q, 256)).astype(np.float32) for _, t in cases]
        gates = [rng.standard_normal((t, n_q, 256)).astype(np.float32) for _, t in cases]
        tw.pool.timing_enable(True)
        outs = prefill(tw, 0, seqs, [b for b, _ in cases], qs, n_q, gates)
        device_sync()
        tw.pool.timing_enable(False)
        assert tw.pool.timing_read(L.STAGE_PREFILL_ATTN)[0] == 1
        assert tw.pool.timing_read(L.STAGE_ATTN_MERGE)[0] == 1, "the call was meant to be cut"
        for s, (before, t), q, g, out in zip(seqs, cases, qs, gates, outs):
            for i in sorted({0, t // 3, t // 2, t - 1} & set(range(t))):
                want = tw.oracle_attend(0, s, before + i, q[i], n_q, gate=g[i])
                _, rel = check_attn(out[i], want, "chunk at %d, token %d" % (before, i))
                assert rel <= REF_BAR_MAX_REL, (before, i, rel)


@pytest.mark.parametrize("layout", [L.LAYOUT_Q8V, L.LAYOUT_I8H])
def test_an_unbalanced_call_that_fills_the_chip(layout):
    # 150 and 100 work-groups' worth of rows, walks of 60 to 68 and of 1 to 13 pairs of pages: the long ones are cut
    rng = np.random.Generator(np.random.PCG64(79))
    cases = [(0, 400), (1900, 600)]
    with Twin(n_pages=400, n_kv=2, max_seqs=4, layout=layout) as tw:
        tw.pool.set_free_order(rng.permutation(400).astype(np.int32))
        seqs = [tw.pool.seq_create() for _ in cases]
        for s, (before, t) in zip(seqs, cases):
            fill(tw, s, before + t, rng, chunk=1024)
        qs = [rng.standard_normal((t, 32, 256)).astype(np.float32) for _, t in cases]
        tw.pool.timing_enable(True)
        outs = prefill(tw, 0, seqs, [b for b, _ in cases], qs, 32)
        device_sync()
        tw.pool.timing_enable(False)
        assert tw.pool.timing_read(L.STAGE_ATTN_MERGE)[0] == 1, "the call was meant to be cut"
        for s, (before, t), q, out in zip(seqs, cases, qs, outs):
            for i in (0, 7, 199, t // 2 + 3, t - 1):
                _, rel = check_attn(out[i], tw.oracle_attend(0, s, before + i, q[i], 32), "chunk at %d, token %d" % (before, i))
                assert rel <= REF_BAR_MAX_REL, (before, i, rel)


def test_a_captured_chunk_replays():
    # a captured call stays uncut (its replays leave the pool's workspace to the calls beside them)
    rng = np.random.Generator(np.random.PCG64(78))
    with Twin(n_pages=100, max_seqs=2) as tw:
        s = tw.pool.seq_create()
        fill(tw, s, 600, rng, chunk=600)
        q = rng.standard_normal((30, 16, 256)).astype(np.float32)
        eager = prefill(tw, 0, [s], [570], [q], 16)[0]
        qd, od = DeviceBuffer.from_numpy(q), DeviceBuffer(q.nbytes)
        stream = Stream()
        graph = Graph(stream)
        tw.pool.prefill_attn(0, [s], [570], [30], 16, qd, od, 1.0 / 16.0, stream=stream)
        graph.end()
        for _ in range(3):
            od.upload(np.zeros(q.shape, np.float32))
            graph.launch(stream)
            again = prefill(tw, 0, [s], [570], [q], 16)[0]
            assert np.array_equal(again, eager)
            device_sync()
            got = od.download(np.float32).reshape(q.shape)
            for i in (0, 29):
                check_attn(got[i], tw.oracle_attend(0, s, 570 + i, q[i], 16), "token %d" % i)
        graph.destroy()
        stream.close()
        qd.free()
        od.free()


def test_a_cut_chunk_leaves_captures_on_other_streams_alone():
    # a chunk before the capture of a decode call and one during it, on streams outside the capture
    rng = np.random.Generator(np.random.PCG64(80))
    with Twin(n_pages=100, max_seqs=2) as tw:
        s = tw.pool.seq_create()
        fill(tw, s, 600, rng, chunk=600)
        q = rng.standard_normal((30, 16, 256)).astype(np.float32)
        qd, od = DeviceBuffer.from_numpy(q), DeviceBuffer(q.nbytes)
        last, cd = DeviceBuffer.from_numpy(q[29]), DeviceBuffer(q[29].nbytes)
        one, two = Stream(), Stream()
        device_sync()
        tw.pool.prefill_attn(0, [s], [570], [30], 16, qd, od, 1.0 / 16.0, stream=one)
        one.sync()
        want = od.download(np.float32)
        graph = Graph(two)
        tw.pool.decode_attn(0, [s], [599], 16, last, cd, 1.0 / 16.0, stream=two)
        graph.end()
        graph_again = Graph(one)  # the stream of the chunk is captured now
        tw.pool.prefill_attn(0, [s], [570], [30], 16, qd, od, 1.0 / 16.0, stream=one)
        tw.pool.prefill_attn(0, [s], [570], [30], 16, qd, od, 1.0 / 16.0, stream=two)
        graph_again.end()
        two.sync()
        got = od.download(np.float32)
        check_attn(got.reshape(q.shape)[29], tw.oracle_attend(0, s, 599, q[29], 16), "chunk beside a capture")
        for _ in range(3):
            cd.upload(np.zeros(q[29].shape, np.float32))
            tw.pool.prefill_attn(0, [s], [570], [30], 16, qd, od, 1.0 / 16.0, stream=one)
            one.sync()
            assert np.array_equal(od.download(np.float32), want)
            graph.launch(two)
            two.sync()
            check_attn(cd.download(np.float32).reshape(16, 256), tw.oracle_attend(0, s, 599, q[29], 16), "replayed decode")
        graph_again.destroy()
        graph.destroy()
        for x in (one, two):
            x.close()
        for x in (qd, od, last, cd):
            x.free()
