"""Chunk attention of calls too small to fill the chip: their page walks are cut into ranges whose partial
results a second kernel puts together.  Against the CPU oracle at the bars of test_gpu_prefill.py, over the
places where the cut can go wrong: ranges that end inside a page pair, ranges wholly past some rows' positions,
uncut blocks beside cut ones, empty chunks, one row to several row blocks."""
import numpy as np
import pytest

from breccia_amd import lib as L
from breccia_amd.kv import BkvError, DeviceBuffer, Graph, Stream, device_sync
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
    (16, [(8000, 100)]),                                 # f16: two work-groups a compute unit, the workspace nearly full
    (2, [(9990, 20)]),                                   # 63 ranges in a row block: the merge has 64 lanes for them
])
def test_cut_chunks_match_the_oracle(n_q, cases, layout):
    rng = np.random.Generator(np.random.PCG64(77 + n_q))
    with Twin(n_pages=640, max_seqs=4, layout=layout) as tw:
        tw.pool.fill(0xFF)
        for img in tw.images:
            img.k[:] = 0xFF
            img.v[:] = 0xFF
        tw.pool.set_free_order(rng.permutation(640).astype(np.int32))
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
    # 150 and 100 work-groups' worth of rows, walks of 60 to 79 and of 1 to 13 pairs of pages: the long ones are cut
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


class Chunk:
    """Query rows of `t` tokens behind `before` cells of sequence s, and room for their outputs, on the device."""

    def __init__(self, tw, s, before, t, rng, n_q=16):
        self.tw, self.s, self.before, self.t, self.n_q = tw, s, before, t, n_q
        self.q = rng.standard_normal((t, n_q, 256)).astype(np.float32)
        self.qd, self.od = DeviceBuffer.from_numpy(self.q), DeviceBuffer(self.q.nbytes)
        device_sync()

    def run(self, stream=None):
        self.tw.pool.prefill_attn(0, [self.s], [self.before], [self.t], self.n_q, self.qd, self.od, 1.0 / 16.0, stream=stream)

    def clear(self):
        self.od.upload(np.zeros(self.q.shape, np.float32))

    def out(self):
        return self.od.download(np.float32).reshape(self.q.shape)

    def serial(self):
        """What the call returns with nothing beside it."""
        device_sync()
        self.run()
        device_sync()
        out = self.out()
        self.clear()
        return out

    def free(self):
        self.qd.free()
        self.od.free()


def test_a_captured_chunk_stays_uncut():
    # its replays leave the pool's workspaces to the calls beside them: the bits of the uncut call, next to a cut call
    # on other inputs that runs at the same time
    rng = np.random.Generator(np.random.PCG64(78))
    with Twin(n_pages=100, max_seqs=2) as tw:
        s = tw.pool.seq_create()
        fill(tw, s, 600, rng, chunk=600)
        big = tw.pool.seq_create()
        fill(tw, big, 900, rng, chunk=900)
        chunk, other = Chunk(tw, s, 570, 30, rng), Chunk(tw, s, 570, 30, rng)
        # beside a chunk that fills the chip it is uncut (f16 pools), with the same bits whatever the company
        uncut = prefill(tw, 0, [s, big], [570, 0], [chunk.q, np.zeros((900, 16, 256), np.float32)], 16)[0]
        assert not np.array_equal(uncut, chunk.serial()), "cut and uncut differ in some last bit"
        for i in (0, 29):
            check_attn(uncut[i], tw.oracle_attend(0, s, 570 + i, chunk.q[i], 16), "token %d" % i)
        cut = other.serial()
        one, two = Stream(), Stream()
        other.run(two)
        graph = Graph(one)
        chunk.run(one)
        graph.end()
        for _ in range(4):
            device_sync()
            chunk.clear()
            other.clear()
            graph.launch(one)
            other.run(two)
            graph.launch(one)
            device_sync()
            assert np.array_equal(chunk.out(), uncut)
            assert np.array_equal(other.out(), cut)
        graph.destroy()
        for x in (one, two):
            x.close()
        for x in (chunk, other):
            x.free()


@pytest.mark.parametrize("n_streams", [2, 6])
@pytest.mark.parametrize("layout", [L.LAYOUT_F16, L.LAYOUT_I8H])
def test_cut_chunks_on_several_streams_at_once(layout, n_streams):
    # streams with a workspace of their own and, beyond four, streams that share one: nothing waits on the host
    # between the calls, and every output has the bits of the same call alone
    rng = np.random.Generator(np.random.PCG64(81))
    with Twin(n_pages=300, max_seqs=2, layout=layout) as tw:
        s = tw.pool.seq_create()
        fill(tw, s, 3100, rng, chunk=1024)
        streams = [Stream() for _ in range(n_streams)]
        chunks = [Chunk(tw, s, 3000 - 37 * i, 60 + 7 * i, rng) for i in range(n_streams)]
        want = [c.serial() for c in chunks]
        for _ in range(4):
            for _ in range(3):
                for c, x in zip(chunks, streams):
                    c.run(x)
            device_sync()
            for i, (c, w) in enumerate(zip(chunks, want)):
                assert np.array_equal(c.out(), w), i
                c.clear()
            device_sync()
        for x in streams:
            x.close()
        for c in chunks:
            c.free()


def test_cut_chunks_after_their_streams_are_gone():
    # the streams of earlier chunks are destroyed, another has work left and a third is being captured: the next chunk
    # neither waits on the host nor disturbs the capture
    rng = np.random.Generator(np.random.PCG64(82))
    with Twin(n_pages=100, max_seqs=2) as tw:
        s = tw.pool.seq_create()
        fill(tw, s, 600, rng, chunk=600)
        long, busy = Chunk(tw, s, 0, 600, rng, n_q=64), Stream()
        chunk, captured = Chunk(tw, s, 570, 30, rng), Chunk(tw, s, 500, 40, rng)
        want = chunk.serial()
        capturing = Stream()
        for _ in range(3):
            fresh, *gone = [Stream() for _ in range(6)]  # first, so that it is none of the destroyed ones' handles
            for x in gone:
                chunk.run(x)
            for x in gone:
                x.sync()
                x.close()
            for _ in range(500):  # some 0.1 ms each
                long.run(busy)
            graph = Graph(capturing)
            captured.run(capturing)
            chunk.run(fresh)
            graph.end()
            with pytest.raises(BkvError) as ei:
                busy.wait(1)
            assert ei.value.status == L.ERR_TIMEOUT, "the call waited for everything on the device"
            fresh.sync()
            assert np.array_equal(chunk.out(), want)
            chunk.clear()
            graph.launch(capturing)
            device_sync()
            for i in (0, 39):
                check_attn(captured.out()[i], tw.oracle_attend(0, s, 500 + i, captured.q[i], 16), "token %d" % i)
            captured.clear()
            graph.destroy()
            fresh.close()
        for x in (capturing, busy):
            x.close()
        for c in (chunk, captured, long):
            c.free()


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
