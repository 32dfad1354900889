"""GPU parity of the MFMA prefill attention (causal attention of whole chunks over the paged
cache) against the CPU oracle, token by token, and against the decode kernel.  Tolerances as in
test_gpu_attn.py, including the reference's own 1e-5 bar."""
import numpy as np
import pytest

from breccia_amd import lib as L
from breccia_amd.kv import BkvError, DeviceBuffer, device_sync
from gpu_common import REF_BAR_MAX_REL, Twin, check_attn
from helpers import max_abs
from test_gpu_attn import fill

pytestmark = pytest.mark.gpu


def prefill(tw, layer, seqs, pos0, q_list, n_head, gate_list=None):
    """q_list[i]: [T_i, n_head, 256] -> list of outputs of the same shapes (one call)."""
    n_tok = [q.shape[0] for q in q_list]
    qcat = np.ascontiguousarray(np.concatenate([q.reshape(-1) for q in q_list] + [np.zeros(4, np.float32)]),
                                dtype=np.float32)
    qd, od = DeviceBuffer.from_numpy(qcat), DeviceBuffer(qcat.nbytes)
    gd = None
    if gate_list is not None:
        gd = DeviceBuffer.from_numpy(np.concatenate([g.reshape(-1) for g in gate_list] + [np.zeros(4, np.float32)]))
    try:
        tw.pool.prefill_attn(layer, seqs, pos0, n_tok, n_head, qd, od, 1.0 / 16.0, gate_dev=gd,
                             gate_tok_stride=n_head * 256 if gd else 0, gate_head_stride=256 if gd else 0)
        flat = od.download(np.float32, qcat.size)
    finally:
        for b in (qd, od, gd):
            if b is not None:
                b.free()
    outs, at = [], 0
    for t in n_tok:
        outs.append(flat[at:at + t * n_head * 256].reshape(t, n_head, 256))
        at += t * n_head * 256
    return outs


@pytest.mark.parametrize("layout", [L.LAYOUT_F16, L.LAYOUT_Q8V, L.LAYOUT_I8H])
@pytest.mark.parametrize("n_q", [16, 24])
def test_chunks_match_the_oracle_token_by_token(n_q, layout):
    rng = np.random.Generator(np.random.PCG64(1000 + n_q))
    # (cells before the chunk, chunk length): from scratch, on a prefix, single token, page edges
    cases = [(0, 100), (517, 300), (64, 1), (15, 17), (2048, 130)]
    with Twin(n_pages=400, max_seqs=8, layout=layout) as tw:
        tw.pool.set_free_order(rng.permutation(400).astype(np.int32))
        seqs = [tw.pool.seq_create() for _ in cases]
        for s, (before, t) in zip(seqs, cases):
            fill(tw, s, before + t, rng, chunk=1024)            # the chunk's own K/V are in the cache
        qs = [rng.standard_normal((t, n_q, 256)).astype(np.float32) for _, t in cases]
        gates = [rng.standard_normal((t, n_q, 256)).astype(np.float32) for _, t in cases]
        outs = prefill(tw, 0, seqs, [b for b, _ in cases], qs, n_q, gates)
        worst = 0.0
        for s, (before, t), q, g, out in zip(seqs, cases, qs, gates, outs):
            picks = sorted(set([0, t - 1, t // 2] + [int(x) for x in rng.integers(0, t, size=6)] +
                               [i for i in range(t) if (before + i) % 16 in (0, 15)][:6]))
            for i in picks:
                want = tw.oracle_attend(0, s, before + i, q[i], n_q, gate=g[i])
                _, rel = check_attn(out[i], want, "chunk at %d, token %d" % (before, i))
                worst = max(worst, rel)
        assert worst <= REF_BAR_MAX_REL, worst
        # the decode kernel on the same positions agrees to f32 noise
        s, (before, t) = seqs[1], cases[1]
        pos = list(range(before + t - 40, before + t))
        dec = tw.decode_attn(0, [s] * 40, pos, qs[1][-40:], n_q, scale=1.0 / 16.0, gate=gates[1][-40:])
        assert max_abs(dec, outs[1][-40:]) < 5e-6


@pytest.mark.parametrize("layout", [L.LAYOUT_Q8V, L.LAYOUT_I8H])
@pytest.mark.parametrize("v_mag", [1.2e-2, 1.0, 900.0])
def test_quantised_chunks_across_the_scale_range(v_mag, layout):
    # quantised V with block scales from near 2^-14 up to 7, blocks of one row and rows of one page
    # on different scales (the quietest rows of the int8 layout have scales below 2^-14, which pool
    # and oracle alike read as zero): the result stays at the reference's bar relative to the
    # largest output
    rng = np.random.Generator(np.random.PCG64(1020))
    with Twin(n_pages=80, max_seqs=2, layout=layout) as tw:
        s = tw.pool.seq_create()
        n = 1203
        tw.pool.seq_reserve(s, n)
        k = rng.standard_normal((n, 2, 256)).astype(np.float32)
        v = (rng.standard_normal((n, 2, 256)) * v_mag).astype(np.float32)
        v[:, :, 64:96] *= 0.37
        v[5::7] *= 0.11
        v[40:60] *= 1.0e-3      # a page and a half of very quiet rows
        tw.append(0, [s], [0], [k], [v])
        q = rng.standard_normal((203, 16, 256)).astype(np.float32)
        out = prefill(tw, 0, [s], [1000], [q], 16)[0]
        for i in (0, 57, 101, 202):
            want = tw.oracle_attend(0, s, 1000 + i, q[i], 16)
            rel = max_abs(out[i], want) / float(np.max(np.abs(want)))
            assert rel <= REF_BAR_MAX_REL, (i, rel)
        # a short context made of the quiet rows and their neighbours only
        q2 = rng.standard_normal((30, 16, 256)).astype(np.float32)
        out2 = prefill(tw, 0, [s], [35], [q2], 16)[0]
        for i in (0, 10, 29):
            want = tw.oracle_attend(0, s, 35 + i, q2[i], 16)
            rel = max_abs(out2[i], want) / float(np.max(np.abs(want)))
            assert rel <= REF_BAR_MAX_REL, (i, rel)


@pytest.mark.parametrize("rise", [0.0, 4.1])
@pytest.mark.parametrize("n_q, before, tokens, tiny, cut", [
    (16, 0, 130, 64, 0),        # the first tokens see tiny rows only
    (16, 70, 60, 64, 0),
    (16, 600, 41, 64, 1),       # the tiny rows in the first range
    (16, 3000, 41, 1300, 1),    # in several ranges, some of which hold nothing else
    (64, 1400, 1100, 1300, 0),  # more than 1024 of them in one walk
])
def test_rows_of_tiny_values_leave_the_denominator_finite(n_q, before, tokens, tiny, cut, rise):
    # q8_0 V: rows whose block scales lie at 2^-125 are weighed at exp2(logit - 120), and the softmax reference is
    # theirs as long as no larger row follows: the denominator's terms exp2(logit - reference) are then 2^120, and up
    # to 2^126 where the logits rise by the 6 bits the reference may lag behind (4.1 nats).  A handful of such
    # terms is past the end of f32's range.
    rng = np.random.Generator(np.random.PCG64(1022))
    n = before + tokens
    with Twin(n_pages=n // 16 + 8, max_seqs=2, layout=L.LAYOUT_Q8V) as tw:
        s = tw.pool.seq_create()
        tw.pool.seq_reserve(s, n)
        k = (0.05 * rng.standard_normal((n, 2, 256))).astype(np.float32)
        k[:, :, 0] = 0.0
        k[tiny // 2:tiny, :, 0] = rise
        v = rng.standard_normal((n, 2, 256)).astype(np.float32)
        v[:tiny] *= np.float32(3e-36)
        tw.append(0, [s], [0], [k], [v])
        q = (0.3 * rng.standard_normal((tokens, n_q, 256))).astype(np.float32)
        q[:, :, 0] = 16.0
        tw.pool.timing_enable(True)
        out = prefill(tw, 0, [s], [before], [q], n_q)[0]
        device_sync()
        tw.pool.timing_enable(False)
        assert tw.pool.timing_read(L.STAGE_ATTN_MERGE)[0] == cut
        for i in sorted({0, 7, 40, tokens // 2, 63 + tokens // 3, tokens - 1} & set(range(tokens))):
            want = tw.oracle_attend(0, s, before + i, q[i], n_q)
            rel = max_abs(out[i], want) / float(np.max(np.abs(want)))
            assert rel <= REF_BAR_MAX_REL, (i, rel)


@pytest.mark.parametrize("layout", [L.LAYOUT_Q8V, L.LAYOUT_I8H])
def test_quantised_prefill_ignores_poisoned_cells(layout):
    # every unwritten byte of the pools is 0xFF (NaN scales, NaN K): chunks that end inside a page
    rng = np.random.Generator(np.random.PCG64(1021))
    with Twin(n_pages=32, max_seqs=2, layout=layout) as tw:
        tw.pool.fill(0xFF)
        for img in tw.images:
            img.k[:] = 0xFF
            img.v[:] = 0xFF
        s = tw.pool.seq_create()
        for n, t in ((1, 1), (17, 16), (40, 23), (200, 130), (203, 3)):
            fill(tw, s, n, rng, chunk=64)
            q = rng.standard_normal((t, 16, 256)).astype(np.float32)
            out = prefill(tw, 0, [s], [n - t], [q], 16)[0]
            assert np.all(np.isfinite(out))
            for i in sorted({0, t // 2, t - 1}):
                check_attn(out[i], tw.oracle_attend(0, s, n - t + i, q[i], 16), "len %d token %d" % (n, i))


def test_prefill_ignores_poisoned_cells_and_future_tokens():
    rng = np.random.Generator(np.random.PCG64(1010))
    with Twin(n_pages=64, max_seqs=4) as tw:
        s = tw.pool.seq_create()
        fill(tw, s, 200, rng, chunk=200)
        # attend a chunk that ends before the cache does (tokens 100..149): cells 150..199 are real
        # but in the future; cells 200..207 of the last page hold NaN patterns
        kp = tw.pool.read_layer(0, 0).view(np.uint16).copy()
        vp = tw.pool.read_layer(0, 1).view(np.uint16).copy()
        t = tw.pool.block_table(s)
        for c in range(200, 208):
            for h in range(2):
                row = ((int(t[c // 16]) * 2 + h) * 16 + c % 16) * 256
                kp[row:row + 256] = 0x7E00
                vp[row:row + 256] = 0xFE01
        tw.pool.write_layer(0, 0, kp.view(np.uint8))
        tw.pool.write_layer(0, 1, vp.view(np.uint8))
        q = rng.standard_normal((50, 16, 256)).astype(np.float32)
        out = prefill(tw, 0, [s], [100], [q], 16)[0]
        assert np.all(np.isfinite(out))
        for i in (0, 11, 27, 49):
            check_attn(out[i], tw.oracle_attend(0, s, 100 + i, q[i], 16), "token %d" % i)
        # a chunk that ends exactly at the poisoned page's last live cell
        q2 = rng.standard_normal((9, 16, 256)).astype(np.float32)
        out2 = prefill(tw, 0, [s], [191], [q2], 16)[0]
        assert np.all(np.isfinite(out2))
        check_attn(out2[8], tw.oracle_attend(0, s, 199, q2[8], 16), "last cell")


def test_prefill_errors_come_before_any_launch():
    with Twin(n_pages=8, max_seqs=2) as tw:
        s = tw.pool.seq_create()
        tw.pool.seq_reserve(s, 40)
        z = DeviceBuffer(1 << 20)
        for kw, status in [(dict(pos0=[30], n_tokens=[19]), L.ERR_RANGE), (dict(n_q_head=15), L.ERR_INVALID),
                           (dict(q_dev=None), L.ERR_INVALID), (dict(layer=2), L.ERR_RANGE),
                           (dict(seqs=[1]), L.ERR_RANGE)]:
            a = dict(layer=0, seqs=[s], pos0=[0], n_tokens=[40], n_q_head=16, q_dev=z, out_dev=z, scale=0.0625)
            a.update(kw)
            with pytest.raises(BkvError) as ei:
                tw.pool.prefill_attn(**a)
            assert ei.value.status == status, kw
        z.free()


@pytest.mark.parametrize("layout", [L.LAYOUT_F16, L.LAYOUT_Q8V, L.LAYOUT_I8H])
def test_the_largest_batch_of_chunks_in_one_call(layout):
    # 64 chunks (the limit of one call) over 8 sequences, lengths 0..70 tokens, several chunks of
    # one sequence in the same call: every token agrees with the decode kernel at its position, and
    # a sample with the oracle; 65 chunks are refused
    rng = np.random.Generator(np.random.PCG64(1030 + layout))
    with Twin(n_pages=300, max_seqs=10, layout=layout) as tw:
        tw.pool.set_free_order(rng.permutation(300).astype(np.int32))
        lens = [int(x) for x in rng.integers(200, 520, size=8)]
        seqs = [tw.pool.seq_create() for _ in lens]
        for s, n in zip(seqs, lens):
            fill(tw, s, n, rng, chunk=256)
        ent_seq, pos0, n_tok = [], [], []
        for i in range(64):
            j = i % 8
            t = [0, 1, 15, 16, 17, 33, 64, 70][(i // 8 + j) % 8]
            p0 = int(rng.integers(0, lens[j] - t + 1))
            ent_seq.append(seqs[j])
            pos0.append(p0)
            n_tok.append(t)
        qs = [rng.standard_normal((t, 16, 256)).astype(np.float32) for t in n_tok]
        outs = prefill(tw, 0, ent_seq, pos0, qs, 16)
        checked = 0
        for i in range(64):
            t = n_tok[i]
            if t == 0:
                assert outs[i].shape[0] == 0
                continue
            for at in range(0, t, 64):
                m = min(64, t - at)
                dec = tw.decode_attn(0, [ent_seq[i]] * m, list(range(pos0[i] + at, pos0[i] + at + m)),
                                     qs[i][at:at + m], 16, scale=1.0 / 16.0)
                assert max_abs(dec, outs[i][at:at + m]) < 5e-6, (i, at)
            if i % 9 == 0:
                tok = t - 1
                want = tw.oracle_attend(0, ent_seq[i], pos0[i] + tok, qs[i][tok], 16)
                _, rel = check_attn(outs[i][tok], want, "chunk %d" % i)
                assert rel <= REF_BAR_MAX_REL, (i, rel)
                checked += 1
        assert checked >= 5
        z = DeviceBuffer(1 << 16)
        with pytest.raises(BkvError) as ei:
            tw.pool.prefill_attn(0, ent_seq + [seqs[0]], pos0 + [0], [1] * 65, 16, z, z, 0.0625)
        assert ei.value.status == L.ERR_INVALID
        z.free()


@pytest.mark.parametrize("first,head_stride,tok_extra", [(1, 256, 0), (0, 257, 0), (0, 256, 2), (4, 260, 8)])
def test_gate_values_at_any_alignment(first, head_stride, tok_extra):
    # gate values that can be read four at a time, and those that cannot (by their first address, by either stride): the
    # same numbers, so the same bits
    n_q, t = 6, 37
    rng = np.random.Generator(np.random.PCG64(1050))
    tok_stride = n_q * head_stride + tok_extra
    with Twin(n_pages=16, max_seqs=1) as tw:
        s = tw.pool.seq_create()
        fill(tw, s, t, rng, chunk=64)
        q = rng.standard_normal((t, n_q, 256)).astype(np.float32)
        gate = rng.standard_normal((t, n_q, 256)).astype(np.float32) * 3
        want = prefill(tw, 0, [s], [0], [q], n_q, [gate])[0]
        spread = np.zeros(first + t * tok_stride + 4, np.float32)
        for i in range(t):
            for h in range(n_q):
                at = first + i * tok_stride + h * head_stride
                spread[at:at + 256] = gate[i, h]
        qd, gd, od = DeviceBuffer.from_numpy(q), DeviceBuffer.from_numpy(spread), DeviceBuffer(q.nbytes)
        tw.pool.prefill_attn(0, [s], [0], [t], n_q, qd, od, 1.0 / 16.0, gate_dev=gd.ptr.value + 4 * first,
                             gate_tok_stride=tok_stride, gate_head_stride=head_stride)
        got = od.download(np.float32, q.size).reshape(q.shape)
        for b in (qd, gd, od):
            b.free()
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("layout", [L.LAYOUT_F16, L.LAYOUT_Q8V, L.LAYOUT_I8H])
def test_short_walks_of_wide_work_groups(layout):
    # Work-groups of 128 rows (on f16 pools: 544 and more of 64 rows) whose walks are 1 to 9 pairs of pages, odd page counts
    # among them, with waves and lanes that have no query row; every byte that was not written is 0xFF.
    rng = np.random.Generator(np.random.PCG64(1040 + layout))
    befores = [0, 1, 14, 15, 16, 17, 30, 31, 32, 33, 47, 48, 63, 64, 100, 111]
    with Twin(n_pages=320, max_seqs=16, layout=layout) as tw:
        tw.pool.fill(0xFF)
        for img in tw.images:
            img.k[:] = 0xFF
            img.v[:] = 0xFF
        tw.pool.set_free_order(rng.permutation(320).astype(np.int32))
        lens = [int(x) for x in rng.integers(130, 151, size=16)]
        seqs = [tw.pool.seq_create() for _ in befores]
        for s, before, t in zip(seqs, befores, lens):
            fill(tw, s, before + t, rng, chunk=512)
        qs = [rng.standard_normal((t, 16, 256)).astype(np.float32) for t in lens]
        gates = [rng.standard_normal((t, 16, 256)).astype(np.float32) for t in lens]
        outs = prefill(tw, 0, seqs, befores, qs, 16, gates)
        for s, before, t, q, g, out in zip(seqs, befores, lens, qs, gates, outs):
            assert np.all(np.isfinite(out))
            for i in sorted({0, 15, 16, int(rng.integers(17, t - 1)), t - 1}):
                want = tw.oracle_attend(0, s, before + i, q[i], 16, gate=g[i])
                _, rel = check_attn(out[i], want, "chunk at %d, token %d" % (before, i))
                assert rel <= REF_BAR_MAX_REL, (before, i, rel)


@pytest.mark.parametrize("before, tokens, cut", [(0, 37, 0), (517, 41, 1)])
def test_gates_of_any_size_act_as_in_the_decode_kernel(before, tokens, cut):
    # sigmoid(gate) where its exponential is subnormal or 0 (below -87.3, -103.9), saturated, infinite or NaN, and 160000
    # ordinary gates: a row's output is the same bits as its output without a gate times what the decode kernel multiplies by
    # (read off a sequence of one cell whose V is 1).
    n_q = 16
    edges = np.float32([0.0, -0.0, 1e-30, -1e-30, 17.3, -17.3, 87.0, -87.0, -87.3, -87.4, 88.0, -88.0, -88.8, 100.0, -100.0,
                        -103.2, -103.9, -104.5, -110.0, 150.5, -150.5, -3e38, 3e38, np.inf, -np.inf, np.nan])
    rng = np.random.Generator(np.random.PCG64(1060))
    with Twin(n_pages=48, max_seqs=2) as tw:
        s, one = tw.pool.seq_create(), tw.pool.seq_create()
        fill(tw, s, before + tokens, rng, chunk=64)
        tw.pool.seq_reserve(one, 1)
        tw.append(0, [one], [0], [np.zeros((1, 2, 256), np.float32)], [np.ones((1, 2, 256), np.float32)])
        q = rng.standard_normal((tokens, n_q, 256)).astype(np.float32)
        gate = (rng.standard_normal((tokens, n_q, 256)) * 20).astype(np.float32)
        gate[:, :, 3:3 + edges.size] = edges
        sig = tw.decode_attn(0, [one] * tokens, [0] * tokens, q, n_q, scale=1.0 / 16.0, gate=gate)
        # the exponential is good to 1 ulp (2^-23), the sum and the quotient add 2^-24 each; subnormal results have steps of 2^-149
        with np.errstate(over="ignore", invalid="ignore"):
            g = gate.astype(np.float64)
            want = np.where(g >= 0, 1.0 / (1.0 + np.exp(-g)), np.exp(g) / (1.0 + np.exp(g)))
            want[g == np.inf] = 1.0
            off = np.abs(sig.astype(np.float64) - want) <= want * 2.0 ** -22 + 2.0 ** -148
        assert np.all(off | np.isnan(g)) and np.all(np.isnan(sig) == np.isnan(g))
        plain = prefill(tw, 0, [s], [before], [q], n_q)[0]
        tw.pool.timing_enable(True)
        gated = prefill(tw, 0, [s], [before], [q], n_q, [gate])[0]
        device_sync()
        tw.pool.timing_enable(False)
        assert tw.pool.timing_read(L.STAGE_ATTN_MERGE)[0] == cut
        same = gated.view(np.uint32) == (plain * sig).view(np.uint32)
        bad = np.argwhere(~(same | np.isnan(g)))
        assert bad.size == 0, (len(bad), [float(gate[tuple(i)]) for i in bad[:8]])
        assert np.all(np.isnan(gated) == np.isnan(g))


@pytest.mark.parametrize("layout", [L.LAYOUT_F16, L.LAYOUT_Q8V, L.LAYOUT_I8H])
@pytest.mark.parametrize("n_q, before, tokens, bad", [
    (16, 24, 40, 32),     # rows of the first waves end a pair of pages before the work-group does
    (16, 26, 40, 32),     # and those of a wave's first sixteen rows before its others
    (2, 5, 130, 64),      # 128 tokens to a work-group: four pairs of pages between its first rows and its last
    (16, 528 + 26, 41, 576),   # cut
    (16, 26, 2100, 32 * 51),   # f16: 1051 work-groups of 64 rows, so two tiles a wave
])
def test_values_that_are_not_finite_stay_with_later_rows(n_q, before, tokens, bad, layout):
    # V of cell `bad` overflows.  A weight of 0 does not undo that, so rows must not meet the cell's pair of pages at all
    # where the last of their sixteen rows lies before it: the same bits as with an ordinary row there.
    rng = np.random.Generator(np.random.PCG64(1070))
    with Twin(n_pages=(before + tokens) // 16 + 2, max_seqs=1, layout=layout) as tw:
        s = tw.pool.seq_create()
        fill(tw, s, before + tokens, rng, chunk=1024)
        q = rng.standard_normal((tokens, n_q, 256)).astype(np.float32)
        want = prefill(tw, 0, [s], [before], [q], n_q)[0]
        assert np.all(np.isfinite(want))
        kd = DeviceBuffer.from_numpy(rng.standard_normal((1, 2, 256)).astype(np.float32))
        vd = DeviceBuffer.from_numpy(np.full((1, 2, 256), np.inf, np.float32))
        tw.pool.append(0, [s], [bad], [1], kd, vd)
        got = prefill(tw, 0, [s], [before], [q], n_q)[0]
        kd.free()
        vd.free()
        group = n_q // 2
        rows = np.arange(tokens * group)
        last = np.minimum(rows // 16 * 16 + 15, rows[-1]) // group + before  # of the row's sixteen
        clear = (last < bad // 32 * 32).reshape(tokens, group)
        clear = np.concatenate([clear, clear], axis=1)  # two kv heads
        assert np.any(clear) and not np.all(np.isfinite(got))
        assert np.array_equal(got[clear].view(np.uint32), want[clear].view(np.uint32))


@pytest.mark.parametrize("layout", [L.LAYOUT_Q8V, L.LAYOUT_I8H])
@pytest.mark.parametrize("n_q, tokens", [(16, 1), (16, 3), (16, 8), (6, 20), (2, 64)])
def test_blocks_of_few_rows_give_the_same_bits(n_q, tokens, layout):
    # Up to 64 rows of a block of 128 (8, 24, 64, 60, 64 here): a tile of sixteen a wave instead of two.  The same rows in a
    # full block, which takes two, must agree in every bit; the oracle checks a sample.  (f16 pools take blocks of 64 here;
    # their blocks of 128 are those of test_short_walks_of_wide_work_groups.)
    rng = np.random.Generator(np.random.PCG64(1080 + n_q))
    full = 128 // (n_q // 2)
    with Twin(n_pages=48, max_seqs=4, layout=layout) as tw:
        tw.pool.fill(0xFF)
        for img in tw.images:
            img.k[:] = 0xFF
            img.v[:] = 0xFF
        befores = [0, 15, 31, 60]  # at most 188 cells, 6 pairs of pages: a walk of 7 may be cut, and sums in another order
        seqs = [tw.pool.seq_create() for _ in befores]
        q = [rng.standard_normal((full, n_q, 256)).astype(np.float32) for _ in befores]
        for s, before in zip(seqs, befores):
            fill(tw, s, before + tokens, rng, chunk=512)
        few = prefill(tw, 0, seqs, befores, [x[:tokens] for x in q], n_q)
        for s, before, x, out in zip(seqs, befores, q, few):
            _, rel = check_attn(out[-1], tw.oracle_attend(0, s, before + tokens - 1, x[tokens - 1], n_q), "behind %d" % before)
            assert rel <= REF_BAR_MAX_REL, (before, rel)
            fill(tw, s, before + full, rng, chunk=512)
        tw.pool.timing_enable(True)
        full_blocks = prefill(tw, 0, seqs, befores, q, n_q)
        device_sync()
        tw.pool.timing_enable(False)
        assert tw.pool.timing_read(L.STAGE_ATTN_MERGE)[0] == 0, "no walk was meant to be cut"
        for out, wide in zip(few, full_blocks):
            assert np.array_equal(out.view(np.uint32), wide[:tokens].view(np.uint32))


def test_work_group_width_does_not_change_a_bit():
    # On f16 pools a call whose chunks fill the chip runs work-groups of 128 query rows (two tiles of
    # sixteen a wave), a smaller one work-groups of 64 (one tile).  A tile's rows are computed
    # the same way in both, so three chunks in one call (566 work-groups of 64 rows: two tiles a wave) and
    # the same chunks one call each (one; each keeps more than half of the chip busy, so that
    # none has its walks cut) must agree in every bit; the oracle checks a sample.
    rng = np.random.Generator(np.random.PCG64(1234))
    cases = [(100, 700), (37, 650), (515, 900)]
    with Twin(n_pages=200, max_seqs=4) as tw:
        tw.pool.set_free_order(rng.permutation(200).astype(np.int32))
        seqs = [tw.pool.seq_create() for _ in cases]
        for s, (before, t) in zip(seqs, cases):
            fill(tw, s, before + t, rng, chunk=1024)
        qs = [rng.standard_normal((t, 16, 256)).astype(np.float32) for _, t in cases]
        gates = [rng.standard_normal((t, 16, 256)).astype(np.float32) for _, t in cases]
        together = prefill(tw, 0, seqs, [b for b, _ in cases], qs, 16, gates)
        for i, (s, (before, t)) in enumerate(zip(seqs, cases)):
            alone = prefill(tw, 0, [s], [before], [qs[i]], 16, [gates[i]])[0]
            assert np.array_equal(alone.view(np.uint32), together[i].view(np.uint32)), i
            for tok in (0, t - 1, int(rng.integers(0, t))):
                want = tw.oracle_attend(0, s, before + tok, qs[i][tok], 16, gate=gates[i][tok])
                check_attn(together[i][tok], want, "chunk %d, token %d" % (i, tok))
