"""Ranges of one page a wave (what short contexts are cut into: four pages a work-group), against the oracle: dense, as
the fused step and over selection lists, on all layouts, at the edges of pages and of ranges, in pools whose other cells
hold 0xFF.  Up to 64 entries a call: each work-group finds its entry with one lane per entry."""
import numpy as np
import pytest

from breccia_amd import lib as L
from breccia_amd.kv import attn_plan, device_info
from gpu_common import REF_BAR_MAX_REL, Twin, check_attn
from test_gpu_attn_select import oracle_select, select_attn
from test_gpu_step import step

pytestmark = pytest.mark.gpu

EDGES = [1, 2, 15, 16, 17, 33, 47, 48, 49, 63, 64, 65, 81, 127, 128, 129, 257]
SHAPES = [(2, 8, EDGES), (1, 16, EDGES[:9]), (2, 12, EDGES[:8]), (4, 4, [64]), (2, 3, (EDGES * 4)[:64])]


@pytest.mark.parametrize("layout", [L.LAYOUT_F16, L.LAYOUT_Q8V, L.LAYOUT_I8H])
@pytest.mark.parametrize("n_kv,group,lens", SHAPES)
def test_dense_step_and_lists_at_the_edges_of_pages_and_ranges(layout, n_kv, group, lens):
    rng = np.random.Generator(np.random.PCG64(4100 + 10 * layout + group + len(lens)))
    n, n_q = len(lens), n_kv * group
    _, pps, _ = attn_plan(device_info()[1], n_kv, n_q, [c - 1 for c in lens])
    assert np.all(pps == 4)
    pages = sum(c // 16 + 1 for c in lens) + 8
    with Twin(n_pages=pages, n_kv=n_kv, max_seqs=n, layout=layout) as tw:
        tw.pool.fill(0xFF)
        tw.pool.set_free_order(rng.permutation(pages).astype(np.int32))
        seqs = [tw.pool.seq_create() for _ in lens]
        for s, c in zip(seqs, lens):
            tw.pool.seq_reserve(s, c + 1)
            rows = rng.standard_normal((2, c, n_kv, 256)).astype(np.float32)
            rows[1, c // 2] *= 30.0  # one loud V row: the quantised layouts' exponents and scales differ
            tw.append(0, [s], [0], [rows[0]], [rows[1]])
        q = rng.standard_normal((n, n_q, 256)).astype(np.float32)
        gate = rng.standard_normal((n, n_q, 256)).astype(np.float32)

        def check(got, pos, what):
            for i, s in enumerate(seqs):
                _, rel = check_attn(got[i], tw.oracle_attend(0, s, pos[i], q[i], n_q, gate=gate[i]), "%s, %d cells" % (what, pos[i] + 1))
                assert rel <= REF_BAR_MAX_REL, (what, pos[i], rel)

        pos = [c - 1 for c in lens]
        check(tw.decode_attn(0, seqs, pos, q, n_q, scale=1.0 / 16.0, gate=gate), pos, "dense")
        if n_kv == 2:
            # every fourth list is empty, the others are shuffled, with a block past the position and one listed twice
            lists = [[] if i % 4 == 3 else list(rng.permutation(c // 4 + 2)[:33]) + [0] for i, c in enumerate(lens)]
            got = select_attn(tw, 0, seqs, pos, q, n_q, lists, max_ids=40, gate=gate)
            for i, s in enumerate(seqs):
                if not any(4 * b <= pos[i] for b in lists[i]):
                    assert not got[i].any(), "an empty list"
                    continue
                want = oracle_select(tw, 0, s, pos[i], q[i], n_q, lists[i], gate=gate[i])
                _, rel = check_attn(got[i], want, "list of %d" % len(lists[i]))
                assert rel <= REF_BAR_MAX_REL, (i, rel)
        new = rng.standard_normal((2, n, n_kv, 256)).astype(np.float32)
        got = step(tw, 0, seqs, list(lens), new[0], new[1], q, n_q, gate=gate)
        for i, s in enumerate(seqs):
            tw.images[0].append(tw.pool.block_table(s), lens[i], new[0, i], new[1, i], capacity_cells=tw.pool.seq_capacity(s))
        check(got, list(lens), "step")
        for i, s in enumerate(seqs):  # the new rows' bytes, and nothing beside them
            table = tw.pool.block_table(s)
            for which, img in ((0, tw.images[0].k), (1, tw.images[0].v)):
                have = tw.pool.read_layer(0, which).reshape(pages, n_kv, 16, -1)[table[lens[i] // 16], :, lens[i] % 16]
                want = img.reshape(pages, n_kv, 16, -1)[table[lens[i] // 16], :, lens[i] % 16]
                assert np.array_equal(have, want), (which, lens[i])
