"""Batches on both sides of the line where a batch moves to the smaller of a kernel's argument structs (16 entries):
appends, decode steps, selection lists and block selection at 1, 15, 16, 17 and 64 entries, against the oracle."""
import numpy as np
import pytest

import oracle
from breccia_amd import lib as L
from breccia_amd.kv import Pool
from gpu_common import REF_BAR_MAX_REL, Twin, check_attn
from test_gpu_attn_select import oracle_select, select_attn
from test_gpu_select import gpu_select
from test_gpu_step import step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", [L.LAYOUT_F16, L.LAYOUT_Q8V, L.LAYOUT_I8H])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 64])
def test_every_entry_of_a_batch(n, layout):
    rng = np.random.Generator(np.random.PCG64(5200 + 10 * n + layout))
    lens = [int(c) for c in rng.integers(1, 150, n)]
    with Twin(n_pages=sum(c // 16 + 1 for c in lens) + 8, max_seqs=n, layout=layout) as tw:
        seqs = [tw.pool.seq_create() for _ in lens]
        for s, c in zip(seqs, lens):
            tw.pool.seq_reserve(s, c + 1)
        # all prompts in one call: f32 rows, and again as binary16 rows
        rows = [rng.standard_normal((2, c, 2, 256)).astype(np.float32) for c in lens]
        tw.append(0, seqs, [0] * n, [r[0] for r in rows], [r[1] for r in rows])
        tw.assert_pools_equal()
        codes = [r.astype(np.float16).view(np.uint16) for r in rows]
        tw.append(0, seqs, [0] * n, [c[0] for c in codes], [c[1] for c in codes], f16_rows=True)
        tw.assert_pools_equal()
        q = rng.standard_normal((n, 16, 256)).astype(np.float32)
        pos = [c - 1 for c in lens]
        lists = [list(rng.permutation(c // 4 + 1)[:9]) for c in lens]
        new = rng.standard_normal((2, n, 2, 256)).astype(np.float32)
        dense = tw.decode_attn(0, seqs, pos, q, 16, scale=1.0 / 16.0)
        listed = select_attn(tw, 0, seqs, pos, q, 16, lists, max_ids=16)
        stepped = step(tw, 0, seqs, lens, new[0], new[1], q, 16)
        for i, s in enumerate(seqs):
            wants = [(dense[i], tw.oracle_attend(0, s, pos[i], q[i], 16)), (listed[i], oracle_select(tw, 0, s, pos[i], q[i], 16, lists[i]))]
            tw.images[0].append(tw.pool.block_table(s), lens[i], new[0, i], new[1, i], capacity_cells=tw.pool.seq_capacity(s))
            for got, want in wants + [(stepped[i], tw.oracle_attend(0, s, lens[i], q[i], 16))]:
                _, rel = check_attn(got, want, "entry %d of %d" % (i, n))
                assert rel <= REF_BAR_MAX_REL, (i, rel)
        tw.assert_pools_equal()


@pytest.mark.parametrize("n", [15, 16, 17, 64])
def test_every_list_of_a_selection(n):
    rng = np.random.Generator(np.random.PCG64(5300 + n))
    pos = [int(c) for c in rng.integers(40, 700, n)]
    pooled = [rng.standard_normal((p // 4 + 1, 128)).astype(np.float32) for p in pos]
    q = rng.standard_normal((n, 4, 128)).astype(np.float32)
    with Pool(n_pages=4, max_seqs=1) as pool:
        listed, ids, counts = gpu_select(pool, pos, q, pooled, 24, 32)
        listed.free()
    for i, p in enumerate(pos):
        want = oracle.topk_blocks(oracle.indexer_score(q[i], pooled[i], p // 4 + 1, p), 24, p // 4)
        assert np.array_equal(ids[i, :counts[i]], want), i
