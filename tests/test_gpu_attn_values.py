"""Values that decode attention meets seldom, in ranges of one page a wave as in longer walks."""
import numpy as np
import pytest

from breccia_amd import lib as L
from gpu_common import REF_BAR_MAX_REL, Twin, check_attn
from test_gpu_attn_select import oracle_select, select_attn

pytestmark = pytest.mark.gpu

LAYOUTS = [L.LAYOUT_F16, L.LAYOUT_Q8V, L.LAYOUT_I8H]


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("below", [14, 20])
@pytest.mark.parametrize("cells", [64, 150])
def test_a_quiet_page_keeps_its_bits(layout, below, cells):
    """Cells 32..47 have weights `below` powers of two under the others' and V 10000 times theirs.  A weight is carried as two
    f16 numbers relative to its own page's largest: off by 2^-22 of itself or 2^-25 of that, at most 16 x 5 x 10^4 x 2^-(25 +
    below) of the output.  Relative to the largest weight of four pages it would be 2^-25 of that one: 2e-2 of the output
    at worst, 1e-4 with these values."""
    rng = np.random.Generator(np.random.PCG64(6100 + 10 * layout + below + cells))
    k, v = rng.standard_normal((2, cells, 2, 256)).astype(np.float32)
    q = rng.standard_normal((1, 16, 256)).astype(np.float32)
    k *= 0.3
    q[..., 0], k[..., 0] = 16.0, 0.0  # times the scale of 1/16: a logit of k's first element
    k[32:48, :, 0] = -below * np.log(2.0)
    v[32:48] *= 1e4
    with Twin(n_pages=16, max_seqs=1, layout=layout) as tw:
        s = tw.pool.seq_create()
        tw.pool.seq_reserve(s, cells)
        tw.append(0, [s], [0], [k], [v])
        blocks = list(range((cells + 3) // 4))
        for what, got, want in [
                ("dense", tw.decode_attn(0, [s], [cells - 1], q, 16, scale=1.0 / 16.0), tw.oracle_attend(0, s, cells - 1, q[0], 16)),
                ("list", select_attn(tw, 0, [s], [cells - 1], q, 16, [blocks]), oracle_select(tw, 0, s, cells - 1, q[0], 16, blocks))]:
            _, rel = check_attn(got[0], want, what)
            assert rel <= REF_BAR_MAX_REL, (what, rel)


@pytest.mark.parametrize("layout", [L.LAYOUT_F16, L.LAYOUT_Q8V])
@pytest.mark.parametrize("cells,at", [(65, 64), (65, 10), (64, 63), (1, 0), (300, 256), (300, 40)])
def test_a_score_that_is_not_a_number(layout, cells, at):
    """A key of infinities (what the cache makes of NaN) has scores of NaN.  A head with one among them has no sum, and its
    output is zeros, whether that cell shares its range with others or is alone in it."""
    rng = np.random.Generator(np.random.PCG64(6200 + 10 * layout + cells + at))
    k, v = rng.standard_normal((2, cells, 2, 256)).astype(np.float32)
    k[at, 1] = np.nan
    q = rng.standard_normal((1, 16, 256)).astype(np.float32)
    with Twin(n_pages=24, max_seqs=1, layout=layout) as tw:
        s = tw.pool.seq_create()
        tw.pool.seq_reserve(s, cells)
        tw.append(0, [s], [0], [k], [v])
        got = tw.decode_attn(0, [s], [cells - 1], q, 16, scale=1.0 / 16.0)[0]
        want = tw.oracle_attend(0, s, cells - 1, q[0], 16)
        check_attn(got[:8], want[:8], "the other kv head")
        assert not got[8:].any()


@pytest.mark.parametrize("cells", [2, 40, 64, 130, 1100])
def test_infinite_v(cells):
    """An output over one infinite V value is that infinity, in its own column only and however many ranges are merged.  The
    cell's weight is exp(-1/2) of its page's largest, whose f16 parts are both positive (0.60645 + 0.00009)."""
    rng = np.random.Generator(np.random.PCG64(6300 + cells))
    k, v = np.zeros((cells, 2, 256), np.float32), rng.standard_normal((cells, 2, 256)).astype(np.float32)
    at = cells - 1
    k[at, :, 0] = -0.5
    v[at, 0, 17], v[at, 1, 200] = np.inf, -np.inf
    q = np.zeros((1, 16, 256), np.float32)
    q[..., 0] = 16.0
    with Twin(n_pages=80, max_seqs=1) as tw:
        s = tw.pool.seq_create()
        tw.pool.seq_reserve(s, cells)
        tw.append(0, [s], [0], [k], [v])
        got = tw.decode_attn(0, [s], [cells - 1], q, 16, scale=1.0 / 16.0)[0]
        want = tw.oracle_attend(0, s, cells - 1, q[0], 16)
        assert np.all(got[:8, 17] == np.inf) and np.all(got[8:, 200] == -np.inf)
        got[:8, 17], got[8:, 200], want[:8, 17], want[8:, 200] = 0.0, 0.0, 0.0, 0.0
        check_attn(got, want, "the other columns")
