"""The per-layer calls past ctypes (breccia_amd._hot): what they take, what they leave to ctypes, and that both ways
come to the same."""
import ctypes as C
import os
import shutil
import subprocess
import sys

import numpy as np
import pytest

from breccia_amd import build
from breccia_amd import lib as L
from breccia_amd.kv import BkvError, Pool, _hot

SEQS, POS, ONE = np.zeros(1, np.int32), np.zeros(1, np.int64), np.ones(1, np.int32)
ADDR = 0x1000  # never touched: a host-only pool is refused before any launch
CALLS = {
    "append": ("append", lambda s, p, n: (0, s, p, n, ADDR, ADDR), lambda a: a + (None, False)),
    "append_kprep": ("append_kprep", lambda s, p, n: (0, s, p, n, ADDR, ADDR, ADDR, 1e-6, ADDR, 64, 16), lambda a: a + (None, None)),
    "decode_attn": ("decode_attn", lambda s, p, n: (0, s, p, 16, ADDR, ADDR, 0.5), lambda a: a + (None, 0, 0, None)),
    "decode_step": ("decode_step", lambda s, p, n: (0, s, p, ADDR, ADDR, 16, ADDR, ADDR, 0.5), lambda a: a + (None, 0, 0, None)),
    "decode_attn_select": ("decode_attn_select", lambda s, p, n: (0, s, p, 16, ADDR, ADDR, 0.5, ADDR, 4, ADDR, 4),
                           lambda a: a + (None, 0, 0, None)),
    "prefill_attn": ("prefill_attn", lambda s, p, n: (0, s, p, n, 16, ADDR, ADDR, 0.5), lambda a: a + (None, 0, 0, None)),
    "select_blocks": ("select_blocks", lambda s, p, n: (p, ADDR, [ADDR], n, 4, 128, 16, ADDR, 32, ADDR, 32), lambda a: a + (None,)),
}


@pytest.fixture()
def pool(monkeypatch):
    # a failed call into the bench library that nobody passed to check() would lend the next error its message
    monkeypatch.setattr(L, "_bench_error", None)
    with Pool(n_pages=8, max_seqs=2, host_only=True) as p:
        assert p.seq_create() == 0
        p.seq_reserve(0, 17)
        yield p


def _error(call):
    with pytest.raises(BkvError) as e:
        call()
    return e.value.status, e.value.message


@pytest.mark.parametrize("name", sorted(CALLS))
@pytest.mark.parametrize("pos", [0, -1])
def test_both_ways_come_to_the_same_refusal(pool, name, pos):
    method, args, full = CALLS[name]
    at = np.array([pos], np.int64)
    plain = args(SEQS, at, ONE)
    assert getattr(_hot, name)(pool.handle, *full(plain)) in range(1, 9)     # taken: no argument was left over
    fast = _error(lambda: getattr(pool, method)(*plain))
    general = _error(lambda: getattr(pool, method)(*args(SEQS.tolist(), at.tolist(), ONE.tolist())))
    assert fast == general
    assert fast[0] == (L.ERR_NO_DEVICE if pos == 0 else L.ERR_RANGE)


def test_indexer_pooling(pool):
    plain = (ADDR, 4, ADDR, ADDR, 0, 1, ADDR, 1e-6, ADDR, 64, 16)
    assert _hot.idx_pool(pool.handle, *plain, 128, None) == L.ERR_NO_DEVICE
    assert _error(lambda: pool.idx_pool(*plain)) == _error(lambda: pool.idx_pool(ADDR, np.int32(4), *plain[2:]))


def _strided():
    return np.zeros(4, np.int32)[::2]


@pytest.mark.parametrize("seqs,pos,layer,q,scale", [
    ([0], POS, 0, ADDR, 0.5), ((0,), POS, 0, ADDR, 0.5), (SEQS.astype(np.int64), POS, 0, ADDR, 0.5),
    (SEQS, POS.astype(np.int32), 0, ADDR, 0.5), (_strided(), np.zeros(2, np.int64), 0, ADDR, 0.5), (SEQS.astype(">i4"), POS, 0, ADDR, 0.5),
    (SEQS.view(np.uint32), POS, 0, ADDR, 0.5), (np.zeros(2, np.int32), POS, 0, ADDR, 0.5),
    (SEQS, POS, np.int32(0), ADDR, 0.5), (SEQS, POS, False, ADDR, 0.5), (SEQS, POS, 1 << 40, ADDR, 0.5), (SEQS, POS, 0, -1, 0.5),
    (SEQS, POS, 0, 1 << 70, 0.5), (SEQS, POS, 0, C.c_uint64(ADDR), 0.5), (SEQS, POS, 0, ADDR, 1), (SEQS, POS, 0, ADDR, np.float32(0.5))])
def test_what_is_not_plain_is_left_to_ctypes(pool, seqs, pos, layer, q, scale):
    assert _hot.decode_attn(pool.handle, layer, seqs, pos, 16, q, ADDR, scale, None, 0, 0, None) is NotImplemented


@pytest.mark.parametrize("q", [ADDR, C.c_void_p(ADDR), None])
@pytest.mark.parametrize("seqs", [SEQS, SEQS[:0], SEQS.reshape(1, 1)])
def test_what_is_plain(pool, q, seqs):
    frozen = seqs.copy()
    frozen.setflags(write=False)
    for s in (seqs, frozen):
        got = _hot.decode_attn(pool.handle, 0, s, POS[:s.size], 16, q, ADDR, 0.5, None, 0, 0, None)
        assert got == L.lib.bkv_decode_attn(pool.handle, 0, s.size, s.ctypes.data_as(C.POINTER(C.c_int32)),
                                            POS.ctypes.data_as(C.POINTER(C.c_int64)), 16, q, None, 0, 0, 0.5, ADDR, None)


def test_sizes_that_disagree_and_a_destroyed_pool(pool):
    with pytest.raises(AssertionError):
        pool.decode_attn(0, SEQS, np.zeros(2, np.int64), 16, ADDR, ADDR, 0.5)
    gone = Pool(n_pages=2, host_only=True)
    gone.destroy()
    assert _error(lambda: gone.decode_attn(0, SEQS, POS, 16, ADDR, ADDR, 0.5))[0] == L.ERR_INVALID
    assert _error(lambda: gone.seq_reserve(0, 1))[0] == L.ERR_INVALID


@pytest.mark.parametrize("capacity", [1, 4, 64, 65])
def test_reserve_reports_its_copies(capacity):
    """A fork that writes into the shared, partly filled page: one pair, the same on both ways (65: ctypes)."""
    with Pool(n_pages=8, max_seqs=2, host_only=True) as p:
        a = p.seq_create()
        assert p.seq_reserve(a, 20, capacity) == []
        b = p.seq_fork(a, 20)
        shared = int(p.block_table(a)[1])
        assert p.seq_reserve(b, 21, capacity) == [(shared, int(p.block_table(b)[1]))]
        assert _error(lambda: p.seq_reserve(b, 5, capacity))[0] == L.ERR_RANGE
        assert _hot.seq_reserve(p.handle, b, 21, 0) is NotImplemented


def test_pages_that_are_out_are_counted():
    """Attention over a page that is out is refused, below it not, and the allocator's check compares the count."""
    def attend(p, cell):
        return _error(lambda: p.decode_attn(0, SEQS, POS + cell, 16, ADDR, ADDR, 0.5))[0]  # NO_DEVICE: passed everything else

    host = C.c_void_p(ADDR)
    with Pool(n_pages=8, max_seqs=2, host_only=True) as p:
        s = p.seq_create()
        p.seq_reserve(s, 70)
        assert attend(p, 69) == L.ERR_NO_DEVICE
        for first, n in ((1, 2), (3, 1)):
            assert L.lib.bkv_seq_evict(p.handle, s, first, n, host, None) == L.OK
            p.check()
        assert (attend(p, 15), attend(p, 16), attend(p, 69)) == (L.ERR_NO_DEVICE, L.ERR_STATE, L.ERR_STATE)
        assert L.lib.bkv_seq_restore(p.handle, s, 2, 2, host, None) == L.OK
        p.check()
        assert (attend(p, 15), attend(p, 69)) == (L.ERR_NO_DEVICE, L.ERR_STATE)
        assert L.lib.bkv_seq_restore(p.handle, s, 1, 1, host, None) == L.OK
        p.check()
        assert attend(p, 69) == L.ERR_NO_DEVICE
        assert L.lib.bkv_seq_evict(p.handle, s, 0, 1, host, None) == L.OK
        p.seq_free(s)
        assert p.seq_create() == s      # a new sequence in the slot begins with none out
        p.seq_reserve(s, 20)
        p.check()
        assert attend(p, 19) == L.ERR_NO_DEVICE


def test_the_library_that_is_called_is_the_one_that_was_loaded(tmp_path):
    """Another copy of the library on LD_LIBRARY_PATH: pools are made and read by one of them."""
    shutil.copy(L.LIB_PATH, tmp_path)
    script = """
import numpy as np
from breccia_amd.kv import BkvError, Pool, _hot
with Pool(n_pages=4, host_only=True) as p:
    said = []
    for seqs in (np.ones(1, np.int32), [1]):
        try:
            p.decode_attn(0, seqs, np.zeros(1, np.int64), 16, 0x1000, 0x1000, 0.5)
        except BkvError as e:
            said.append((e.status, e.message))
assert len(said) == 2 and said[0] == said[1] and said[0][1], said
maps = {line.split()[-1] for line in open("/proc/self/maps") if line.rstrip().endswith("libbreccia_kv.so")}
assert len(maps) == 1, maps
"""
    env = dict(os.environ, LD_LIBRARY_PATH=str(tmp_path))
    subprocess.run([sys.executable, "-c", script], check=True, env=env, cwd=os.path.dirname(os.path.dirname(L.LIB_PATH)), timeout=100)


def test_not_bound_yet_means_not_taken():
    """In a fresh interpreter, before kv.py has handed over the classes and the entry points."""
    script = """
import importlib.util
spec = importlib.util.spec_from_file_location("_hot", %r)
hot = importlib.util.module_from_spec(spec)
spec.loader.exec_module(hot)
assert hot.seq_reserve(0, 0, 1, 4) is NotImplemented
for wrong in [(), (int, int, int), (int, int, int, {}), (int, int, int, {"bkv_append": 0}), (int, int, int, {"bkv_append": "x"})]:
    try:
        hot.bind(*wrong)
    except (TypeError, ValueError):
        pass
    else:
        raise AssertionError(wrong)
assert hot.seq_reserve(0, 0, 1, 4) is NotImplemented
""" % _hot.__file__
    subprocess.run([sys.executable, "-c", script], check=True, timeout=100)


def test_without_the_module_calls_go_through_ctypes():
    script = """
import sys, warnings
sys.modules["breccia_amd._hot"] = None  # as if it were not built
import numpy as np
with warnings.catch_warnings(record=True) as said:
    warnings.simplefilter("always")
    from breccia_amd.kv import BkvError, Pool
assert any("ctypes" in str(w.message) for w in said)
with Pool(n_pages=4, host_only=True) as p:
    s = p.seq_create()
    assert p.seq_reserve(s, 17) == []
    one, at = np.ones(1, np.int32), np.zeros(1, np.int64)
    calls = [lambda: p.append(0, [s], at, one, 64, 64), lambda: p.append_kprep(0, [s], at, one, 64, 64, 64, 1e-6, 64, 64, 16),
             lambda: p.decode_attn(0, [s], at, 16, 64, 64, 0.5), lambda: p.decode_step(0, [s], at, 64, 64, 16, 64, 64, 0.5),
             lambda: p.decode_attn_select(0, [s], at, 16, 64, 64, 0.5, 64, 4, 64, 4), lambda: p.prefill_attn(0, [s], at, one, 16, 64, 64, 0.5),
             lambda: p.select_blocks(at, 64, [64], one, 4, 128, 16, 64, 32, 64, 32), lambda: p.idx_pool(64, 4, 64, 64, 0, 1, 64, 1e-6, 64, 64, 16)]
    for call in calls:
        try:
            call()
        except BkvError as e:
            assert e.status == %d, e
        else:
            raise AssertionError("not refused")
""" % L.ERR_NO_DEVICE
    subprocess.run([sys.executable, "-c", script], check=True, cwd=os.path.dirname(os.path.dirname(L.LIB_PATH)), timeout=100)


def test_a_build_without_headers_goes_on_without_the_module(monkeypatch, tmp_path, capsys):
    stale = tmp_path / "_hot.so"
    stale.write_bytes(b"of other sources")
    monkeypatch.setattr(build, "HOT_MODULE", str(stale))
    monkeypatch.setattr(build.sysconfig, "get_paths", lambda: {"include": str(tmp_path / "none")})
    assert build.build_hot_calls() is None and not stale.exists()
    assert "ctypes" in capsys.readouterr().err
