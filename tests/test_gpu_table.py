"""Copying the table out: its rows arrive partition after partition whatever the partitions' sizes and
number (chunks of the dense table that end inside a partition, on a partition's end, and after 1024
partitions), with keys or counts alone, for 64- and 128-bit keys. Whole numbers: equal."""
import numpy as np
import pytest

import oracle_api as oa
from rapidgkc_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,p,parts,reads,empty", [
    (31, 11, 1, 30_000, 0),      # one partition over several chunks
    (31, 11, 1000, 30_000, 0),   # chunk ends inside partitions
    (55, 13, 64, 12_000, 0),     # 128-bit keys, several chunks
    (31, 11, 700, 400, 1700),    # 2400 partitions, most of them empty: more than one gather takes
    (31, 11, 16, 1, 0),          # one read: a few rows, most partitions empty
])
def test_copy_table(k, p, parts, reads, empty):
    from rapidgkc_amd import native
    print(f"[gpu] case copy table k{k} parts{parts}+{empty} reads{reads}", flush=True)
    g = synth.genome(k + parts, 300_000, gc=0.45)
    chars, offs = synth.short_reads(g, 17, reads, 150, 0.01)
    st, opo, _, _ = oa.store(chars, offs, k, p, parts)
    ok_, oc_, oro = oa.count_store(st, opo, k)
    # empty partitions among the others: three runs, at the front, in the middle and at the end
    at = np.sort(np.concatenate([np.arange(parts + 1), np.zeros(empty // 3, int), np.full(empty // 3, parts // 2),
                                 np.full(empty - 2 * (empty // 3), parts)]))
    c = native.Counter(0)
    rows, distinct = c.count_host_store(st, opo[at], parts, k, p)
    assert len(rows) == parts + empty and int(rows.sum()) == distinct == len(ok_)
    c.sort_rows()
    keys, cnts, ro = c.table(rows)
    assert np.array_equal(rows[rows > 0], np.diff(oro)[np.diff(oro) > 0])
    assert np.array_equal(keys, ok_) and np.array_equal(cnts, oc_)
    k2, c2 = np.zeros_like(keys), np.zeros_like(cnts)
    assert native.lib().rgkc_copy_table(c._h, k2.ctypes.data, None) == 0
    assert native.lib().rgkc_copy_table(c._h, None, c2.ctypes.data) == 0
    assert np.array_equal(k2, keys) and np.array_equal(c2, cnts)
    c.close()
