"""Batched input through the superkmer lists: batches far smaller than the capacity the grid covers, empty
ones and ones without a whole k-mer, lists that overflow (tiles rescanned) and no lists, with and without
the captured graph; the store and table are the oracle's. Whole numbers: equal."""
import numpy as np
import pytest

import oracle_api as oa
from rapidgkc_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_graph", [True, False])
@pytest.mark.parametrize("k,p,parts,lists", [(25, 9, 64, 0), (25, 9, 64, 64), (25, 9, 64, 0xFFFFFFFF), (55, 13, 600, 0),
                                             (55, 13, 600, 64)])
def test_stream_lists(k, p, parts, lists, use_graph):
    from rapidgkc_amd import native
    print(f"[gpu] case stream lists k{k} parts{parts} lists{lists:#x} graph{use_graph}", flush=True)
    g = synth.genome(21, 120_000, gc=0.5, tandem_frac=0.05)
    short = synth.short_reads(g, 22, 4000, 150, 0.005)
    lr = synth.long_reads(g, 23, 30, mean=5000, sd=3000, err=0.05, max_len=20000)
    chars, offs = synth.interleave_csr(short, lr, 24)
    st, po, ps, pk = oa.store(chars, offs, k, p, parts)
    n = len(offs) - 1
    bounds = [0, 1, 1, 3, 40, 41, 900, 1700, 1700, n - 2, n]
    c = native.Counter(0)
    c.set_p1_lists(lists)
    for again in range(2):
        c.stream_begin(k, p, parts, n + 1000, len(chars) + 300_000, np.diff(po), ps, use_graph)
        for a, b in zip(bounds[:-1], bounds[1:]):
            c.stream_add(chars[int(offs[a]):int(offs[b])], (offs[a:b + 1] - offs[a]).astype(np.uint64))
        c.stream_add(np.frombuffer(b"ACGT" * 2, dtype=np.uint8).copy(), np.array([0, 3, 8], dtype=np.uint64))
        pb, sc, kc = c.stream_end()
        assert np.array_equal(pb, np.diff(po)) and np.array_equal(sc, ps) and np.array_equal(kc, pk)
        rows, _ = c.count(1, 0xFFFFFFFF)
        c.sort_rows()
        keys, cnts, _ = c.table(rows)
        ok_, oc_, oro = oa.count_store(st, po, k)
        assert np.array_equal(rows, np.diff(oro)) and np.array_equal(keys, ok_) and np.array_equal(cnts, oc_)
    c.close()
