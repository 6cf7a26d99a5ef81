"""The list statistics of batched input: tiles rescanned because their list overflowed and tiles written in list
order, summed over the batches, as phase 1 counts them on each batch alone; and none of them left over for a call
without phase 1. Whole numbers: equal."""
import numpy as np
import pytest

from rapidgkc_amd import native, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_graph", [True, False])
@pytest.mark.parametrize("k,p,lists", [(25, 9, 64), (21, 11, 0), (21, 11, 4500), (25, 9, 0xFFFFFFFF)])
def test_stream_list_stats(k, p, lists, use_graph):
    print(f"[gpu] case stream list stats k{k} lists{lists:#x} graph{use_graph}", flush=True)
    parts = 32
    chars, offs = synth.short_reads(synth.genome(51, 100_000, gc=0.5), 52, 3_000, 148, 0.005)  # k=21: one full segment a read
    bounds = [0, 300, 301, 1500, 1500, 3000]
    batches = [(chars[int(offs[a]):int(offs[b])], (offs[a:b + 1] - offs[a]).astype(np.uint64)) for a, b in zip(bounds[:-1], bounds[1:])]
    c = native.Counter(0)
    c.set_p1_lists(lists)
    rescans = order = 0
    for b in batches:
        c.set_reads(*b)
        c.superkmers(k, p, parts)
        s = c.stats()
        rescans, order = rescans + s["p1_rescans"], order + s["p1_list_order"]
    assert (rescans > 0) == (lists in (64, 4500)) and (order > 0) == (k == 21)
    c.set_reads(chars, offs)
    po, ps, _ = c.superkmers(k, p, parts)
    for _ in range(2):
        c.stream_begin(k, p, parts, 3_000, len(chars), np.diff(po), ps, use_graph)
        for b in batches:
            c.stream_add(*b)
        c.stream_end()
        s = c.stats()
        assert (s["p1_rescans"], s["p1_list_order"]) == (rescans, order)
    st = c.copy_store(int(po[-1]))
    c.count_host_store(st, po, parts, k, p)
    s = c.stats()
    assert (s["p1_rescans"], s["p1_list_order"]) == (0, 0)
    c.close()
