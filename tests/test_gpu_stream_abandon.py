"""Calls between a stream's batches that replace its buffers (larger reads, another phase 1, a host store): the
stream ends there, and adding to it or ending it reports so instead of running on memory that is gone. Reads that fit
the stream's buffers leave it as it is. Whole numbers: equal."""
import numpy as np
import pytest

import oracle_api as oa
from rapidgkc_amd import native, synth

pytestmark = pytest.mark.gpu
K, PM, PARTS = 31, 11, 32


@pytest.mark.parametrize("use_graph", [True, False])
@pytest.mark.parametrize("what", ["larger reads", "phase 1", "sized", "host store", "smaller reads"])
def test_calls_between_batches(what, use_graph):
    print(f"[gpu] case stream abandoned by {what} graph{use_graph}", flush=True)
    g = synth.genome(97, 60_000, gc=0.45)
    chars, offs = synth.short_reads(g, 98, 1_000, 150, 0.01)
    few = synth.short_reads(g, 99, 50, 150, 0.01)
    many = synth.short_reads(g, 100, 20_000, 150, 0.01)
    st, po, ps, pk = oa.store(chars, offs, K, PM, PARTS)
    c = native.Counter(0)
    for again in range(1 if what == "larger reads" else 2):  # the second time the context's buffers hold them
        c.stream_begin(K, PM, PARTS, 1_000, len(chars), np.diff(po), ps, use_graph)
        c.stream_add(chars[:150 * 400], offs[:401])
        if what == "larger reads":
            c.set_reads(*many)
        elif what == "host store":
            c.count_host_store(st, po, PARTS, K, PM)
        else:
            c.set_reads(*few)
        if what == "phase 1":
            c.superkmers(K, PM, 2 * PARTS)
        elif what == "sized":
            c.superkmers_sized(K, PM, PARTS, np.diff(po) + np.uint64(20_000), ps + np.uint64(1_000))
        rest = (chars[150 * 400:], (offs[400:] - offs[400]).astype(np.uint64))
        if what == "smaller reads":
            c.stream_add(*rest)
            pb, sc, kc = c.stream_end()
            assert np.array_equal(pb, np.diff(po)) and np.array_equal(sc, ps) and np.array_equal(kc, pk)
        else:
            for call in (lambda: c.stream_add(*rest), c.stream_end):
                with pytest.raises(native.RgkcError) as e:
                    call()
                assert e.value.code == -6
    # what took the stream's place is whole
    if what == "larger reads":
        c.superkmers(K, PM, PARTS)
        _, distinct = c.count()
        st2, po2, _, _ = oa.store(*many, K, PM, PARTS)
        assert distinct == len(oa.count_store(st2, po2, K)[0])
    c.close()
