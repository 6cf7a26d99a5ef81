"""Ways through the count stage that depend on the data's units, each shown to be taken by its statistics and with the
oracle's table: key regions that exceed the memory limit (planned again, counted from the records), slices that
overflow their key region (an exact one in a second pass), and a partition of more units than the small grouping
kernel takes. Whole numbers: equal."""
import numpy as np
import pytest

import oracle_api as oa
from rapidgkc_amd import native, synth

pytestmark = pytest.mark.gpu


def _case(name, chars, offs, k, p, parts, cap):
    print(f"[gpu] case {name} k{k} p{p} parts{parts} cap{cap}", flush=True)
    st, opo, _, _ = oa.store(chars, offs, k, p, parts)
    c = native.Counter(0)
    c.set_tuning(cap)
    c.set_reads(chars, offs)
    c.superkmers(k, p, parts)

    def check():
        ok_, oc_, oro = oa.count_store(st, opo, k)
        rows, distinct = c.count(1, 0xFFFFFFFF)
        c.sort_rows()
        keys, cnts, _ = c.table(rows)
        assert np.array_equal(rows, np.diff(oro)) and distinct == len(ok_)
        assert np.array_equal(keys, ok_) and np.array_equal(cnts, oc_)
        return c.stats()
    return c, check


@pytest.mark.parametrize("k,p,cap", [(21, 3, 1024), (55, 4, 1024), (31, 5, 0)])
def test_key_regions_beyond_the_limit(k, p, cap):
    chars, offs = synth.short_reads(synth.genome(81, 60_000, gc=0.45), 82, 6_000, 150, 0.01)
    c, check = _case("key regions beyond the limit", chars, offs, k, p, 1, cap)
    with_keys = check()
    assert with_keys["heavy_groups"] > 0
    c.set_memory_limit(64 << 10)
    without = check()
    assert without["heavy_groups"] == 0 and without["items"] > 0
    c.set_memory_limit(0)
    assert check()["heavy_groups"] == with_keys["heavy_groups"]
    c.close()


@pytest.mark.parametrize("k,p,cap", [(31, 11, 256), (63, 11, 256)])
def test_slices_that_overflow(k, p, cap):
    reads = [b"A" * 150, b"ACGTTGCATT" * 15] * 1_500
    offs = np.arange(len(reads) + 1, dtype=np.uint64) * np.uint64(150)
    c, check = _case("slices that overflow", np.frombuffer(b"".join(reads), dtype=np.uint8).copy(), offs, k, p, 1, cap)
    s = check()
    assert s["heavy_groups"] > 0 and s["ovf_keys"] > 0
    c.close()


@pytest.mark.parametrize("k", [31, 55])
def test_more_units_than_the_small_grouping_kernel_takes(k):
    chars, offs = synth.short_reads(synth.genome(83, 150_000, gc=0.5), 84, 9_000, 150, 0.01)
    c, check = _case("many units", chars, offs, k, 11, 1, 256)
    assert check()["items"] > 1024  # of one partition
    c.close()
