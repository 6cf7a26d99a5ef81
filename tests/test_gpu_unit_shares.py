"""Units far larger than a sweep, counted from their records: a work item covers at most four sweeps'
instances of one, so that a few minimizers do not leave the device to a few workgroups. A minimizer length
with few values, runs of a few k-mers, 128-bit keys, and sweeps that overflow. The table is the oracle's; whole
numbers: equal."""
import numpy as np
import pytest

import oracle_api as oa
from rapidgkc_amd import native, synth

pytestmark = pytest.mark.gpu


def _random():
    return synth.short_reads(synth.genome(41, 60_000, gc=0.45), 42, 4_000, 150, 0.01)


def _low_complexity():
    rng = np.random.default_rng(43)
    reads = [b"A" * 150, b"AC" * 75, b"ACGTTGCATT" * 15] * 900 + [bytes(rng.choice(list(b"ACGT"), 150)) for _ in range(300)]
    offs = np.arange(len(reads) + 1, dtype=np.uint64) * np.uint64(150)
    return np.frombuffer(b"".join(reads), dtype=np.uint8).copy(), offs


@pytest.mark.parametrize("make,k,p,parts,cap", [
    (_random, 21, 3, 1, 256), (_random, 21, 3, 5, 1024), (_random, 31, 3, 1, 16384), (_random, 55, 5, 1, 256),
    (_random, 55, 4, 2, 20_000), (_random, 8, 8, 1, 300), (_low_complexity, 31, 11, 3, 256), (_low_complexity, 63, 11, 1, 6144)])
def test_unit_shares(make, k, p, parts, cap):
    print(f"[gpu] case unit shares {make.__name__} k{k} p{p} parts{parts} cap{cap}", flush=True)
    chars, offs = make()
    st, opo, _, okm = oa.store(chars, offs, k, p, parts)
    ok_, oc_, oro = oa.count_store(st, opo, k)
    c = native.Counter(0)
    c.set_tuning(cap)
    c.set_heavy_expand(1)
    c.set_reads(chars, offs)
    c.superkmers(k, p, parts)
    for _ in range(2):
        rows, distinct = c.count(1, 0xFFFFFFFF)
        c.sort_rows()
        keys, cnts, _ = c.table(rows)
        assert np.array_equal(rows, np.diff(oro)) and distinct == len(ok_)
        assert np.array_equal(keys, ok_) and np.array_equal(cnts, oc_)
        assert c.stats()["heavy_groups"] == 0 and c.stats()["items"] * 4 * cap >= int(okm.sum())
    c.close()
