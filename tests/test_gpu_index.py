"""Counting stores that arrive as bytes: record boundaries and minimizers found piece by piece (8 KiB) by
the device. Records across piece ends, records longer than several pieces, partitions that end at and
around a piece's and a thread's bytes, stores without p or the partition count, and a store cut in the
middle of a record. Whole numbers: equal."""
import numpy as np
import pytest

import oracle_api as oa
from rapidgkc_amd import synth

pytestmark = pytest.mark.gpu


def _reads(kind):
    rng = np.random.default_rng(11)
    if kind == "long":  # one superkmer each: up to 45 000 bases, 15 000 bytes
        reads = [(bytes(rng.choice(list(b"ACGT"), u)) * (n // u + 1))[:n] for n in (900, 20_000, 45_000) for u in (2, 3, 7)]
        reads += [bytes(rng.choice(list(b"ACGT"), 300)) for _ in range(200)]
        offs = np.zeros(len(reads) + 1, dtype=np.uint64)
        np.cumsum([len(r) for r in reads], out=offs[1:])
        return np.frombuffer(b"".join(reads), dtype=np.uint8).copy(), offs
    g = synth.genome(12, 100_000, gc=0.45)
    return synth.short_reads(g, 13, 4_000, 150, 0.01)


@pytest.mark.parametrize("kind,k,p,parts,known", [
    ("long", 31, 11, 3, True), ("long", 55, 13, 1, True), ("short", 31, 11, 1, True), ("short", 63, 15, 7, True),
    ("short", 16, 5, 2, True), ("short", 31, 11, 5, False)])
def test_index(kind, k, p, parts, known):
    from rapidgkc_amd import native
    print(f"[gpu] case index {kind} k{k} parts{parts} known{known}", flush=True)
    chars, offs = _reads(kind)
    st, po, ps, pk = oa.store(chars, offs, k, p, parts)
    ok_, oc_, oro = oa.count_store(st, po, k)
    c = native.Counter(0)
    rows, distinct = c.count_host_store(st, po, parts if known else 0, k, p if known else 0)
    s = c.stats()
    assert s["n_records"] == int(ps.sum()) and s["n_kmers"] == int(pk.sum())
    c.sort_rows()
    keys, cnts, _ = c.table(rows)
    assert np.array_equal(rows, np.diff(oro)) and distinct == len(ok_)
    assert np.array_equal(keys, ok_) and np.array_equal(cnts, oc_)
    c.close()


def test_index_piece_ends():
    """A partition's leading records whose bytes end just before, on and after multiples of a thread's 32
    bytes and a piece's 8192."""
    from rapidgkc_amd import native
    print("[gpu] case index piece ends", flush=True)
    k, p = 31, 11
    chars, offs = _reads("short")
    st, po, _, _ = oa.store(chars, offs, k, p, 1)
    full = st >= 0xC0
    ends = np.flatnonzero(~full[1:] & full[:-1]) + 2  # bytes up to each record's end
    c = native.Counter(0)
    for at in (32, 64, 8192, 16384, 24576):
        i = int(np.searchsorted(ends, at))
        for e in ends[max(0, i - 1):i + 2]:
            e = int(e)
            rows, _ = c.count_host_store(st[:e], np.array([0, e], dtype=np.uint64), 1, k, p)
            assert c.stats()["n_records"] == int(np.count_nonzero(ends <= e))
            assert int(rows[0]) == oa.count_partition(st[:e], k)[2]
        cut = int(ends[i]) - 1  # the last record's last byte is missing
        with pytest.raises(native.RgkcError):
            c.count_host_store(st[:cut], np.array([0, cut], dtype=np.uint64), 1, k, p)
    c.close()
