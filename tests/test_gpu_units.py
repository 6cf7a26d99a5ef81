"""The count stage's units of work against the oracle, where its kernels change path: records longer
than a chunk's piece map, its staged words or the grouping's word map (tandem repeats are one superkmer);
partitions of more units than the small grouping kernel takes; equal records; runs of one k-mer; a
read of exactly one k-mer; 128-bit keys that differ in one half. Both with the largest units expanded into
keys and without. Whole numbers: equal."""
import numpy as np
import pytest

import oracle_api as oa
from rapidgkc_amd import synth

pytestmark = pytest.mark.gpu


def _csr(reads):
    offs = np.zeros(len(reads) + 1, dtype=np.uint64)
    np.cumsum([len(r) for r in reads], out=offs[1:])
    return np.frombuffer(b"".join(reads), dtype=np.uint8).copy(), offs


def _tandem(rng, unit, length):
    u = bytes(rng.choice(list(b"ACGT"), unit))
    return (u * (length // unit + 1))[:length]


def _long_records():
    rng = np.random.default_rng(3)
    reads = [_tandem(rng, int(u), n) for n in (600, 700, 3_000, 45_000, 70_000, 120_000) for u in (2, 3, 5, 7, 9)]
    reads += [bytes(rng.choice(list(b"ACGT"), int(rng.integers(40, 400)))) for _ in range(400)]
    return _csr([reads[i] for i in rng.permutation(len(reads))])


def _equal_records():
    rng = np.random.default_rng(4)
    few = [bytes(rng.choice(list(b"ACGT"), 150)) for _ in range(7)]
    comp = bytes.maketrans(b"ACGT", b"TGCA")
    reads = [few[i % 7] if i % 2 else few[i % 7].translate(comp)[::-1] for i in range(6_000)]
    reads += [b"A" * 200] * 300 + [b"T" * 400] * 50 + [b"AC" * 100] * 200 + [b"ACGTTGCA" * 8] * 40
    return _csr(reads)


def _many_units():
    g = synth.genome(8, 150_000, gc=0.5)
    return synth.short_reads(g, 9, 9_000, 150, 0.01)


def _same_halves(k):
    """k-mers that end in the same 32 bases, 16 of each: many meet in one group of the 128-bit table."""
    def make():
        rng = np.random.default_rng(k)
        reads = []
        for _ in range(900):
            tail = bytes(rng.choice(list(b"ACGT"), 32))
            for v in range(16):
                head = bytes(rng.choice(list(b"ACGT"), k - 34)) if k > 34 else b""
                reads += [(head + bytes([b"ACGT"[v % 4], b"ACGT"[v // 4]]))[-(k - 32):] + tail] * (1 + v % 3)
        return _csr([reads[i] for i in rng.permutation(len(reads))])
    return make


def _one_kmer_records(n, k):
    """n records of one k-mer: a chunk of the unit to its last record, one less and one more."""
    def make():
        rng = np.random.default_rng(n)
        return _csr([bytes(rng.choice(list(b"ACGT"), k)) for _ in range(n - 3)] + [b"ACGTTGCA" * 8 + b"A" * k] * 3)
    return make


@pytest.mark.parametrize("make,k,p,parts,cap", [
    *[(_one_kmer_records(n, 31), 31, 9, 1, 0) for n in (2047, 2048, 2049, 4097)],
    *[(_one_kmer_records(n, 63), 63, 9, 1, 0) for n in (1023, 1024, 1025)],
    (_same_halves(33), 33, 5, 1, 30_000),
    (_same_halves(34), 34, 5, 1, 30_000),
    (_same_halves(63), 63, 5, 2, 0),
    (_long_records, 31, 11, 3, 0),
    (_long_records, 55, 13, 3, 0),
    (_long_records, 21, 7, 1, 700),
    (_equal_records, 31, 11, 2, 0),
    (_equal_records, 63, 11, 1, 300),
    (_many_units, 31, 11, 1, 256),   # about 2000 units in one partition, 128-bit keys below
    (_many_units, 55, 11, 1, 256),
    (lambda: _csr([b"ACGTTGCATTGACCATGGACTAGGACTCATG"]), 31, 11, 64, 0),
], ids=[*[f"chunk31_{n}" for n in (2047, 2048, 2049, 4097)], *[f"chunk63_{n}" for n in (1023, 1024, 1025)], "halves33", "halves34", "halves63", "long31", "long55", "long21", "equal31", "equal63", "many31", "many55", "one"])
def test_units(make, k, p, parts, cap):
    from rapidgkc_amd import native
    chars, offs = make()
    st, opo, _, _ = oa.store(chars, offs, k, p, parts)
    ok_, oc_, oro = oa.count_store(st, opo, k)
    c = native.Counter(0)
    c.set_tuning(cap)
    c.set_reads(chars, offs)
    c.superkmers(k, p, parts)
    for mode in (0, 1):
        print(f"[gpu] case units k{k} parts{parts} cap{cap} mode{mode}", flush=True)
        c.set_heavy_expand(mode)
        rows, distinct = c.count(1, 0xFFFFFFFF)
        c.sort_rows()
        keys, cnts, _ = c.table(rows)
        assert np.array_equal(rows, np.diff(oro)) and distinct == len(ok_)
        assert np.array_equal(keys, ok_) and np.array_equal(cnts, oc_)
        rows2, distinct2 = c.count(2, 100)
        assert distinct2 == distinct and int(rows2.sum()) == int(((oc_ >= 2) & (oc_ <= 100)).sum())
    c.close()
