"""Records of the list emit, written four bytes at a time from entries in store order: reads that end 0, 1
or 2 bases past a byte, first bytes at each of a read's three phases, records of each length modulo four,
short reads (a tile's words all staged) and long ones (only some of them), 1 partition and both table sizes,
tiles of 256 and of 128 segments, and windows so short that a tile has more records than it can put in
order; and the minimizers that cut them. Bytes: equal to the oracle's."""
import numpy as np
import pytest

from test_gpu_parity import check_store

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,p,parts", [(25, 9, 1), (25, 9, 512), (25, 9, 513), (26, 9, 31), (27, 9, 31), (9, 7, 64),
                                       (12, 11, 31), (55, 13, 512), (55, 13, 1000), (57, 13, 31)])
@pytest.mark.parametrize("long", [False, True])
def test_list_records(k, p, parts, long):
    from rapidgkc_amd import native
    print(f"[gpu] case list records k{k} p{p} parts{parts} long{long}", flush=True)
    rng = np.random.default_rng(100 * k + parts)
    lens = np.concatenate([np.arange(k, k + 40), rng.integers(k, 200, 2000)])
    if long:
        lens = np.concatenate([lens, rng.integers(5000, 30000, 12), [k, k + 1, k + 2]])
    offs = np.zeros(len(lens) + 1, dtype=np.uint64)
    np.cumsum(lens, out=offs[1:])
    chars = rng.choice(np.frombuffer(b"ACGT", dtype=np.uint8), int(offs[-1]))
    c = native.Counter(0)
    c.set_reads(chars, offs)
    for _ in range(2):
        check_store(c, chars, offs, k, p, parts)
    c.close()


@pytest.mark.parametrize("k,p", [(8, 8), (8, 3), (16, 16), (17, 16), (31, 16), (32, 16), (33, 16), (31, 15), (31, 14), (22, 7),
                                 (24, 9), (25, 9), (39, 8), (40, 9), (42, 11), (63, 16), (63, 4), (63, 3)])
def test_minimizers(k, p):
    """p-mers cut out of the packed words: every phase of a window to the 16-base words (w = k - p + 1 from 1 to
    61, blocks of 8, 4 and 1 suffix minima), p = 16 (one word back), reads that start anywhere in a word,
    and reads of which the filter drops all p-mers, those of one strand, or many."""
    from rapidgkc_amd import native
    print(f"[gpu] case minimizers k{k} p{p}", flush=True)
    rng = np.random.default_rng(1000 * k + p)
    reads = [rng.choice(np.frombuffer(b"ACGT", dtype=np.uint8), int(n)) for n in rng.integers(k, 330, 1500)]
    reads += [rng.choice(np.frombuffer(alpha, dtype=np.uint8), int(n)) for alpha in (b"A", b"T", b"AC", b"GT", b"AT", b"AAAAAAAC",
              b"TTTTTTTG", b"CG") for n in (k, k + 1, k + 17, 200, 500)]
    offs = np.zeros(len(reads) + 1, dtype=np.uint64)
    np.cumsum([len(r) for r in reads], out=offs[1:])
    chars = np.concatenate(reads)
    c = native.Counter(0)
    c.set_reads(chars, offs)
    check_store(c, chars, offs, k, p, 31)
    c.close()
