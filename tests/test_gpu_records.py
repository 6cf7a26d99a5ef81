"""Records of the list emit, written four bytes at a time from entries in store order: reads that end 0, 1
or 2 bases past a byte, first bytes at each of a read's three phases, records of each length modulo four,
short reads (a tile's words all staged) and long ones (only some of them), 1 partition and both table sizes,
tiles of 256 and of 128 segments, and windows so short that a tile has more records than it can put in
order. Bytes: equal to the oracle's."""
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
