"""Host stores whose bytes never end a record: reported as malformed, and in the time of a long record, not of the whole
run of bytes. The longest record that a count takes is one k-mer short of 2^18."""
import time

import numpy as np
import pytest

from rapidgkc_amd import native, synth

pytestmark = pytest.mark.gpu


def _record(bases):
    n = (len(bases) + 3) // 3
    b = np.zeros(3 * n, dtype=np.uint8)
    b[:len(bases)] = bases
    b = b.reshape(n, 3)
    out = 0xC0 | (b[:, 0] << 4) | (b[:, 1] << 2) | b[:, 2]
    out[-1] = (out[-1] & 0x3F) | ((len(bases) % 3) << 6)
    return out.astype(np.uint8)


@pytest.mark.parametrize("k,p", [(31, 11), (63, 13)])
def test_the_longest_record(k, p):
    unit = np.array([0, 1, 2, 3, 3, 2, 1, 0, 3, 3], dtype=np.uint8)
    c = native.Counter(0)
    for kmers, code in ((0x3FFFF, None), (0x40000, -5)):
        print(f"[gpu] case longest record k{k} {kmers} k-mers", flush=True)
        st = _record(np.tile(unit, kmers // 10 + 20)[:kmers + k - 1])
        po = np.array([0, len(st)], dtype=np.uint64)
        if code:
            with pytest.raises(native.RgkcError) as e:
                c.count_host_store(st, po, 1, k, p)
            assert e.value.code == code
        else:
            rows, distinct = c.count_host_store(st, po, 1, k, p)
            _, cnts, _ = c.table(rows)
            assert distinct == 10 and int(cnts.sum()) == kmers
    c.close()


def test_bytes_without_an_end():
    chars, offs = synth.short_reads(synth.genome(95, 50_000, gc=0.45), 96, 2_000, 150, 0.01)
    c = native.Counter(0)
    c.set_reads(chars, offs)
    po, _, _ = c.superkmers(31, 11, 1)
    good = c.copy_store(int(po[-1]))
    want = c.count_host_store(good, po, 1, 31, 11)[1]
    for run in (1, 100_000, 60_000_000):
        st = np.concatenate([good, np.full(run, 0xFF, dtype=np.uint8)])
        print(f"[gpu] case {run} bytes without an end", flush=True)
        t = time.perf_counter()
        with pytest.raises(native.RgkcError) as e:
            c.count_host_store(st, np.array([0, len(st)], dtype=np.uint64), 1, 31, 11)
        assert e.value.code == -5 and time.perf_counter() - t < 0.5
    assert c.count_host_store(good, po, 1, 31, 11)[1] == want
    c.close()
