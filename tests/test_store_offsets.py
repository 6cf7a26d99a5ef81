"""Partition offsets that decrease: the store's length is the last offset, so a partition before it would be
read past the bytes that are there. Both entry points that take a store refuse them; equal offsets (empty
partitions) are accepted."""
import numpy as np
import pytest

import oracle_api as oa
from rapidgkc_amd import native, synth


def _store(parts):
    chars, offs = synth.short_reads(synth.genome(31, 40_000, gc=0.45), 32, 2_000, 150, 0.01)
    return oa.store(chars, offs, 31, 11, parts)[:2]


def _bad(po):
    """The last partition ends before it starts: by less and by more than a piece of the index kernels."""
    for back in (100, 20_000):
        b = po.copy()
        b[-1] = b[-2] - np.uint64(back)
        yield b


def test_minimizer_length_refuses_decreasing_offsets():
    st, po = _store(3)
    assert native.store_minimizer_length(st, np.sort(np.append(po, po)), 31) == 11
    for bad in _bad(po):
        with pytest.raises(native.RgkcError) as e:
            native.store_minimizer_length(st, bad, 31)
        assert e.value.code == -2


@pytest.mark.gpu
@pytest.mark.parametrize("p", [11, 0])
def test_count_refuses_decreasing_offsets(p):
    st, po = _store(3)
    c = native.Counter(0)
    want = c.count_host_store(st, po, 3, 31, 11)[1]
    for bad in _bad(po):
        print(f"[gpu] case store offsets p{p} {bad}", flush=True)
        with pytest.raises(native.RgkcError) as e:
            c.count_host_store(st, bad, 3, 31, p)
        assert e.value.code == -2
    assert c.count_host_store(st, np.sort(np.append(po, po)), 3, 31, p)[1] == want
    c.close()
