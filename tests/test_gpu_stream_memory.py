"""What a stream keeps: no histograms on the device when its superkmer lists do not fit half the free memory (the
emit pass scans then), and its records either way."""
import numpy as np
import pytest
import torch

from rapidgkc_amd import native, synth

pytestmark = pytest.mark.gpu


def test_lists_that_do_not_fit_cost_nothing():
    parts, k, p, lists = 32, 31, 11, 32768  # the largest list: 256 KB per 256 segments
    chars, offs = synth.short_reads(synth.genome(61, 50_000, gc=0.45), 62, 1_000, 150, 0.01)
    maker = native.Counter(0)
    maker.set_reads(chars, offs)
    po, ps, pk = maker.superkmers(k, p, parts)
    maker.close()
    # as many reads as make lists of 60% of the free memory; the histograms of the tiles are a thousandth
    max_reads = int(torch.cuda.mem_get_info()[0] * 0.6) // 32768 // 8 * 256
    used = []
    for cap in (0xFFFFFFFF, lists):
        print(f"[gpu] case stream memory lists{cap:#x} reads{max_reads}", flush=True)
        c = native.Counter(0)
        c.set_p1_lists(cap)
        free = torch.cuda.mem_get_info()[0]
        c.stream_begin(k, p, parts, max_reads, len(chars), np.diff(po), ps)
        used.append(free - torch.cuda.mem_get_info()[0])
        c.stream_add(chars, offs)
        pb, sc, kc = c.stream_end()
        assert np.array_equal(pb, np.diff(po)) and np.array_equal(sc, ps) and np.array_equal(kc, pk)
        c.close()
    assert abs(used[1] - used[0]) <= 32 << 20, used


def _mapped():
    """Address space of the process: pinned host memory, and the device's buffers too."""
    with open("/proc/self/status") as f:
        return next(int(line.split()[1]) << 10 for line in f if line.startswith("VmSize:"))


@pytest.mark.parametrize("max_bases,kept", [(300_000_000, False), (100_000_000, True)])
def test_staging_memory_is_given_back(max_bases, kept):
    """The staging sets of a large batch capacity go with their stream, those of a small one stay."""
    chars, offs = synth.short_reads(synth.genome(63, 50_000, gc=0.45), 64, 1_000, 150, 0.01)
    c = native.Counter(0)
    c.set_reads(chars, offs)
    po, ps, _ = c.superkmers(31, 11, 32)
    c.stream_begin(31, 11, 32, 1_000, len(chars), np.diff(po), ps)  # all that is allocated once
    c.stream_add(chars, offs)
    c.stream_end()
    print(f"[gpu] case staging memory {max_bases}", flush=True)
    c.stream_begin(31, 11, 32, 1_000, max_bases, np.diff(po), ps)
    during = _mapped()
    c.stream_add(chars, offs)
    pb, _, _ = c.stream_end()
    after = _mapped()
    assert np.array_equal(pb, np.diff(po))
    assert (during - after >= 2 * max_bases) == (not kept), (during, after)
    c.close()
