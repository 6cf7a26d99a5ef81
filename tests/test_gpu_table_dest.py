"""Where the table is copied to: ordinary and pinned host memory, one of each, a pinned buffer's inside, an
address no wider than the counts', and memory of the device; with more partitions than one gather takes and with one.
The rows are those of the copy into ordinary memory. Whole numbers: equal."""
import numpy as np
import pytest
import torch

from rapidgkc_amd import native, synth

pytestmark = pytest.mark.gpu


def _buffer(kind, nbytes, shift):
    """(address, bytes as an array after the copy) of a buffer of the kind, `shift` bytes into it."""
    if kind == "host":
        b = np.zeros(nbytes + shift, dtype=np.uint8)
        return b.ctypes.data + shift, lambda: b[shift:shift + nbytes]
    t = torch.zeros(nbytes + shift + 64, dtype=torch.uint8, pin_memory=kind == "pinned",
                    device="cuda" if kind == "device" else "cpu")
    torch.cuda.synchronize()
    return t.data_ptr() + shift, lambda: t.cpu().numpy()[shift:shift + nbytes]


@pytest.mark.parametrize("k,p,parts,empty", [(31, 11, 1, 0), (31, 11, 700, 1700), (55, 13, 64, 0)])
def test_copy_table_destinations(k, p, parts, empty):
    g = synth.genome(3 * k, 200_000, gc=0.45)
    chars, offs = synth.short_reads(g, 5, 8_000, 150, 0.01)
    c = native.Counter(0)
    c.set_reads(chars, offs)
    po, _, _ = c.superkmers(k, p, parts)
    st = c.copy_store(int(po[-1]))
    at = np.sort(np.concatenate([np.arange(parts + 1), np.full(empty, parts // 2)]))
    rows, _ = c.count_host_store(st, po[at], parts, k, p)
    c.sort_rows()
    keys, cnts, _ = c.table(rows)
    keys, cnts = keys.view(np.uint8), cnts.view(np.uint8)
    for kk, kc, sk, sc in [("host", "host", 0, 0), ("pinned", "pinned", 0, 0), ("host", "pinned", 0, 0), ("pinned", "host", 0, 0),
                           ("pinned", "pinned", 32, 12), ("pinned", "pinned", 4, 1), ("host", "host", 1, 3), ("device", "device", 0, 0),
                           ("device", "host", 16, 0), ("device", "device", 4, 2)]:
        print(f"[gpu] case copy table k{k} parts{parts}+{empty} to {kk}+{sk} {kc}+{sc}", flush=True)
        (ka, kb), (ca, cb) = _buffer(kk, len(keys), sk), _buffer(kc, len(cnts), sc)
        for to_k, to_c in ((ka, ca), (ka, None), (None, ca)):
            assert native.lib().rgkc_copy_table(c._h, to_k, to_c) == 0
            assert to_k is None or np.array_equal(kb(), keys)
            assert to_c is None or np.array_equal(cb(), cnts)
    c.close()
