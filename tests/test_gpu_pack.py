"""Base codes, four bytes at a time: every byte value at every place of a word, among bases of each kind. The
oracle reads the same characters: stores are equal, byte for byte."""
import numpy as np
import pytest

from test_gpu_parity import check_store

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift", [0, 1, 2, 3])
def test_every_byte(shift):
    from rapidgkc_amd import native
    print(f"[gpu] case pack every byte at place {shift}", flush=True)
    rng = np.random.default_rng(shift)
    codes = {**{ord(c): ord(c) for c in "ACGT"}, **{ord(c): ord(c.upper()) for c in "acgt"}}
    chars = rng.choice(np.frombuffer(b"ACGTacgt", dtype=np.uint8), 4 * 4 * 256 + 64)
    chars[shift:shift + 4 * 4 * 256:4] = np.tile(np.arange(256, dtype=np.uint8), 4)
    plain = np.array([codes.get(int(c), ord("A")) for c in chars], dtype=np.uint8)  # any other byte counts as A
    offs = np.array([0, len(chars)], dtype=np.uint64)
    c = native.Counter(0)
    c.set_reads(chars, offs)
    check_store(c, plain, offs, 21, 7, 5)
    c.close()
