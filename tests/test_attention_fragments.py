"""Where the matrix-core attention kernels read a key's row, walked over on the CPU: the offsets come from the
compiled module, which needs no GPU to be asked for them."""

from __future__ import annotations

import ctypes

import pytest

from kvforge_amd.kernels import library


@pytest.mark.parametrize("d", range(16, 257, 16))
@pytest.mark.parametrize("pages,KV,bs", [(1, 1, 8), (2, 3, 16)])
def test_every_fragment_of_a_key_lies_in_its_row(d, pages, KV, bs):
    """A key's row is d / 8 fragments of 16 bytes, and a step takes four of them, one a lane group.  A step that
    reaches past the row (d / 16 odd) reads inside it all the same: behind the last head's last slot of the last
    page the tensor ends."""
    fragment = ctypes.CDLL(library.build_module("attn_mfma")).kvf_attn_mfma_key_fragment
    steps, row = (d // 16 + 1) // 2, d // 8
    size = pages * KV * bs * row
    for page in range(pages):
        for head in range(KV):
            for slot in range(bs):
                base = ((page * KV + head) * bs + slot) * row
                read = [base + fragment(d, c, group) for c in range(steps) for group in range(4)]
                assert all(base <= at < base + row and at < size for at in read)
                assert read[:row] == list(range(base, base + row))
