"""The engine workspace's layout (make_layout in astra-cuda_amd/csrc/market.hip), for
tests that compare two workspaces byte for byte.

The book state must agree exactly, but the head-size cache may know more in one
workspace than in the other: a multi-step launch caches the size of every head it
hands out as a BBO, single calls only those whose order record they hold in
registers (get_bbos reads the others from the book, so both give the same
BBOs). ``normalized`` clears the cache's flags (bit 15 of each half of the tob
word that holds a slot; an empty head, 0xFFFF, keeps its value) and its size
array. Nor has an empty level's word a value (its mask bit says that it is empty,
and what its last orders left there is not read): ``normalized`` sets both words of
each side without its bit to NULL. Everything else stays as it is.

The workspace starts with 256 bytes of control words (int32): the TID counter
of a book with no markets (otherwise every market keeps a copy in ``tids``) and
the count of helper wavefronts that gave up waiting.
"""
from __future__ import annotations


def _align(x: int, a: int = 256) -> int:
    return (x + a - 1) // a * a


def mask_words(L: int) -> int:
    w = 1
    while w * 64 < L:
        w *= 2
    return w


def layout(M: int, L: int, O: int, C: int) -> dict:
    """(byte offset, bytes) of each array of the workspace."""
    W = mask_words(L)
    off, out = 0, {}
    for name, nbytes in (("ctl", 256), ("masks", 2 * W * M * 8), ("next_slot", M * 4), ("tids", M * 4),
                         ("bbo", 2 * M * 4),
                         ("tob", M * 4), ("hsz", 2 * M * 4), ("levels", M * L * 8),
                         ("records", M * O * 16), ("portfolios", M * C * 8)):
        out[name] = (off, nbytes)
        off = _align(off + nbytes)
    out["total"] = (0, off)
    return out


def normalized(ws, M: int, L: int, O: int, C: int):
    """A copy of the workspace bytes (a numpy or torch uint8 array) with the
    head-size cache cleared and the empty levels' words NULL."""
    import numpy as np
    if not isinstance(ws, np.ndarray):
        import torch
        return torch.from_numpy(normalized(ws.cpu().numpy(), M, L, O, C))
    w, lay = ws.copy(), layout(M, L, O, C)

    def array(name, dtype):
        o, n = lay[name]
        return w[o:o + n].view(dtype)

    # bit 15 of a half flags a cached size; 0xFFFF (empty) carries no flag
    h = array("tob", np.uint16)
    h[h != 0xFFFF] &= 0x7FFF
    array("hsz", np.uint8)[:] = 0
    bits = array("masks", np.uint64).reshape(2, mask_words(L), M).transpose(2, 0, 1)
    bits = np.ascontiguousarray(bits).view(np.uint8)
    live = np.unpackbits(bits, axis=2, count=L, bitorder="little").transpose(0, 2, 1)  # [M, L, 2]
    array("levels", np.uint32).reshape(M, L, 2)[live == 0] = 0xFFFFFFFF  # {head, tail} of a side
    return w
