"""Chunked streams edited by hand: chunks that are not back to back, empty or
cut short, which the rounds of the speculative runs leave to other paths."""
import dataclasses

import numpy as np

# Edits that keep every chunk's codewords, and edits that do not.
LOSSLESS = ["swapped", "gap", "gap-late", "padded", "shuffled"]
LOSSY = ["empty", "empty-first", "short-last", "cut"]


def edited(enc, kind):
    """enc with one edit: the middle two chunks' bytes exchanged, 16 bytes
    before the middle chunk or one near the end, every chunk padded to 16
    bytes, the chunks in a random order, the middle or first chunk empty, the
    last one cut short, or every chunk from the middle on without its last
    byte (the stream re-packed, so that they stay back to back)."""
    packed = np.asarray(enc.packed, np.uint8)
    offs = np.array(enc.chunk_offsets, np.int32)
    nb = np.array(enc.chunk_nbytes, np.int32)
    k = len(offs) // 2
    if kind.startswith("gap"):
        at = k if kind == "gap" else 7 * len(offs) // 8
        packed = np.concatenate([packed[: offs[at]], np.full(16, 0x5A, np.uint8), packed[offs[at]:]])
        offs[at:] += 16
    elif kind == "empty":
        nb[k] = 0
    elif kind == "empty-first":
        nb[0] = 0
    elif kind == "short-last":
        nb[-1] -= 60
    else:
        if kind == "cut":
            nb[k:] -= 1
        order = np.arange(len(offs))
        if kind == "swapped":
            order[[k, k + 1]] = order[[k + 1, k]]
        elif kind == "shuffled":
            order = np.random.default_rng(7).permutation(order)
        parts = [packed[offs[c]: offs[c] + nb[c]] for c in order]
        if kind == "padded":
            parts = [np.pad(q, (0, -len(q) % 16), constant_values=0x5A) for q in parts]
        offs[order] = np.concatenate([[0], np.cumsum([len(q) for q in parts])[:-1]])
        packed = np.concatenate(parts + [np.zeros(8, np.uint8)])
    return dataclasses.replace(enc, packed=packed, chunk_offsets=offs, chunk_nbytes=nb)
