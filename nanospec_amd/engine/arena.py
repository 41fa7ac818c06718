"""A bump allocator for the intermediates of one step.

Every buffer a part needs between kernels comes from here, so a step allocates nothing from the
framework's general allocator once the arena has grown to its working size, and a captured graph
owns an arena of fixed size whose addresses never change.  ``mark``/``release`` let a layer hand its
buffers back for the next layer.
"""

from __future__ import annotations

import torch

_ALIGN = 256
_ESIZE: dict = {}  # bytes per element of the types asked for so far


class Arena:
    def __init__(self, device, nbytes: int = 0, fixed: bool = False) -> None:
        self.device, self.fixed = device, fixed
        self._chunks: list[torch.Tensor] = []
        self._sizes: list[int] = []  # bytes of each chunk
        self._typed: dict = {}  # (chunk, dtype) -> the chunk seen as that type
        self._cur, self._off = -1, 0
        # of a captured step that ends in padding: how many rows it has, and (int32 [1] on the device) how many of them are read by anyone.  Products of so many rows
        # may leave the others undone
        self.read_rows: tuple[int, torch.Tensor] | None = None
        self.high_water = 0  # the most bytes that were in use at once since the arena was made (tails of chunks that a buffer
        #                      did not fit into count as used: one chunk of this size holds the same sequence of buffers)
        if nbytes:
            self._add(nbytes)
            self._cur = 0

    def _add(self, nbytes: int) -> None:
        self._chunks.append(torch.empty(nbytes, dtype=torch.uint8, device=self.device))
        self._sizes.append(nbytes)

    def take(self, shape, dtype) -> torch.Tensor:
        esize = _ESIZE.get(dtype) or _ESIZE.setdefault(dtype, torch.empty(0, dtype=dtype).element_size())
        # (a step of a small model asks a hundred times, kernel by kernel, and is bound by the host there: one view a buffer, no
        # tensor asked for its size)
        count, strides = 1, []
        for s in reversed(shape):
            strides.append(count)
            count *= int(s)
        strides.reverse()
        need = -(-max(1, count) * esize // _ALIGN) * _ALIGN
        while self._cur < 0 or self._off + need > self._sizes[self._cur]:
            if self._cur + 1 < len(self._chunks):
                self._cur, self._off = self._cur + 1, 0
                continue
            if self.fixed:
                raise RuntimeError(f"a fixed arena of {sum(self._sizes)} bytes is exhausted")
            self._add(max(need, 2 * sum(self._sizes), 1 << 20))
            self._cur, self._off = len(self._chunks) - 1, 0
        # a view of the chunk in the wanted type is kept, so a buffer costs one view (offsets are multiples of 256 bytes,
        # hence of every element size)
        typed = self._typed.get((self._cur, dtype))
        if typed is None:
            chunk = self._chunks[self._cur]
            typed = self._typed[self._cur, dtype] = chunk[: self._sizes[self._cur] // esize * esize].view(dtype)
        out = typed.as_strided(tuple(shape), tuple(strides), self._off // esize)
        self._off += need
        used = self._off + (sum(self._sizes[: self._cur]) if self._cur else 0)
        if used > self.high_water:
            self.high_water = used
        return out

    @property
    def capacity(self) -> int:
        return sum(self._sizes)

    def mark(self) -> tuple[int, int]:
        return self._cur, self._off

    def release(self, mark: tuple[int, int]) -> None:
        self._cur, self._off = mark

    def reset(self) -> None:
        """Start of a step.  Several chunks mean the arena grew during the last step: merge them."""
        if len(self._chunks) > 1 and not self.fixed:
            total = sum(self._sizes)
            self._chunks, self._sizes = [], []
            self._typed.clear()
            self._cur, self._off = -1, 0  # (one chunk of that size may not be had where the several were: the next buffers then start anew)
            self._add(total)
        self._cur, self._off = (0, 0) if self._chunks else (-1, 0)
