"""Pinned host rows for steps that are queued without a wait for the one before."""
from __future__ import annotations

from typing import Callable, Generic, List, Optional, TypeVar

import torch

T = TypeVar("T")


class StagingRing(Generic[T]):
    """``n`` sets of rows in turn, one a step: a queued step reads its own set, and a set is written again only when the step that
    had it is through, which an event behind every half of the ring tells.  (An event a step costs the stream a few us.)  One
    stream at a time, as the device buffers that the rows go to.  Without a GPU one set is enough.

    ``make(n)`` allocates all of them (pinned memory costs a few us a piece) -> the function that gives set i when it is first
    used: views of sixteen sets at once were 30 us of an engine's construction."""

    def __init__(self, make: Callable[[int], Callable[[int], T]], cuda: bool, n: int = 16):
        self.sets: List[Optional[T]] = [None] * (n if cuda else 1)
        self._make = make(len(self.sets))
        self._done = [torch.cuda.Event(), torch.cuda.Event()] if cuda else []  # behind the last use of either half
        self._at, self._used = 0, False  # the next step's set

    def __len__(self) -> int:
        return len(self.sets)

    def peek(self) -> T:
        """The next step's set, free to be written; it stays the next one until take()."""
        if self._done:
            half, first = divmod(self._at, len(self.sets) // 2)
            if first == 0:
                self._done[1 - half].record()  # (behind every step queued so far)
                if self._used:
                    self._done[half].synchronize()
                self._used = self._used or half == 1
        st = self.sets[self._at]
        if st is None:
            st = self.sets[self._at] = self._make(self._at)
        return st

    def take(self) -> None:
        """What reads that set is queued."""
        self._at = (self._at + 1) % len(self.sets)

    def next(self) -> T:
        """peek() and take(), where what reads the set is queued right behind."""
        st = self.peek()
        self.take()
        return st
