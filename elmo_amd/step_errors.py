"""Failures of the persistent step kernels, reported without synchronising.

The reference has no counterpart: its kernels do not wait for one another.  Here the workgroups that share a tile sequence
do, with a bound; the last kernel of a step ORs the step's error word into a sticky word of the workspace, and while that
is not zero every step also changes a word of host memory (include/elmo_xmc.h, xmc_failure_word).  Looking at that word is
an ordinary memory read, so a layer does it before every step; only when it has changed does it wait for the device and
read the sticky words of its own workspaces.
"""
import ctypes

import torch

from . import _lib


def _failure_words(device):
    """The host addresses of the device's two failure words, as ctypes integers."""
    with torch.cuda.device(device):
        address = _lib.load().xmc_failure_word()
    if not address:
        raise _lib.XmcError("no failure word: not a gfx950 device, or no pinned host memory")
    return ctypes.c_int.from_address(address), ctypes.c_int.from_address(address + 4)


def _failure(word):
    return RuntimeError(
        f"a classifier step failed (error word {word}): "
        + ("a workgroup gave up waiting for its partners (another stream kept the device busy?); " if word & 1 else "")
        + ("workgroups that exchange data were not placed on one XCD; " if word & 2 else "")
        + "the weights and grad_input of that step are incomplete")


class UnkeptStepErrors:
    """Failures of the steps on a device that were given no workspace: the one they ran in went away with the call, and
    its error word was passed on to the device's second failure word."""

    def __init__(self, device):
        self.device = torch.device(device)
        self._word = _failure_words(self.device)[1]
        self._seen = 0

    def check(self):
        """Raises if such a step has announced a failure.  Waits only if one has."""
        if self._word.value != self._seen:
            self.check_now()

    def check_now(self):
        """Waits for the steps enqueued so far and raises if such a step among them failed."""
        torch.cuda.synchronize(self.device)
        word = self._word.value      # (never cleared: a failure announced from here on changes it again)
        if word != self._seen:
            self._seen = word
            raise _failure(word & 3)


class StepErrors:
    """The sticky error words of a layer's workspaces.  `words`: int32 device tensors of one element each."""

    def __init__(self, device, words):
        self.device = torch.device(device)
        self.words = list(words)
        self._watch()

    def _watch(self):
        self._word = _failure_words(self.device)[0]
        self._seen = self._word.value

    def __getstate__(self):      # copies and pickles of a layer watch the word of the process they live in
        return {"device": self.device, "words": self.words}

    def __setstate__(self, state):
        self.__dict__.update(state)
        self._watch()

    def pending(self):
        """Whether a step on the device has announced a failure that this layer has not looked into."""
        return self._word.value != self._seen

    def check(self):
        """Raises if a step of this layer failed and has announced it.  Waits only if some step on the device has."""
        if self._word.value != self._seen:
            self.check_now()

    def check_now(self):
        """Waits for the steps enqueued so far and raises if any of this layer's failed."""
        torch.cuda.synchronize(self.device)
        word = 0
        for w in self.words:
            word |= int(w.item())
        if word != 0:
            for w in self.words:
                w.zero_()
            torch.cuda.synchronize(self.device)
        self._seen = self._word.value
        if word != 0:
            raise _failure(word)
