"""A device buffer of the context, filled before a run and read back whole: for tests that look at every word around a
result (a result in host memory goes through staging, so a stray store of the kernel would not show there)."""
import numpy as np

import ork


class Filled:
    def __init__(self, npu, shape, dtype, fill):
        self.npu = npu
        self.init = np.full(shape, fill, dtype)
        self.base = ork.lib().ork_dev_alloc(npu.h, self.init.nbytes)
        assert self.base and ork.lib().ork_dev_upload(npu.h, self.base, ork.ptr(self.init), self.init.nbytes) == 0

    def at(self, words):
        """the address of word `words` (4-byte elements)"""
        return self.base + 4 * words

    def get(self):
        out = np.empty_like(self.init)
        assert ork.lib().ork_dev_download(self.npu.h, ork.ptr(out), self.base, out.nbytes) == 0
        return out

    def free(self):
        ork.lib().ork_dev_free(self.npu.h, self.base)
