"""Device memory of the incremental evolve: where its buffers cannot be had the iterations are full
ones, with the same results; and calls that repeat at the same sizes allocate nothing (an allocation
in one context would make every stream of the device wait for it)."""

import numpy as np
import pytest

from ridgedetection_amd import synth

pytestmark = pytest.mark.gpu


def _context(dtype):
    from ridgedetection_amd._lib import Context, OPT_LOCAL
    c = Context(3, dtype)
    c.set_option(OPT_LOCAL, 0)
    return c
