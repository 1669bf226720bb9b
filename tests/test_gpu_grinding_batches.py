"""Nonce searches whose answer lies past the first batch (2^(g+2) candidates, at
least 2^16) or on a search limit, through both entry points (smallest nonce, exact)."""
import ctypes as C
import random

import pytest

pytestmark = pytest.mark.gpu


def _search(name, seed, g, limit):
    from lambda_vm_amd import _native as N

    out = C.c_uint64(0)
    rc = getattr(N.lib(), name)((C.c_uint8 * 32)(*seed), C.c_uint8(g), C.c_uint64(limit), C.byref(out))
    return rc, out.value


@pytest.mark.parametrize("g", [14, 15])
def test_nonce_past_the_first_batch(gpu, ora, g):
    rng = random.Random(g)
    found = 0
    for _ in range(600):
        seed = bytes(rng.getrandbits(8) for _ in range(32))
        want = ora.generate_nonce(seed, g)
        if want < 1 << (g + 2):
            continue
        found += 1
        for name in ("lvm_generate_nonce", "lvm_generate_nonce_noalloc"):
            assert _search(name, seed, g, 1 << 40) == (0, want)
            # the limit is exclusive: the answer itself is not below it, or it is by one
            assert _search(name, seed, g, want)[0] != 0
            assert _search(name, seed, g, want + 1) == (0, want)
        if found == 3:
            return
    assert found, "no seed of the run needs a second batch"
