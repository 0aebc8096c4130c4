"""Values on their way to and from the device: the ring of pinned slots uploads go through, the polled pieces of a read."""
import numpy as np
import pytest


# the ring's slots are used again and again: every upload reads what the host wrote last, at each size and remainder
@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 3, 5, 64, 1023, 4097, 16384])
def test_a_slot_of_the_ring_is_read_anew(hip, n):
    for again in range(4):
        sent = [np.arange(n, dtype=np.uint32) * np.uint32(2654435761) + np.uint32(again * 100 + i) for i in range(20)]
        held = [hip.ndarray_from_vec_u32(a, [n]) for a in sent]
        for a, t in zip(sent, held):
            assert np.array_equal(hip.to_vec(t), a)
