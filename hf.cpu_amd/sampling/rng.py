"""The sampler's random numbers: xorshift64*, bit for bit the reference's
(src/sample.c:9-23), so that a seed means the same sequence of draws."""
import numpy as np

MASK64 = (1 << 64) - 1


class Rng:
    def __init__(self, seed):
        self.s = (int(seed) * 0x9e3779b97f4a7c15 + 0x1234567) & MASK64
        if self.s == 0:
            self.s = 0x2545f4914f6cdd1d

    def next_u64(self):
        x = self.s
        x ^= x >> 12
        x ^= (x << 25) & MASK64
        x ^= x >> 27
        self.s = x
        return (x * 0x2545f4914f6cdd1d) & MASK64

    def uniform(self):
        """A float32 in [0, 1) with 24 random bits."""
        return np.float32((self.next_u64() >> 40) * 2.0 ** -24)      # (exact in 64 bits and in 32)


def uniforms(rngs):
    """``[r.uniform() for r in rngs]`` as an fp32 array; many generators move on together in 64-bit integers (64 of them: 15 us, 50 one by one)."""
    if len(rngs) < 8 or len({id(r) for r in rngs}) != len(rngs):     # (one that stands twice draws twice, in order)
        return np.array([r.uniform() for r in rngs], dtype=np.float32)
    x = np.array([r.s for r in rngs], dtype=np.uint64)
    x ^= x >> np.uint64(12)
    x ^= x << np.uint64(25)
    x ^= x >> np.uint64(27)
    for r, s in zip(rngs, x.tolist()):
        r.s = s
    return ((x * np.uint64(0x2545f4914f6cdd1d)) >> np.uint64(40)).astype(np.float32) * np.float32(2.0 ** -24)
