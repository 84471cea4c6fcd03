"""Counter-based uniform numbers: u = f(seed, counter), no state to carry."""

from __future__ import annotations

import numpy as np

_MASK = (1 << 64) - 1


def _mix(x: int) -> int:
    """One round of the splitmix64 finaliser."""
    x = (x + 0x9E3779B97F4A7C15) & _MASK
    x = ((x ^ (x >> 30)) * 0xBF58476D1CE4E5B9) & _MASK
    x = ((x ^ (x >> 27)) * 0x94D049BB133111EB) & _MASK
    return x ^ (x >> 31)


def uniform(seed: int, counter: int) -> float:
    """A number in [0, 1) with 24 random bits (exact in float32), fixed by (seed, counter)."""
    value = _mix(_mix(seed & _MASK) ^ ((counter * 0xD1B54A32D192ED03) & _MASK))
    return (value >> 40) / float(1 << 24)


def _mix_array(x: np.ndarray) -> np.ndarray:
    x = x + np.uint64(0x9E3779B97F4A7C15)
    x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return x ^ (x >> np.uint64(31))


def uniforms(seeds: list[int], counters: list[int]) -> np.ndarray:
    """:func:`uniform` of each pair, as float32 (which holds the 24 bits exactly)."""
    mixed = _mix_array(np.array([s & _MASK for s in seeds], dtype=np.uint64))
    steps = np.array([c & _MASK for c in counters], dtype=np.uint64) * np.uint64(0xD1B54A32D192ED03)
    return (_mix_array(mixed ^ steps) >> np.uint64(40)).astype(np.float32) / np.float32(1 << 24)
