"""A forced kernel is looked up by its name alone, and again once the registry changed or the memo is cleared."""

from __future__ import annotations

import pytest
import torch

from ako_amd.dispatcher.cache import KernelCache
from ako_amd.dispatcher.registry import KernelEntry, KernelRegistry
from ako_amd.dispatcher.selector import KernelSelector


def test_forced_kernels(tmp_path) -> None:
    registry = KernelRegistry()
    first, second = (lambda x: x), (lambda x: x + 1)
    registry.register(KernelEntry("op", "a", first, backend="pytorch", priority=10))
    registry.register(KernelEntry("op", "b", second, backend="hip", priority=5))
    selector = KernelSelector(registry=registry, cache=KernelCache(path=tmp_path / "cache.json"))
    for shape in ((2,), (3, 4)):
        x = torch.zeros(shape)
        assert selector.select("op", x, forced="a") is first
        assert selector.select("op", x, forced="b") is second
        assert selector.select("op", x) is first  # the default on a CPU tensor
    with pytest.raises(ValueError, match="Unknown kernel"):
        selector.select("op", torch.zeros(2), forced="c")
    registry.register(KernelEntry("op", "b", first, backend="hip", priority=5))
    selector.clear_memo()
    assert selector.select("op", torch.zeros(2), forced="b") is first


def test_forced_kernels_follow_the_registry(tmp_path) -> None:
    """A kernel replaced or dropped after a forced call is not called again, at any shape."""
    registry = KernelRegistry()
    first, second = (lambda x: x), (lambda x: x + 1)
    registry.register(KernelEntry("op", "a", first, backend="pytorch", priority=10))
    registry.register(KernelEntry("op", "b", first, backend="hip", priority=5))
    selector = KernelSelector(registry=registry, cache=KernelCache(path=tmp_path / "cache.json"))
    assert selector.select("op", torch.zeros(2), forced="b") is first
    registry.register(KernelEntry("op", "b", second, backend="hip", priority=5))
    assert selector.select("op", torch.zeros(3), forced="b") is second
    assert selector.select("op", torch.zeros(2), forced="b") is second
    registry.unregister("op", "b")
    with pytest.raises(ValueError, match="Unknown kernel"):
        selector.select("op", torch.zeros(3), forced="b")
