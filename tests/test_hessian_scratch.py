"""Scratch of ``hi2x_hessian_accumulate`` by its size query, on the CPU."""

import pytest


@pytest.mark.parametrize("k", [16, 256, 4096, 14336, 28672])
def test_fp32_scratch_does_not_grow_with_the_tokens(k):
    """The planes of fp32 tokens (6 bytes an element) stay within 512 MiB; the rest is the
    partial sums that as many bf16 tokens take, and those of at most 256 tail tiles."""
    from hi2_amd import _lib

    f = _lib.lib().hi2x_hessian_accumulate_workspace_bytes
    parts = max(f(2, t, k) - 2 * t * k for t in (1 << 10, 1 << 13, 1 << 16))
    assert f(0, 1, k) == 0  # the fp32 kernel
    for t in (70, 10 ** 6, (1 << 22) // 3, 10 ** 7, 10 ** 8):
        assert 0 < f(0, t, k) <= (512 << 20) + parts + (64 << 20)
