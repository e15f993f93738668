"""The finish's un-permutation of codes and compensated weights (``hi2x_finish``): rows turned in
LDS by 512 or 1024 threads, and element by element where they do not fit or are not aligned.
Bytes and floats are moved, so the results are equal."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# the smallest rows, one and several float4 a thread, the last row length of 512 and of 1024
# threads, and the first past both; more rows than workgroups
@pytest.mark.parametrize("n,k", [(1, 16), (3, 48), (1030, 2064), (5, 8192), (300, 8208),
                                 (2, 16384), (2, 16400)])
@pytest.mark.parametrize("comp", [True, False])
@pytest.mark.parametrize("shift", [0, 1])
def test_finish_unpermutes(n, k, comp, shift, dev):
    from hi2_amd import _lib

    g = torch.Generator(device=dev).manual_seed(n + k)
    codes_ro = torch.randint(0, 256, (n, k), generator=g, device=dev, dtype=torch.uint8)
    # shift: outputs that are not aligned for the wide accesses
    codes = torch.full((n * k + shift,), 77, dtype=torch.uint8, device=dev)[shift:].view(n, k)
    comp_ro = torch.randn(n, k, generator=g, device=dev) if comp else None
    out = torch.zeros(n * k + shift, device=dev)[shift:].view(n, k) if comp else None
    perm = torch.randperm(k, generator=g, device=dev)
    zeros = torch.zeros(n, k // 16, device=dev)
    w, d, sse = torch.zeros(n, k, device=dev), torch.ones(k, device=dev), torch.empty(n, device=dev)
    print(f"finish n={n} k={k} comp={comp} shift={shift}", flush=True)
    _lib.call("hi2x_finish", w.device, _lib.ptr(codes_ro), _lib.ptr(comp_ro), _lib.ptr(perm), n, k,
              16, _lib.ptr(zeros), _lib.ptr(zeros), k // 16, _lib.ptr(w), _lib.ptr(d),
              _lib.ptr(codes), _lib.ptr(out), _lib.ptr(sse))
    want = torch.empty_like(codes_ro)
    want[:, perm] = codes_ro
    assert torch.equal(codes, want)
    if comp:
        back = torch.empty_like(comp_ro)
        back[:, perm] = comp_ro
        assert torch.equal(out, back)
    assert torch.equal(sse, torch.zeros_like(sse))
