"""The super-block column loops of few-row batches (``gptq_super_kernel``) on the MI355X: equal
bit for bit to the per-block schedule, which runs the separate kernels, at the edges of its
16-row workgroups, 128-column blocks, super-blocks and factor runs, and in the waves that leave
the fast loop's numerical range."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(n, k, dev, seed, groups=1):
    g = torch.Generator(device=dev).manual_seed(seed)
    w = torch.randn(n, k, generator=g, device=dev) * 0.02
    us = []
    for _ in range(groups):
        u = torch.triu(torch.randn(k, k, generator=g, device=dev) / (4 * k) ** 0.5, 1)
        u.diagonal().copy_(torch.rand(k, generator=g, device=dev) + 0.5)
        us.append(u)
    d = torch.rand(k, generator=g, device=dev) + 0.1
    return w, d, us


def _same(a, b):
    for x, y in zip(a, b):
        for f in ("codes", "params", "consts", "sse", "comp"):
            p, q = getattr(x, f), getattr(y, f)
            assert torch.equal(p.view(torch.uint8) if p.dtype.is_floating_point else p,
                               q.view(torch.uint8) if q.dtype.is_floating_point else q), f


@pytest.mark.parametrize("n,k,sb", [
    (1, 256, 2), (15, 384, 4), (16, 512, 4), (17, 640, 4), (33, 1056, 4), (100, 1088, 8),
    (64, 1152, 8), (250, 2112, 8), (4096, 512, 4), (4097, 512, 4), (48, 16, 4), (31, 144, 8)])
def test_equals_the_separate_schedule(n, k, sb, dev):
    from hi2_amd.hessian import GptqJob, encode_jobs_gptq

    w, d, (u,) = _inputs(n, k, dev, n + k)
    b = 64 if k % 64 == 0 else 16
    jobs = [GptqJob(w, d, u, 4, b)]
    if n > 8:  # a second row class of the same factor in one batch
        jobs = [GptqJob(w[: n // 3], d, u, 2, 32 if k % 32 == 0 else 16),
                GptqJob(w[n // 3:], d, u, 4, b)]
    print(f"fused n={n} k={k} sb={sb}", flush=True)
    _same(encode_jobs_gptq(jobs, comp=True, super_blocks=sb),
          encode_jobs_gptq(jobs, comp=True, super_blocks=1))


def test_workgroups_of_two_factors(dev):
    """Unpadded runs of two factors inside one 16-row workgroup (callers of the C entry)."""
    from hi2_amd import _lib

    n, k = 40, 512
    w, d, us = _inputs(n, k, dev, 9, groups=2)
    grp = torch.tensor([0] * 5 + [1] * 14 + [0] * 0 + [2] * 21, dtype=torch.int32, device=dev)
    ptrs = torch.tensor([us[0].data_ptr(), us[1].data_ptr(), us[0].data_ptr()],
                        dtype=torch.int64, device=dev)
    blk = (torch.arange(k, device=dev, dtype=torch.int32) // 64).repeat(3, 1).contiguous()
    nmax = torch.tensor([15.0, 3.0, 15.0], device=dev)
    lo = w.reshape(n, 8, 64).amin(-1).contiguous()
    st = ((w.reshape(n, 8, 64).amax(-1) - lo) / nmax[grp.long()][:, None]).half().float().contiguous()
    lo = lo.half().float()
    out = []
    for sb in (1, 4):
        wc, codes = w.clone(), torch.zeros(n, k, dtype=torch.uint8, device=dev)
        comp, ws = torch.zeros(n, k, device=dev), torch.empty(n, 128 * sb, device=dev)
        print(f"two factors sb={sb}", flush=True)
        _lib.call("hi2x_gptq_run", w.device, _lib.ptr(wc), n, k, _lib.ptr(codes), _lib.ptr(lo),
                  _lib.ptr(st), 8, _lib.ptr(grp), _lib.ptr(ptrs), _lib.ptr(blk), _lib.ptr(nmax),
                  _lib.ptr(comp), _lib.ptr(ws), sb)
        out.append((codes, comp))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


@pytest.mark.parametrize("n,k,runs", [(1, 256, [1]), (17, 1088, [17]), (40, 640, [5, 14, 21]),
                                      (64, 1168, [16, 48])])
@pytest.mark.parametrize("sb", [4, 8])
def test_working_copy_is_updated_in_place(n, k, runs, sb, dev):
    """``hi2x_gptq_run`` leaves every column of ``wc`` with the updates of the blocks before its
    own, whatever the schedule: the per-block one's bits."""
    from hi2_amd import _lib

    w, d, us = _inputs(n, k, dev, n + k, groups=2)
    grp = torch.repeat_interleave(torch.arange(len(runs)), torch.tensor(runs)).int().to(dev)
    ptrs = torch.tensor([us[i % 2].data_ptr() for i in range(len(runs))], dtype=torch.int64,
                        device=dev)
    blk = (torch.arange(k, device=dev, dtype=torch.int32) // 16).repeat(len(runs), 1).contiguous()
    nmax = torch.full((len(runs),), 15.0, device=dev)
    lo = w.reshape(n, -1, 16).amin(-1).half().float().contiguous()
    st = ((w.reshape(n, -1, 16).amax(-1) - lo) / 15.0).half().float().contiguous()
    out = []
    for s in (1, sb):
        wc, codes = w.clone(), torch.zeros(n, k, dtype=torch.uint8, device=dev)
        ws = torch.empty(n, 128 * s, device=dev)
        print(f"working copy n={n} k={k} sb={s}", flush=True)
        _lib.call("hi2x_gptq_run", w.device, _lib.ptr(wc), n, k, _lib.ptr(codes), _lib.ptr(lo),
                  _lib.ptr(st), k // 16, _lib.ptr(grp), _lib.ptr(ptrs), _lib.ptr(blk),
                  _lib.ptr(nmax), None, _lib.ptr(ws), s)
        out.append((wc, codes))
    assert not torch.equal(out[0][0], w)
    assert torch.equal(out[0][0].view(torch.int32), out[1][0].view(torch.int32))
    assert torch.equal(out[0][1], out[1][1])


@pytest.mark.parametrize("value", [0.0, -0.0, 1e-30, -1e-30, 3e20, float("inf"), float("nan")])
def test_values_outside_the_fast_range(value, dev):
    from hi2_amd.hessian import GptqJob, encode_jobs_gptq

    n, k = 20, 512
    w, d, (u,) = _inputs(n, k, dev, 4)
    w[3, :] = value
    w[7, 130] = value
    jobs = [GptqJob(w, d, u, 4, 64)]
    print(f"fused value {value}", flush=True)
    _same(encode_jobs_gptq(jobs, comp=True, super_blocks=4),
          encode_jobs_gptq(jobs, comp=True, super_blocks=1))
