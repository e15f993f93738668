"""The QAD decode with its transform in one pass (``hi2x_qad_weights_fwd/bwd``) equals the decode
and ``wht_scale`` one after the other, bit for bit, in values and every gradient."""

from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu


def _fq(n, k, unit, has_scale, flags, dev, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    p = torch.randperm(n, generator=g, device=dev)
    cuts = [(p[: n // 3], 2, 32), (p[n // 3: n // 2], 8, 64), (p[n // 2:], 4, 16)]
    groups = []
    for rows, nb, b in cuts:
        if rows.numel() == 0 or k % b:
            continue
        m = rows.numel()
        consts = torch.stack([torch.rand(m, generator=g, device=dev) * -0.05,
                              torch.full((m,), 2e-4, device=dev),
                              torch.full((m,), 1e-4, device=dev)], 1).half()
        lo, st = (torch.rand(m, k // b, generator=g, device=dev) * 255 for _ in range(2))
        st[:, 0] = 0.0  # a zero step
        groups.append(SimpleNamespace(rows=rows.sort().values, consts=consts, nbits=nb, block=b,
                                      lo_u=lo.requires_grad_(), step_u=st.requires_grad_()))
    latent = (torch.randn(n, k, generator=g, device=dev) * 0.02).requires_grad_()
    u = torch.rand(n, k, generator=g, device=dev) + 0.5 if unit else torch.ones(0, device=dev)
    had = (torch.rand(k // 16, generator=g, device=dev) < 0.5).to(torch.uint8) if flags else \
        torch.zeros(k // 16, dtype=torch.uint8, device=dev)
    scale = (torch.rand(k, generator=g, device=dev) + 0.5).half()
    return SimpleNamespace(latent=latent, unit=u, groups=groups, had=had, col_scale=scale,
                           has_had=flags, has_scale=has_scale)


@pytest.mark.parametrize("n,k", [(3, 64), (7, 192), (64, 320), (129, 4096)])
@pytest.mark.parametrize("unit", [False, True])
@pytest.mark.parametrize("flags,scale", [(True, False), (True, True), (False, True)])
def test_fused_equals_two_passes(n, k, unit, flags, scale, dev):
    from hi2_amd.qad_kernel import _StoredDecode, _Transform, original

    fq = _fq(n, k, unit, scale, flags, dev, n + k)
    meta = [(g.rows, g.consts, g.nbits, g.block) for g in fq.groups]
    params = [p for g in fq.groups for p in (g.lo_u, g.step_u)]
    leaves = [fq.latent] + params
    cs = fq.col_scale if scale else fq.col_scale[:0]
    grad = torch.randn(n, k, device=dev)
    print(f"qad fused n={n} k={k}", flush=True)
    rows = torch.cat([g.rows for g in fq.groups])
    two = _Transform.apply(_StoredDecode.apply(fq.latent, fq.unit, meta, *params), fq.had, cs)
    one = original(fq)
    assert torch.equal(one[rows], two[rows])
    a, b = torch.autograd.grad(one, leaves, grad), torch.autograd.grad(two, leaves, grad)
    assert torch.equal(a[0][rows], b[0][rows])
    assert all(torch.equal(x, y) for x, y in zip(a[1:], b[1:]))
    with torch.no_grad():
        assert torch.equal(original(fq)[rows], two[rows])


def test_an_absent_smoothing_vector_may_be_anywhere(dev):
    """Without smoothing, ``col_scale`` is not read and need not be on the device."""
    from hi2_amd.qad_kernel import original

    fq = _fq(7, 192, True, False, True, dev, 3)
    rows = torch.cat([g.rows for g in fq.groups])
    grad = torch.randn(7, 192, device=dev)
    want = original(fq)
    gw, = torch.autograd.grad(want, [fq.latent], grad)
    for cs in (fq.col_scale.cpu(), torch.empty(0)):
        fq.col_scale = cs
        got = original(fq)
        gg, = torch.autograd.grad(got, [fq.latent], grad)
        assert torch.equal(got[rows], want[rows]) and torch.equal(gg[rows], gw[rows])
