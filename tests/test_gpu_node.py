"""The factor of one recursion node (``node_kernel``, up to 256 columns in one workgroup) on
the MI355X against float64: sizes at the edges of its 16-column tiles and 128-column halves,
several matrices per launch, and pivots that fail in either half; and the products that join two
nodes and more, at ranks and widths that end inside a 64-tile and a 32-rank chunk."""

import pytest
import torch

pytestmark = pytest.mark.gpu

# one workgroup (<= 256 columns), the smallest sizes of two, and several joined by products
SIZES = [4, 12, 16, 20, 60, 124, 128, 132, 240, 252, 256, 260, 388, 516, 772, 1020, 1156]


def _hessian(k, dev, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    x = torch.randn(4 * k + 64, k, generator=g, device=dev, dtype=torch.float64)
    x[:, ::7] *= 20.0
    return x.T @ x / x.shape[0]


def _factor64(h, damp=0.01):
    a = h + damp * h.diagonal().mean() * torch.eye(h.shape[0], dtype=h.dtype, device=h.device)
    low = torch.linalg.cholesky(a.flip(0, 1))
    eye = torch.eye(h.shape[0], dtype=h.dtype, device=h.device)
    return torch.linalg.solve_triangular(low, eye, upper=False).flip(0, 1)


@pytest.mark.parametrize("k", SIZES)
def test_node_sizes_against_float64(k, dev):
    from hi2_amd.hessian import inverse_factor, inverse_factors_batched

    hs = torch.stack([_hessian(k, dev, 100 * k + i) for i in range(3)]).float()
    print(f"node k={k}", flush=True)
    us = inverse_factors_batched(hs, 0.01)
    for h, u in zip(hs, us):
        want = _factor64(h.double())
        # the damped Hessian's condition is at most about 400 / 0.01 / 4: fp32 rounding of its
        # k-term sums, u = 2^-24, moves the factor by well under cond u sqrt(k) = 1e-2; the
        # measured error is below 3e-6 at every size, held to four times that
        assert torch.linalg.norm(u.double() - want) <= 1.2e-5 * torch.linalg.norm(want)
        assert torch.equal(u.tril(-1), torch.zeros_like(u))
        assert torch.equal(u, inverse_factor(h, 0.01))


@pytest.mark.parametrize("at", [0, 17, 127, 128, 200, 255])
def test_node_reports_a_failing_pivot(at, dev):
    from hi2_amd import _lib

    k = 256
    h = _hessian(k, dev, 3).float()
    i = k - 1 - at  # the factor runs on the reversed matrix
    h[i, i] = -1e4
    u = torch.empty_like(h)
    ws = _lib.workspace(dev, "hi2x_chol_workspace_bytes", k)
    print(f"node failing pivot {at}", flush=True)
    with pytest.raises(_lib.NotPositiveDefinite, match=f"block at {at // 128 * 128} "):
        _lib.call("hi2x_chol_inv_upper", h.device, _lib.ptr(h), k, 0.0, 0, _lib.ptr(u),
                  _lib.ptr(ws), ws.numel())


@pytest.mark.parametrize("k", [16, 64, 260, 516])
def test_an_overflowed_diagonal_gives_a_factor_of_zeros(k, dev):
    """The damping is a share of the diagonal's mean: one infinite entry makes every pivot
    infinite and its row 1 / sqrt of that."""
    from hi2_amd.hessian import inverse_factor

    h = _hessian(k, dev, 5).float()
    h[k // 2, k // 2] = float("inf")
    print(f"overflowed diagonal k={k}", flush=True)
    assert not bool(inverse_factor(h, 0.01).any())
