"""``HessianStats`` on fp16 and fp32 tokens (``hi2x_hessian_accumulate``) against float64: the
edges of the 256-feature tiles, 64-token padding and token splits, values the bf16 planes of
fp32 cannot hold, and the first update's unread sum."""

import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(1, 16), (63, 40), (64, 250), (65, 256), (200, 257), (1000, 272), (129, 1544),
          (4500, 512), (70, 8208)]


def _x(t, k, dtype, dev, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    x = torch.randn(t, k, generator=g, device=dev)
    x[:, ::13] *= 20.0
    x[::7, 1] *= 1e-3
    return x.to(dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32, torch.bfloat16])
@pytest.mark.parametrize("t,k", SHAPES)
def test_against_float64(t, k, dtype, dev):
    from hi2_amd.hessian import HessianStats

    print(f"hessian {dtype} t={t} k={k}", flush=True)
    st = HessianStats(k, dev)
    a, b = _x(t, k, dtype, dev, t + k), _x(t + 3, k, dtype, dev, t * k)
    st.update(a)
    st.update(b)
    x = torch.cat([a, b]).double()
    want, mag = x.T @ x, x.abs().T @ x.abs()
    # every element: products exact (or to 3 x 2^-24 of themselves), then an fp32 sum of n
    # terms in some order: at most (n + 4) 2^-24 of the sum of magnitudes
    bound = (x.shape[0] + 4) * 2.0 ** -24
    assert bool(((st.S.double() - want).abs() <= bound * mag + 1e-30).all())
    assert torch.equal(st.S, st.S.T) and st.n == x.shape[0]


def test_fp32_elements_keep_their_own_precision(dev):
    """Rare tokens 1e5 times the others must not cost the others' products (a scaled fp16 split
    would lose them: its error is relative to a feature's largest token)."""
    from hi2_amd.hessian import HessianStats

    t, k = 512, 64
    x = _x(t, k, torch.float32, dev, 5)
    x[3, 0] = 1e5
    x[9, 1] = -1e5
    st = HessianStats(k, dev)
    st.update(x)
    xd = x.double()
    assert bool(((st.S.double() - xd.T @ xd).abs() <= (t + 4) * 2.0 ** -24
                 * (xd.abs().T @ xd.abs())).all())


@pytest.mark.parametrize("value", [float("inf"), float("nan"), 3.4e38])
@pytest.mark.parametrize("first", [True, False])
def test_fp32_values_beyond_the_planes(value, first, dev):
    """Infinities, NaN and the largest fp32 values, first and later updates."""
    from hi2_amd.hessian import HessianStats

    t, k = 96, 300
    x = _x(t, k, torch.float32, dev, 11)
    st = HessianStats(k, dev)
    if not first:
        st.update(x)
    y = x.clone()
    y[5, 7] = value
    st.update(y)
    s = st.S
    want = (y.double().T @ y.double() + (0 if first else x.double().T @ x.double())).float()
    fin = torch.isfinite(want)
    assert torch.equal(torch.isnan(s), torch.isnan(want))
    assert torch.equal(s[torch.isinf(want)], want[torch.isinf(want)])
    assert torch.allclose(s[fin], want[fin], rtol=1e-4, atol=1e-4 * 400 * t)


def _fp32_kernel(x, dev, s=None):
    """Both triangles of ``x^T x`` (plus ``s``) on the fp32 MFMA (the C entry without a
    workspace)."""
    from hi2_amd import _lib

    s = torch.zeros(x.shape[1], x.shape[1], device=dev) if s is None else s
    _lib.call("hi2x_hessian_syrk", x.device, _lib.ptr(x), 0, x.shape[0], x.shape[1], _lib.ptr(s),
              None, 0)
    return s


# squares that pass the largest fp32 (their planes' products of unlike sign too), and magnitudes
# whose planes cannot hold them; alone and beside their negative, K for both load widths
@pytest.mark.parametrize("value", [2.0 ** 53, 1e20, 1.5e21, 1e22, 7e25, 3e30, 2.0 ** -111, 1e-36,
                                   1e-40])
@pytest.mark.parametrize("pair", [False, True])
@pytest.mark.parametrize("k", [300, 301])
def test_fp32_values_outside_the_planes_range(value, pair, k, dev):
    """They give the bits of fp32 products and sums."""
    from hi2_amd.hessian import HessianStats

    x = _x(96, k, torch.float32, dev, 12)
    x[5, 7] = value
    if pair:
        x[9, 20] = x[9, 7] = -value
    st = HessianStats(k, dev)
    print(f"outside the planes {value} k={k}", flush=True)
    st.update(x)
    want = _fp32_kernel(x, dev)
    nan = torch.isnan(want)
    assert torch.equal(torch.isnan(st.S), nan)
    assert torch.equal(st.S[~nan], want[~nan])


def _integers(t, k, dtype, dev, seed):
    """Tokens whose sums of products are whole numbers below 2^24 for up to 2^22 / 2 tokens."""
    g = torch.Generator(device=dev).manual_seed(seed)
    return torch.randint(-2, 3, (t, k), generator=g, device=dev).to(dtype)


# both sides of each line of the rule, tiles of 128 that are whole and not
@pytest.mark.parametrize("t,k,few", [(64, 48, True), (65, 48, False), (64, 2048, True),
                                     (65, 2048, False), (56, 2049, True), (57, 2049, False),
                                     (34, 2816, True), (4, 2817, False), (3, 2817, True),
                                     (1, 4100, True), (4, 4100, False)])
def test_few_fp32_tokens(t, k, few, dev):
    """Few fp32 tokens run on the fp32 kernel, without scratch and with its bits, first and later
    updates; past them, every element as the planes' bound has it."""
    from hi2_amd import _lib
    from hi2_amd.hessian import HessianStats

    x = _x(t, k, torch.float32, dev, t + k)
    f = _lib.lib().hi2x_hessian_accumulate_workspace_bytes
    assert (f(0, t, k) == 0) == few
    print(f"few fp32 tokens t={t} k={k}", flush=True)
    st = HessianStats(k, dev)
    st.update(x)
    st.update(x[: t // 2])
    if few:
        assert torch.equal(st.S, _fp32_kernel(x[: t // 2], dev, _fp32_kernel(x, dev)))
    x = torch.cat([x, x[: t // 2]]).double()
    bound = (x.shape[0] + 4) * 2.0 ** -24
    assert bool(((st.S.double() - x.T @ x).abs() <= bound * (x.abs().T @ x.abs())).all())


@pytest.mark.parametrize("t", [13, 129, 192, 193])
@pytest.mark.parametrize("k", [250, 1030, 1536])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_split_and_whole_token_ranges(t, k, dtype, dev):
    """Either side of the line between one token range and several: whole numbers, so every
    order of the sums is exact."""
    from hi2_amd.hessian import HessianStats

    x = _integers(t, k, dtype, dev, t + k)
    st = HessianStats(k, dev)
    print(f"token ranges {dtype} t={t} k={k}", flush=True)
    st.update(x)
    st.update(x)
    xd = x.double()
    assert torch.equal(st.S.double(), 2.0 * (xd.T @ xd))


@pytest.mark.parametrize("value", [2.0 ** -110 * (1 + 2.0 ** -23), 1.7e-30, 2.0 ** 53 * (1 - 2.0 ** -24)])
def test_fp32_values_at_the_ends_of_the_planes_range(value, dev):
    """A feature of such magnitudes only, against float64: the bound of the other magnitudes."""
    from hi2_amd.hessian import HessianStats

    t, k = 96, 64
    x = _x(t, k, torch.float32, dev, 13)
    x[:, 3] = value * (1 + 2.0 ** -12) ** torch.arange(t, device=dev) if value < 1 else value
    st = HessianStats(k, dev)
    st.update(x)
    xd = x.double()
    ok = (st.S.double() - xd.T @ xd).abs() <= (t + 4) * 2.0 ** -24 * (xd.abs().T @ xd.abs())
    ok[3, 3] |= value ** 2 < 2.0 ** -126  # the square of the feature is below the normal fp32
    assert bool(ok.all())


@pytest.mark.parametrize("t,k", [(1 << 18, 16), ((1 << 18) + 1, 260), ((1 << 19) + 70, 37)])
@pytest.mark.parametrize("outside", [False, True])
def test_fp32_passes(t, k, outside, dev):
    """More tokens than one pass's planes hold: exact sums, first and later update, also where a
    value outside the planes' range sends one of the passes to the fp32 kernel."""
    from hi2_amd.hessian import HessianStats

    x = _integers(t, k, torch.float32, dev, t + k)
    if outside:
        x[t - 3, 2] = 2.0 ** 60  # its own row and column of the sum are not compared
    st = HessianStats(k, dev)
    print(f"fp32 passes t={t} k={k}", flush=True)
    st.update(x)
    st.update(x[:70])
    xd = x.double()
    want = xd.T @ xd + xd[:70].T @ xd[:70]
    keep = torch.ones(k, dtype=torch.bool, device=dev)
    keep[2] = not outside
    assert torch.equal(st.S.double()[keep][:, keep], want[keep][:, keep])
    assert st.n == t + 70


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("t,k", [((1 << 21) + 1, 24), ((1 << 23) + 70, 16)])
def test_16_bit_passes(t, k, dtype, dev):
    """More tokens than a pass takes (2^23 rows of a 256-feature panel no longer fit 32-bit
    offsets): exact sums, through ``HessianStats`` and for bf16 through the other entries."""
    from hi2_amd import _lib
    from hi2_amd.hessian import HessianStats

    g = torch.Generator(device=dev).manual_seed(k)
    x = torch.randint(-1, 2, (t, k), generator=g, device=dev, dtype=torch.int8).to(dtype)
    st = HessianStats(k, dev)
    print(f"16-bit passes {dtype} t={t} k={k}", flush=True)
    st.update(x)
    want = sum(c.double().T @ c.double() for c in x.split(1 << 20))
    assert torch.equal(st.S.double(), want)
    if dtype == torch.bfloat16:
        ws = _lib.workspace(dev, "hi2x_hessian_workspace_bytes", 2, t, k)
        assert ws.numel() < 2 * k * (1 << 22)  # one pass of the copy, and partial sums
        for name in ("hi2x_hessian_syrk", "hi2x_hessian_syrk_upper"):
            s = torch.zeros(k, k, device=dev)
            _lib.call(name, x.device, _lib.ptr(x), 2, t, k, _lib.ptr(s), _lib.ptr(ws), ws.numel())
            assert torch.equal(s.double().triu(), want.triu())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("t,k", [(500, 1040), (70, 37), (0, 48)])
def test_upper_entry(t, k, dtype, dev):
    """``hi2x_hessian_syrk_upper`` leaves the upper triangle of ``hi2x_hessian_syrk``."""
    from hi2_amd import _lib

    x = _x(max(t, 1), k, dtype, dev, t + k)[:t].contiguous()
    code = 2 if dtype == torch.bfloat16 else 0
    ws = _lib.workspace(dev, "hi2x_hessian_workspace_bytes", code, t, k)
    out = []
    for name in ("hi2x_hessian_syrk", "hi2x_hessian_syrk_upper"):
        s = torch.ones(k, k, device=dev)
        _lib.call(name, x.device, _lib.ptr(x), code, t, k, _lib.ptr(s), _lib.ptr(ws), ws.numel())
        out.append(s.triu())
    assert torch.equal(*out)


def test_fp16_specials(dev):
    """fp16 infinities, NaN and subnormals multiply as their fp32 values do."""
    from hi2_amd.hessian import HessianStats

    t, k = 64, 64
    x = torch.zeros(t, k, dtype=torch.float16, device=dev)
    x[0, 0], x[0, 1], x[1, 2], x[2, 3] = float("inf"), 2.0, float("nan"), 6e-8
    x[2, 4], x[3, 5] = 65504.0, 65504.0
    st = HessianStats(k, dev)
    st.update(x)
    want = x.float().T @ x.float()
    assert torch.equal(torch.isnan(st.S), torch.isnan(want))
    m = ~torch.isnan(want)
    assert torch.equal(st.S[m], want[m])


def test_sum_without_an_update_is_zero(dev):
    from hi2_amd.hessian import HessianStats

    st = HessianStats(48, dev)
    st.update(torch.empty(0, 48, device=dev))
    assert st.n == 0 and not bool(st.S.any())
    had = torch.ones(3, dtype=torch.uint8, device=dev)
    assert not bool(HessianStats(48, dev).transformed(None, had).any())


def test_first_update_that_raises_leaves_the_sum_unmade(dev, monkeypatch):
    """A caller that catches the error and updates again adds to zero, not to unset memory."""
    from hi2_amd import _lib
    from hi2_amd.hessian import HessianStats

    x = _x(64, 48, torch.float32, dev, 5)
    want = HessianStats(48, dev)
    want.update(x)
    st = HessianStats(48, "cuda")

    def fail(*a):
        raise RuntimeError("no workspace")

    with monkeypatch.context() as m:
        m.setattr(_lib, "workspace", fail)
        with pytest.raises(RuntimeError):
            st.update(x)
    assert st.n == 0 and not st._upper_only and st._sum is None
    st.update(x)
    assert torch.equal(st.S, want.S)


def test_the_constructor_refuses(dev):
    """A device that is not there and a sum that does not fit raise in the constructor."""
    from hi2_amd.hessian import HessianStats

    with pytest.raises(RuntimeError):
        HessianStats(16, "cuda:99")
    with pytest.raises(RuntimeError):
        HessianStats(1 << 20, dev)  # 4 TiB
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    st = HessianStats(1024, dev)
    assert torch.cuda.memory_allocated() - before >= 4 << 20 and not bool(st.S.any())
