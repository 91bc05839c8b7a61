"""The convolution kernels that take fp32 operands as three bf16 pieces each: every tile shape, at sizes
around the ends of tiles and of the ranges a tile shape serves, against sums in 64 bits over the exported
rules; operands of any size; and rows and weights that are no finite numbers.

Tolerance: the pieces hold every operand exactly, the products left out are below 1.001 2^-24 of a product with factors in
[1, 2) and of either sign, and the sums of 32 channels are added in fp32, so that one result of m additions is off by at most
about (m + 4) 2^-24 of the sum of the products' magnitudes.  Over a whole output the roundings are of either sign: a
2-norm below sqrt(m / 2) 2^-24 of the result's (partial sums of either sign grow like it), and 2^-23 for the six roundings of a chain, which are not to nearest.  That
bound is below half of what any one of the six products amounts to, which each test makes sure of for its inputs."""
import numpy as np
import pytest

from sparseconvnet_amd import synthetic

pytestmark = pytest.mark.gpu


def _scene(n, seed):
    from hip_path import HipPath
    spatial = 126 if n < 30000 else 1022
    coords = synthetic.room_scene(seed=seed, target=max(n, 2000), spatial=spatial)[:n]
    p = HipPath(3)
    assert p.input_layer(spatial, coords, 0, 0) == len(coords) == n
    return p, spatial


def _reference(rules, x, w):
    """sum over rules (tap, in, out), and the same of the magnitudes; on the GPU, in 64 bits."""
    import torch
    x, w = torch.as_tensor(x).cuda().double(), torch.as_tensor(w).cuda().double()
    y = torch.zeros((len(x), w.shape[-1]), dtype=torch.float64, device="cuda")
    a = torch.zeros_like(y)
    for k in range(w.shape[0]):
        r = torch.as_tensor(rules[k]).cuda().long()
        if len(r):
            y.index_add_(0, r[:, 1], x[r[:, 0]] @ w[k, 0])
            a.index_add_(0, r[:, 1], x[r[:, 0]].abs() @ w[k, 0].abs())
    return y.cpu().numpy(), a.cpu().numpy()


def _pieces(v):
    """The three bf16 pieces of an fp32 array, each as fp32."""
    import torch
    v, out = torch.as_tensor(v), []
    for _ in range(3):
        out.append(v.bfloat16().float())
        v = v - out[-1]
    return [o.numpy() for o in out]


def _two_norm(err, want, additions, products):
    """The 2-norm bound; products: the sum over one pair of pieces instead of the operands (three smallest pairs that count)."""
    limit = ((additions / 2) ** 0.5 + 2) * 2.0 ** -24 * np.linalg.norm(want)
    assert np.linalg.norm(err) <= limit, np.linalg.norm(err) / limit
    for missing in products:
        assert np.linalg.norm(missing) > 2 * limit, "a product left out would pass"


# widths at and beside every number of 16-column blocks; sites around 16, 32, 64 and 128 rows, 1024, and 300 k
@pytest.mark.parametrize("n,cin,cout", [
    (1, 20, 5), (15, 32, 32), (17, 36, 33), (33, 64, 64), (65, 100, 96), (127, 32, 128), (129, 48, 130), (1023, 64, 192),
    (1023, 40, 209), (1023, 224, 224), (1023, 32, 256), (1024, 64, 48), (1024, 52, 80), (1025, 96, 112), (1500, 160, 160),
    (1500, 20, 177), (2000, 44, 200), (2100, 256, 256), (5000, 64, 24), (20011, 32, 64), (33333, 64, 32), (33333, 24, 96),
    (299999, 32, 40), (300001, 32, 17), (300001, 36, 64), (300001, 32, 90), (300001, 64, 128)])
def test_split_operands_against_64_bits(n, cin, cout):
    p, spatial = _scene(n, 9000 + n % 97)
    rng = np.random.default_rng(cin * 1000 + cout)
    x = rng.normal(size=(n, cin)).astype(np.float32)
    x *= np.exp(rng.normal(size=(n, 1))).astype(np.float32)  # rows of different size
    w = (rng.normal(size=(27, 1, cin, cout)) * (2.0 / (cin * 27)) ** 0.5).astype(np.float32)
    got, _ = p.subm_conv(spatial, 3, x, w)
    rules = p.submanifold_rules(spatial, 3)
    want, mag = _reference(rules, x, w)
    err = np.abs(got - want)
    additions = 27 * -(-cin // 32)
    assert (err <= (additions + 4) * 2.0 ** -24 * mag).all(), err.max()
    xp, wp = _pieces(x), _pieces(w)
    _two_norm(err, want, additions, (_reference(rules, xp[a], wp[b])[0] for a, b in ((1, 1), (0, 2), (2, 0))))


@pytest.mark.parametrize("n,cin,cout", [(700, 32, 64), (3000, 24, 32), (3000, 64, 160)])
def test_values_that_are_not_finite_spread_as_the_sum_says(n, cin, cout):
    """An infinity reaches exactly the outputs whose rules read it, with the sign the sum gives; so does a NaN; sums
    past the largest float are infinite; everything else stays as it was.  Weights likewise."""
    p, spatial = _scene(n, 9500 + n)
    rng = np.random.default_rng(n + cout)
    rules = p.submanifold_rules(spatial, 3)

    def check(x, w):
        got, _ = p.subm_conv(spatial, 3, x, w)
        with np.errstate(all="ignore"):
            want = np.zeros((n, cout), np.float64)
            for k in range(27):
                i, o = rules[k][:, 0], rules[k][:, 1]  # (an output occurs once per tap)
                for c in range(cin):
                    want[o] += x[i, c:c + 1].astype(np.float64) * w[k, 0, c][None, :].astype(np.float64)
        assert (np.isnan(got) == np.isnan(want)).all()
        big = np.abs(want) > 3.5e38
        assert big.any() or np.isnan(want).any()
        assert (got[big] == np.sign(want[big]) * np.inf).all()
        rest = np.abs(want) < 3e38
        np.testing.assert_allclose(got[rest], want[rest], rtol=1e-4, atol=1e-5 * min(np.abs(x[np.isfinite(x)]).max(), 1e36))

    x = rng.normal(size=(n, cin)).astype(np.float32)
    w = (rng.normal(size=(27, 1, cin, cout)) * 0.05).astype(np.float32)
    w[:, 0, 3, :7] = 1.0  # a weight whose lower pieces are zero
    a = x.copy()
    a[5, 3], a[n // 2, 7], a[n - 1, 3] = np.inf, np.nan, -np.inf
    check(a, w)
    b = x.copy()
    b[:, 0] = np.where(np.arange(n) % 5 == 0, 3.4e38, 0.0)  # near the largest float: rounding it to bf16 would overflow
    v = w * np.float32(1e-3)
    v[13, 0, 0, :] = 2.0
    check(b, v)
    v = w.copy()
    v[13, 0, 2, 4], v[13, 0, 1, 6] = np.inf, np.nan
    check(x, v)


def _weight_gradient(rules, x, d, cin, cout):
    import torch
    x, d = torch.as_tensor(x).cuda().double(), torch.as_tensor(d).cuda().double()
    w, a = np.zeros((27, 1, cin, cout)), np.zeros((27, 1, cin, cout))
    for k in range(27):
        r = torch.as_tensor(rules[k]).cuda().long()
        if len(r):
            i, o = x[r[:, 0]], d[r[:, 1]]
            w[k, 0], a[k, 0] = (i.t() @ o).cpu().numpy(), (i.abs().t() @ o.abs()).cpu().numpy()
    return w, a


# a tile of 64, 96 or 128 channels per side, one to three of them; sites around a granule, a block of eight and
# the ranges of the shares
@pytest.mark.parametrize("n,cin,cout", [
    (1, 68, 36), (17, 36, 100), (129, 96, 128), (1000, 128, 96), (1025, 160, 64), (2100, 196, 132), (5000, 64, 260),
    (29999, 72, 72), (30001, 64, 64), (30001, 36, 60), (30001, 132, 40), (60011, 64, 96), (300001, 64, 64), (300001, 100, 36)])
def test_weight_gradient_from_split_operands_against_64_bits(n, cin, cout):
    """Sums of m rules, 32 positions at a time from zero, then shares (up to about 300): m / 32 + 300 additions at most."""
    p, spatial = _scene(n, 9700 + n % 89)
    rng = np.random.default_rng(cin * 1000 + cout)
    x = rng.normal(size=(n, cin)).astype(np.float32)
    d = (rng.normal(size=(n, cout)) * np.exp(rng.normal(size=(n, 1)))).astype(np.float32)
    w = np.zeros((27, 1, cin, cout), np.float32)
    p.subm_conv(spatial, 3, x, w)
    got = p.subm_conv_bwd(spatial, 3, x, d, w)[1]
    rules = p.submanifold_rules(spatial, 3)
    want, mag = _weight_gradient(rules, x, d, cin, cout)
    err = np.abs(got.reshape(want.shape) - want)
    assert (err <= (n / 32 + 300) * 2.0 ** -24 * mag).all(), err.max()
    # (positions of a share and shares are summed apart: the 2-norm's additions are those of one share and of one sum over shares)
    xp, dp = _pieces(x), _pieces(d)
    _two_norm(err, want, min(n / 32, 30) + min(n / 128, 300),
              (_weight_gradient(rules, xp[a], dp[b], cin, cout)[0] for a, b in ((1, 1), (0, 2), (2, 0))))


def test_weight_gradient_with_values_that_are_not_finite():
    n, cin, cout = 3000, 100, 64
    p, spatial = _scene(n, 9800)
    rng = np.random.default_rng(9)
    x, d = rng.normal(size=(n, cin)).astype(np.float32), rng.normal(size=(n, cout)).astype(np.float32)
    x[11, 5], x[n - 1, 70] = np.inf, np.nan
    w = np.zeros((27, 1, cin, cout), np.float32)
    p.subm_conv(spatial, 3, x, w)
    got = p.subm_conv_bwd(spatial, 3, x, d, w)[1].reshape(w.shape)
    for k, r in enumerate(p.submanifold_rules(spatial, 3)):
        i, o = x[r[:, 0]].astype(np.float64), d[r[:, 1]].astype(np.float64)
        for c in (4, 5, 6, 70, 99):
            with np.errstate(all="ignore"):
                want = (i[:, c:c + 1] * o).sum(0) if len(r) else np.zeros(cout)
            assert (np.isnan(got[k, 0, c]) == np.isnan(want)).all()
            ok = ~np.isnan(want)
            np.testing.assert_allclose(got[k, 0, c][ok], want[ok], rtol=1e-4, atol=1e-3)


def _rules_of(md):
    from hip_path import HipPath

    class Rules(HipPath):
        def __init__(self):
            self.L, self.dim, self.h = md._L, 3, md._h

        def __del__(self):
            pass
    return Rules()


def _table(kind, n, seed):
    """A layer of `kind` on a room of n sites: (call of its convolution, rules per tap (in, out), input rows, output rows,
    Metadata)."""
    import torch
    import sparseconvnet_amd as scn
    spatial = {"up3": 127, "down3": 127}.get(kind, 126) if n < 30000 else {"up3": 1023, "down3": 1023}.get(kind, 1022)
    coords = synthetic.room_scene(seed=seed, target=max(n + n // 10, 2000), spatial=spatial)[:n]
    t = scn.InputLayer(3, spatial, mode=4)([torch.as_tensor(coords), torch.zeros((n, 1)).cuda()])
    md, size = t.metadata, t.spatial_size
    assert md.getNActive(size) == n
    p = _rules_of(md)
    if kind == "nin":
        rules = [np.stack([np.arange(n)] * 2, 1)]
        return lambda x, w, b: md.networkInNetwork(x, w[0, 0], b, want_macs=False)[0], rules, n, n, md
    if kind.startswith("subm"):
        f = torch.LongTensor([int(kind[4:] or 3)] * 3)

        def conv(*a, **k):
            return md.submanifoldConvolution(size, f, *a, want_macs=False, **k)[0]
        conv(torch.zeros((n, 1)).cuda(), torch.zeros(int(f.prod()), 1, 1, 1).cuda(), None)
        return conv, p.submanifold_rules(size, int(f[0])), n, n, md
    f = 3 if kind.endswith("3") else 2
    fs, two, half = torch.LongTensor([f] * 3), torch.LongTensor([2] * 3), (size - f) // 2 + 1
    md.convolution(size, half, fs, two, torch.zeros((n, 1)).cuda(), torch.zeros(f ** 3, 1, 1, 1).cuda(), None, want_macs=False)
    rules, coarse = p.strided_rules(size, half, f, 2), md.getNActive(half)
    if kind.startswith("down"):
        return lambda *a, **k: md.convolution(size, half, fs, two, *a, want_macs=False, **k)[0], rules, n, coarse, md
    rules = [r[:, ::-1].copy() for r in rules]
    return lambda *a, **k: md.deconvolution(half, size, fs, two, *a, want_macs=False, **k)[0], rules, coarse, n, md


def _close_where_finite(got, want, mag, terms):
    """NaNs where the sum in 64 bits has them, infinities of its sign where it is past the largest float, and elsewhere within
    `terms` additions in fp32 of the sum of magnitudes."""
    import torch
    got = got.double()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    big = want.abs() > 3.5e38
    assert torch.equal(got[big], torch.sign(want[big]) * float("inf"))
    rest = want.abs() < 3e38
    assert rest.any() and not rest.all()
    assert ((got - want).abs()[rest] <= terms * 2.0 ** -24 * mag[rest] + 1e-37).all()


# 512 tiles and more (stored by the tile itself) and fewer (its taps dealt out), 32-, 64- and 128-row tiles, each
# form of the call, tables with and without a row map
@pytest.mark.parametrize("kind,n,cin,cout,pre", [
    ("subm", 900, 64, 96, False), ("subm", 1500, 64, 64, True), ("subm", 33333, 24, 48, False), ("subm", 33333, 36, 160, True),
    ("subm", 70001, 20, 32, False), ("subm", 300001, 32, 40, False), ("subm", 300001, 32, 40, True),
    ("down", 20011, 32, 64, False), ("down", 160001, 32, 64, False), ("up", 33333, 64, 48, False), ("up", 3001, 64, 48, True)])
def test_values_that_are_not_finite_in_every_form_of_the_call(kind, n, cin, cout, pre):
    import torch
    conv, rules, rows_in, rows_out, _ = _table(kind, n, 9600 + n % 91)
    taps = len(rules)
    g = torch.Generator().manual_seed(n + cout)

    def normal(*shape):
        return torch.randn(*shape, generator=g).cuda()

    def bn(c):
        return normal(c) * 0.3, torch.rand(c, generator=g).cuda() + 0.5, torch.rand(c, generator=g).cuda() + 0.5, normal(c) * 0.3, 1e-4, 0.2

    def normalise(y, mag, p):
        mean, var, gamma, beta, eps, leak = p
        sc = (gamma.double() / torch.sqrt(var.double() + eps))
        y, mag = (y - mean.double()) * sc + beta.double(), mag * sc + (mean.abs().double() * sc + beta.abs().double())
        return torch.where(y > 0, y, leak * y), mag
    w, bias, front, post, second = normal(taps, 1, cin, cout) * 0.05, normal(cout), bn(cin) if pre else None, bn(cout), bn(cout)
    for case in ("rows", "weights", "overflow"):
        x, v = normal(rows_in, cin), w.clone()
        if case == "rows":
            x[5, 3], x[rows_in // 2, 7], x[rows_in - 1, 3] = float("inf"), float("nan"), float("-inf")
        elif case == "weights":
            v[taps // 2, 0, 2, 4], v[taps - 1, 0, 1, 6] = float("inf"), float("nan")
        else:
            v *= 1e-3
            x[::5, 0], v[taps // 2, 0, 0] = 1e38, 16.0
        f, fm = x.double(), x.double().abs()
        if pre:
            f, fm = normalise(f, fm, front)
        want = bias.double().expand(rows_out, -1).clone()
        mag = want.abs()
        for k, r in enumerate(rules):
            r = torch.as_tensor(r).cuda().long()
            want.index_add_(0, r[:, 1], f[r[:, 0]] @ v[k, 0].double())
            mag.index_add_(0, r[:, 1], fm[r[:, 0]] @ v[k, 0].double().abs())
        terms = taps * cin + 16
        _close_where_finite(conv(x, v, bias, bn=front), want, mag, terms)
        wide, other = torch.full((rows_out, cout + 24), 7.0).cuda(), torch.full((rows_out, cout + 12), 5.0).cuda()
        conv(x, v, bias, bn=front, post=post, out=wide[:, 8:8 + cout], second=(second, other[:, 4:4 + cout]))
        assert (wide[:, :8] == 7.0).all() and (wide[:, 8 + cout:] == 7.0).all()
        assert (other[:, :4] == 5.0).all() and (other[:, 4 + cout:] == 5.0).all()
        raw = torch.where(want.abs() > 3.5e38, torch.sign(want) * float("inf"), want)  # as the fp32 sum in front has it
        for got, p in ((wide[:, 8:8 + cout], post), (other[:, 4:4 + cout], second)):
            y, m = normalise(raw, mag, p)
            _close_where_finite(got, y, m, terms)


def test_rows_of_nans_cost_a_few_times_an_ordinary_pass():
    """Every tile computed twice, the second time on fp32 matrix instructions with nothing prefetched: 2 times an ordinary
    pass at 64 -> 64, 3 at 128 -> 128.  The bound tells that from a loop over single values (60 and 136 times)."""
    import torch
    import sparseconvnet_amd as scn
    coords = synthetic.room_scene(seed=9650, target=20011, spatial=126)
    t = scn.InputLayer(3, 126, mode=4)([torch.as_tensor(coords), torch.zeros((len(coords), 1)).cuda()])
    for planes in (64, 128):
        conv = scn.SubmanifoldConvolution(3, planes, planes, 3, False).cuda()

        def time(x):
            best = float("inf")
            for _ in range(4):
                a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                a.record()
                with torch.no_grad():
                    y = conv(scn.SparseConvNetTensor(x, t.metadata, t.spatial_size)).features
                b.record()
                b.synchronize()
                best = min(best, a.elapsed_time(b))
            return best, y
        x = torch.randn(len(coords), planes).cuda()
        ordinary, _ = time(x)
        x[:, 3] = float("nan")
        nans, y = time(x)
        assert torch.isnan(y).all()
        assert nans < 15 * ordinary, (nans, ordinary)


# (kind of layer, sites of its fine level, planes, what the kernel that runs says of itself)
@pytest.mark.parametrize("kind,n,cin,cout,says", [
    # one rule per position: dealt out only while a tile has several taps; 32-row tiles up to 24 k
    ("up", 301, 96, 96, ("split ", "gw=1", "split=8")), ("up", 1535, 64, 256, ("gw=2", "split=8")),
    ("up", 1537, 64, 256, ("gw=2", "split=1")), ("up", 20011, 64, 256, ("gw=2", "split=1")), ("up", 24001, 64, 96, ("gw=2 ", "split=1")),
    ("up", 6143, 96, 32, ("ncbw=2 wc=1", "split=8")), ("up", 6145, 96, 32, ("ncbw=2 wc=1", "split=1")),
    # eight taps of 32 planes: dealt out on small levels only
    ("down", 4001, 32, 64, ("gw=1", "split=8")), ("down", 12001, 32, 64, ("gw=1", "split=3")), ("down", 40011, 32, 64, ("gw=1", "split=1")),
    # parts of three iterations and more
    ("subm", 2000, 32, 64, ("gw=2", "split=9")), ("subm", 2000, 64, 64, ("gw=2", "split=18")), ("subm", 700, 64, 24, ("split=27",)),
    # filter 3 stride 2, fine side: taps of one parity per tile
    ("up3", 8001, 64, 64, ("gw=2", "split ")), ("up3", 20011, 32, 64, ("split=1",)), ("up3", 700, 64, 64, ("gw=1", "split=18")),
    ("down3", 5001, 64, 96, ("split ",)),
    # 1x1: a tile is one to eight iterations
    ("nin", 1023, 64, 256, ("wc=4 gw=2",)), ("nin", 1024, 64, 256, ("wc=4 gw=2",)), ("nin", 5000, 96, 160, ("gw=1",)),
    ("nin", 23999, 160, 128, ("gw=2",)), ("nin", 24000, 160, 128, ("gw=4",)), ("nin", 5000, 320, 160, ("gw=2",)),
    # up to 32 -> 16 planes at large levels and many taps onto up to 32: the fp32 kernels
    ("subm", 199999, 32, 16, ("split ",)), ("subm", 200000, 32, 16, ("resident",)), ("subm", 299999, 20, 12, ("split ",)),
    ("subm", 300000, 20, 12, ("resident",)), ("subm5", 3000, 64, 32, ("rows",)), ("subm5", 3000, 64, 40, ("split ",)),
    ("down", 12001, 24, 16, ("resident",)), ("down", 90001, 24, 16, ("split ", "split=1")), ("down", 4001, 24, 20, ("split ", "split=1"))])
def test_kernel_and_shares_by_size(kind, n, cin, cout, says):
    import torch
    conv, rules, rows_in, rows_out, md = _table(kind, n, 9700 + n % 83)
    g = torch.Generator().manual_seed(n + cin)
    x, w = torch.randn(rows_in, cin, generator=g).cuda(), torch.randn(len(rules), 1, cin, cout, generator=g).cuda()
    bias = torch.randn(cout, generator=g).cuda()
    got = conv(x, w, bias)
    kernel = md._L.scn_md_last_conv_kernel(md._h).decode()
    assert all(part in kernel + " " for part in says), kernel
    want = bias.double().expand(rows_out, -1).clone()
    mag = want.abs()
    for k, r in enumerate(rules):
        r = torch.as_tensor(r).cuda().long()
        want.index_add_(0, r[:, 1], x[r[:, 0]].double() @ w[k, 0].double())
        mag.index_add_(0, r[:, 1], x[r[:, 0]].double().abs() @ w[k, 0].double().abs())
    # the fp32 kernels add products one by one
    additions = len(rules) * (-(-cin // 32) if kernel.startswith("split") else cin) + 28
    assert ((got.double() - want).abs() <= additions * 2.0 ** -24 * mag).all()


@pytest.mark.parametrize("n,cin,cout", [(200000, 16, 32), (199999, 16, 32), (20011, 24, 64), (3000, 96, 36)])
def test_input_gradients_whichever_kernel_takes_them(n, cin, cout):
    """The packing of k_conv_split reads the forward weights transposed; the others get a transposed copy."""
    import torch
    p, spatial = _scene(n, 9800 + n % 61)
    rng = np.random.default_rng(n + cin)
    d = rng.normal(size=(n, cout)).astype(np.float32)
    w = (rng.normal(size=(27, 1, cin, cout)) * 0.1).astype(np.float32)
    got = p.subm_conv_bwd(spatial, 3, np.zeros((n, cin), np.float32), d, w)[0]
    rules = [r[:, ::-1].copy() for r in p.submanifold_rules(spatial, 3)]
    want, mag = _reference(rules, d, np.ascontiguousarray(w.transpose(0, 1, 3, 2)))
    assert (np.abs(got - want) <= (27 * cout + 4) * 2.0 ** -24 * mag).all()


def _hard_factors(n, seed):
    """fp32 numbers in [1, 2): those whose bits below the first eight are all set or just over half, and any."""
    bits = np.random.default_rng(seed).integers(0x3F800000, 0x40000000, n, dtype=np.uint32)
    bits[:8] = [0x3F80FF7F, 0x3F80FF80, 0x3F807FFF, 0x3F808001, 0x3F807F7F, 0x3FFFFFFF, 0x3FFF7FFF, 0x3F817F80]
    return bits.view(np.float32)


def test_single_products():
    """What the six products leave out is at most 1.001 2^-24 of a product with factors in [1, 2), and the sum of the six is
    rounded to 24 bits, not to nearest: 2^-23 of the result."""
    p, spatial = _scene(3000, 9900)
    u, v = _hard_factors(3000, 1), _hard_factors(128, 2)
    x, w = np.zeros((3000, 32), np.float32), np.zeros((27, 1, 32, 128), np.float32)
    x[:, 5], w[13, 0, 5] = u, v
    got, _ = p.subm_conv(spatial, 3, x, w)
    want = u[:, None].astype(np.float64) * v[None].astype(np.float64)
    assert (np.abs(got - want) <= 3.1 * 2.0 ** -24 * want).all(), (np.abs(got - want) / want).max() * 2.0 ** 24
    x, d, w = np.zeros((3000, 128), np.float32), np.zeros((3000, 128), np.float32), np.zeros((27, 1, 128, 128), np.float32)
    x[7], d[7] = u[:128], v
    got = p.subm_conv_bwd(spatial, 3, x, d, w)[1].reshape(27, 128, 128)
    want = want[:128]
    assert (np.abs(got[13] - want) <= 3.1 * 2.0 ** -24 * want).all(), (np.abs(got[13] - want) / want).max() * 2.0 ** 24
    assert (got[:13] == 0).all() and (got[14:] == 0).all()


def test_weights_near_the_largest_float():
    """Weights that no bf16 rounds, an infinity and a NaN beside them: packed whole."""
    p, spatial = _scene(3000, 9901)
    big = np.array([3.3962e38, -3.4028234e38, 3.39e38, np.inf, -np.inf, np.nan, 1e38, 1.0], np.float32)
    x, w = np.zeros((3000, 32), np.float32), np.zeros((27, 1, 32, 8), np.float32)
    x[:, 9], w[13, 0, 9] = np.linspace(0.25, 0.99, 3000), big
    got, _ = p.subm_conv(spatial, 3, x, w)
    want = (x[:, 9:10] * big[None]).astype(np.float32)
    np.testing.assert_allclose(got, want, rtol=2.0 ** -22)


@pytest.mark.parametrize("ex,ew", [(-112, 60), (-126, 60), (-140, 80), (60, -112), (60, -126), (80, -140), (-100, -38), (-126, 0),
                                   (100, -100), (110, -30), (50, 20)])
def test_operands_of_any_size(ex, ew):
    """Rows of 2^ex and weights (output gradients) of 2^ew: as exact as any others, down to numbers that fp32 holds with fewer bits
    and past 2^104, where the pieces end.  Beside the bound of ordinary operands, each part of a sum that is stored by itself (a
    tile's taps are dealt out over up to 27 workgroups, positions over up to 200 shares) may be off by half of the smallest
    number, 2^-150."""
    p, spatial = _scene(2000, 9910)
    rng = np.random.default_rng(abs(ex * 1000 + ew))

    def normal(e, *shape):
        return np.ldexp(np.clip(rng.normal(size=shape), -4, 4), e).astype(np.float32)
    for cin, cout in ((32, 64), (96, 64)):
        x, w, d = normal(ex, 2000, cin), normal(ew, 27, 1, cin, cout), normal(ew, 2000, cout)
        got, _ = p.subm_conv(spatial, 3, x, w)
        rules = p.submanifold_rules(spatial, 3)
        want, mag = _reference(rules, x, w)
        assert np.linalg.norm(want) > 0
        err = np.abs(got - want)
        assert (err <= (27 * -(-cin // 32) + 4) * 2.0 ** -24 * mag + 27 * 2.0 ** -150).all(), (err / mag.max()).max()
        got = p.subm_conv_bwd(spatial, 3, x, d, w)[1].reshape(w.shape)
        want, mag = _weight_gradient(rules, x, d, cin, cout)
        err = np.abs(got - want)
        assert (err <= (2000 / 32 + 200) * 2.0 ** -24 * mag + 200 * 2.0 ** -150).all(), (err / mag.max()).max()


# one tap, transposed tables (the staged kernel up to 300 k sites where they have many taps), more than 32 taps (not staged),
# sides that leave much of a tile empty
@pytest.mark.parametrize("kind,n,cin,cout", [
    ("nin", 400003, 64, 96), ("nin", 31, 36, 36), ("nin", 40001, 192, 100), ("up", 60001, 96, 64), ("up", 299999, 64, 64),
    ("up", 300000, 64, 64), ("up", 300000, 128, 128), ("up3", 20011, 96, 64), ("up3", 300001, 64, 96), ("down", 160001, 64, 96), ("down3", 30001, 64, 96),
    ("subm", 60011, 36, 48), ("subm", 299999, 48, 96), ("subm", 300000, 48, 96), ("subm5", 3001, 64, 96), ("subm5", 1000, 128, 128)])
def test_weight_gradient_of_every_kind_of_table(kind, n, cin, cout):
    """Within as many additions in fp32 as a tap has rules, of the sum of magnitudes, in whatever order (the fp32 kernels add them one
    by one within a share), and in the 2-norm as the sums of either sign are (see above)."""
    import torch
    _, rules, rows_in, rows_out, md = _table(kind, n, 9900 + n % 79)
    g = torch.Generator().manual_seed(n + cin)
    x, d = torch.randn(rows_in, cin, generator=g).cuda(), torch.randn(rows_out, cout, generator=g).cuda()
    w = torch.zeros(len(rules), 1, cin, cout).cuda()
    two, size = torch.LongTensor([2] * 3), torch.LongTensor([{"up3": 127, "down3": 127}.get(kind, 126) if n < 30000 else
                                                             {"up3": 1023, "down3": 1023}.get(kind, 1022)] * 3)
    f = torch.LongTensor([round(len(rules) ** (1 / 3))] * 3)
    half = (size - f) // 2 + 1
    if kind == "nin":
        got = md.networkInNetworkBackward(x, d, w[0, 0], False)[1][None]
    elif kind.startswith("subm"):
        got = md.submanifoldConvolutionBackward(size, f, x, d, w, False)[1]
    elif kind.startswith("down"):
        got = md.convolutionBackward(size, half, f, two, x, d, w, False)[1]
    else:
        got = md.deconvolutionBackward(half, size, f, two, x, d, w, False)[1]
    got = got.reshape(len(rules), cin, cout).double()
    error = total = 0.0
    for k, r in enumerate(rules):
        r = torch.as_tensor(r).cuda().long()
        if not len(r):
            assert (got[k] == 0).all()
            continue
        a, b = x[r[:, 0]].double(), d[r[:, 1]].double()
        want, mag = a.t().contiguous() @ b, a.abs().t().contiguous() @ b.abs()
        err = (got[k] - want).abs()
        assert (err <= (len(r) + 4) * 2.0 ** -24 * mag).all(), k
        error, total = error + float(err.norm()) ** 2, total + float(want.norm()) ** 2
    assert error ** 0.5 <= ((min(n, 4096) / 2) ** 0.5 + 2) * 2.0 ** -24 * total ** 0.5
