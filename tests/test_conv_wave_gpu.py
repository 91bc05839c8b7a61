"""The split-operand kernel of up to 48 output planes in which a wavefront owns its rows (k_conv_wave): every form of its
dispatch, at sizes around granules, workgroups and the ends of its ranges, against sums in 64 bits over the exported rules.

Tolerance, as for the other split-operand kernels: sums of a chain of six products of up to 32 channels are added in fp32, one per
(tap, 32 channels), two taps of up to 16 channels together, so that one result is off by at most (m + 4) 2^-24 of the sum of the
products' magnitudes, m the number of those additions; four wavefronts that share a row's taps add three."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,n,cin,cout", [
    # one wavefront, a ragged granule, a granule, one more, a workgroup and one more
    ("subm", 1, 16, 16), ("subm", 15, 8, 8), ("subm", 16, 32, 24), ("subm", 17, 12, 20), ("subm", 63, 16, 32), ("subm", 65, 20, 17),
    # taps dealt over four wavefronts of one granule, of two, and not dealt
    ("subm", 1003, 96, 32), ("subm", 23999, 16, 8), ("subm", 24000, 32, 32), ("subm", 24001, 28, 12), ("subm", 100003, 64, 24),
    ("subm", 299999, 16, 16), ("subm", 300001, 24, 20), ("subm", 600001, 12, 28),
    # eight taps and one rule per position; one tap
    ("down", 301, 16, 32), ("down", 20011, 32, 32), ("down", 120007, 48, 16), ("up", 77, 64, 32), ("up", 20011, 48, 32),
    ("up", 25001, 16, 8), ("up", 150001, 64, 16), ("nin", 5, 16, 16), ("nin", 5003, 96, 32), ("nin", 25001, 24, 16),
    # 33 to 48 output planes: every tile, ragged last column groups, fewer iterations than wavefronts
    ("subm", 7, 20, 33), ("subm", 499, 128, 48), ("subm", 500, 160, 40), ("subm", 2501, 96, 48), ("subm", 9999, 64, 36),
    ("subm", 10001, 48, 48), ("subm", 39999, 24, 36), ("down", 900, 192, 48), ("down", 9003, 32, 40), ("down", 60011, 100, 48),
    ("up", 300, 192, 48), ("up", 2003, 64, 48), ("up", 24001, 160, 40), ("up", 44001, 64, 44), ("nin", 77, 224, 48),
    ("nin", 3001, 128, 34), ("nin", 24999, 96, 40)])
@pytest.mark.parametrize("form", ["plain", "normalised"])
def test_rows_owned_by_a_wavefront(kind, n, cin, cout, form):
    import torch
    from test_conv_split_gpu import _table
    conv, rules, rows_in, rows_out, md = _table(kind, n, 8100 + n % 89)
    g = torch.Generator().manual_seed(n + cout)

    def normal(*shape):
        return torch.randn(*shape, generator=g).cuda()

    def bn(c):
        return normal(c) * 0.3, torch.rand(c, generator=g).cuda() + 0.5, torch.rand(c, generator=g).cuda() + 0.5, normal(c) * 0.3, 1e-4, 0.2

    def normalise(y, p):
        mean, var, gamma, beta, eps, leak = p
        y = (y - mean.double()) * (gamma.double() / torch.sqrt(var.double() + eps)) + beta.double()
        return torch.where(y > 0, y, leak * y)
    x, w, bias = normal(rows_in, cin), normal(len(rules), 1, cin, cout) * 0.1, normal(cout)
    x[:, cin // 2] *= 1e-30  # small numbers keep their bits
    front, post = (bn(cin), bn(cout)) if form == "normalised" and kind != "nin" else (None, None)
    f = x.double() if front is None else normalise(x.double(), front)
    want = bias.double().expand(rows_out, -1).clone()
    mag = want.abs()
    for k, r in enumerate(rules):
        r = torch.as_tensor(r).cuda().long()
        want.index_add_(0, r[:, 1], f[r[:, 0]] @ w[k, 0].double())
        mag.index_add_(0, r[:, 1], f[r[:, 0]].abs() @ w[k, 0].double().abs())
    additions = len(rules) * -(-cin // 32) + 3 + 1
    if front is None:
        got = conv(x, w, bias)
        assert ((got.double() - want).abs() <= (additions + 4) * 2.0 ** -24 * mag).all()
    else:  # the folded scale and shift round a normalised value by 4 2^-24 of its terms, here and behind the sum
        wide = torch.full((rows_out, cout + 8), 7.0).cuda()
        conv(x, w, bias, bn=front, post=post, out=wide[:, 4:4 + cout])
        assert (wide[:, :4] == 7.0).all() and (wide[:, 4 + cout:] == 7.0).all()
        terms = x.double().abs() + front[0].double().abs()
        sc = front[2].double() / torch.sqrt(front[1].double() + front[4])
        big = bias.double().abs().expand(rows_out, -1).clone()
        for k, r in enumerate(rules):
            r = torch.as_tensor(r).cuda().long()
            big.index_add_(0, r[:, 1], (terms[r[:, 0]] * sc + front[3].double().abs()) @ w[k, 0].double().abs())
        psc = post[2].double() / torch.sqrt(post[1].double() + post[4])
        bound = ((additions + 4) * mag + 4 * big) * psc + 4 * ((want.abs() + post[0].double().abs()) * psc + post[3].double().abs())
        assert ((wide[:, 4:4 + cout].double() - normalise(want, post)).abs() <= 2.0 ** -24 * bound).all()
    kernel = md._L.scn_md_last_conv_kernel(md._h).decode()
    assert "split wave" in kernel, kernel


@pytest.mark.parametrize("kind,n,cin,cout", [("subm", 3001, 16, 16), ("subm", 3001, 32, 24), ("subm", 60001, 64, 16),
                                             ("subm", 610001, 16, 32), ("up", 30011, 48, 32), ("down", 3001, 12, 20),
                                             ("subm", 301, 64, 48), ("subm", 3001, 96, 40), ("up", 8001, 64, 48)])
def test_values_that_are_not_finite(kind, n, cin, cout):
    """Exactly the outputs whose rules read an infinity or a NaN are not finite, rows and weights alike."""
    import torch
    from test_conv_split_gpu import _table, _close_where_finite
    conv, rules, rows_in, rows_out, md = _table(kind, n, 8200 + n % 89)
    g = torch.Generator().manual_seed(n + cout)
    w = torch.randn(len(rules), 1, cin, cout, generator=g).cuda() * 0.1
    for case in ("rows", "weights", "overflow"):
        x, v = torch.randn(rows_in, cin, generator=g).cuda(), w.clone()
        if case == "rows":
            x[5, 3], x[rows_in // 2, 7], x[rows_in - 1, 3] = float("inf"), float("nan"), float("-inf")
        elif case == "weights":
            v[len(rules) // 2, 0, 2, 4], v[len(rules) - 1, 0, 1, 6] = float("inf"), float("nan")
        else:
            v *= 1e-3
            x[::5, 0], v[len(rules) // 2, 0, 0] = 1e38, 16.0
        want = torch.zeros(rows_out, cout, dtype=torch.float64, device="cuda")
        mag = want.clone()
        for k, r in enumerate(rules):
            r = torch.as_tensor(r).cuda().long()
            want.index_add_(0, r[:, 1], x[r[:, 0]].double() @ v[k, 0].double())
            mag.index_add_(0, r[:, 1], x[r[:, 0]].double().abs() @ v[k, 0].double().abs())
        _close_where_finite(conv(x, v, torch.zeros(cout).cuda()), want, mag, len(rules) * cin + 16)


@pytest.mark.parametrize("kind,n,cin,cout", [("subm", 3001, 16, 16), ("subm", 30001, 12, 24), ("subm", 3001, 64, 24), ("subm", 60001, 48, 16),
                                             ("down", 3001, 16, 20), ("up", 30011, 48, 32), ("subm", 3001, 96, 40), ("up", 8001, 64, 48)])
def test_values_that_are_not_finite_behind_a_batch_norm(kind, n, cin, cout):
    """The same with a batch norm in the gather, which the second computation applies as well, one behind the sums and a second output."""
    import torch
    from test_conv_split_gpu import _table, test_values_that_are_not_finite_in_every_form_of_the_call as every_form
    every_form(kind, n, cin, cout, True)
    conv, rules, rows_in, rows_out, md = _table(kind, n, 9600 + n % 91)  # the table it used
    front = (torch.zeros(cin).cuda(), torch.ones(cin).cuda(), torch.ones(cin).cuda(), torch.zeros(cin).cuda(), 1e-4, 0.2)
    conv(torch.zeros(rows_in, cin).cuda(), torch.zeros(len(rules), 1, cin, cout).cuda(), torch.zeros(cout).cuda(), bn=front)
    kernel = md._L.scn_md_last_conv_kernel(md._h).decode()
    assert "split wave" in kernel and "pre=1" in kernel, kernel


@pytest.mark.parametrize("kind,n,cin,cout", [
    # the gradient's sums run over the layer's output planes and onto its input planes: two taps of up to 16 planes together, slabs of 32,
    # more than 32 planes
    ("subm", 17, 8, 16), ("subm", 3001, 16, 16), ("subm", 3001, 12, 8), ("subm", 60001, 20, 12), ("subm", 3001, 32, 64), ("subm", 24001, 24, 48),
    ("subm", 2501, 48, 40), ("down", 20011, 20, 16), ("down", 20011, 16, 32), ("down", 3001, 48, 64), ("up", 20011, 32, 16),
    ("up", 20011, 24, 48), ("up", 20011, 40, 64), ("nin", 5003, 16, 96), ("nin", 25001, 24, 12), ("nin", 3001, 36, 128)])
def test_input_gradients(kind, n, cin, cout):
    """Weights packed transposed, those of a submanifold convolution with the taps in reverse order."""
    import torch
    from test_conv_split_gpu import _table, _rules_of
    conv, rules, rows_in, rows_out, md = _table(kind, n, 8500 + n % 89)
    g = torch.Generator().manual_seed(n + cin)
    d, w = torch.randn(rows_out, cout, generator=g).cuda(), torch.randn(len(rules), 1, cin, cout, generator=g).cuda() * 0.1
    conv(torch.zeros(rows_in, cin).cuda(), w, torch.zeros(cout).cuda())
    p, size = _rules_of(md), 126 if n < 30000 else 1022
    x, d_out, weight = torch.zeros(rows_in, cin).numpy(), d.cpu().numpy(), w.cpu().numpy()
    if kind == "subm":
        got = p.subm_conv_bwd(size, 3, x, d_out, weight)[0]
    elif kind == "down":
        got = p.conv_bwd(size, size // 2, 2, 2, x, d_out, weight)[0]
    elif kind == "up":
        got = p.deconv_bwd(size // 2, size, 2, 2, x, d_out, weight)[0]
    else:
        got = p.nin_bwd(x, d_out, weight[0, 0])[0]
    kernel = md._L.scn_md_last_conv_kernel(md._h).decode()
    assert "split wave" in kernel and ("pair=1" in kernel) == (cout <= 16), kernel
    want = torch.zeros(rows_in, cin, dtype=torch.float64, device="cuda")
    mag = want.clone()
    for k, r in enumerate(rules):
        r = torch.as_tensor(r).cuda().long()
        want.index_add_(0, r[:, 0], d[r[:, 1]].double() @ w[k, 0].double().t().contiguous())
        mag.index_add_(0, r[:, 0], d[r[:, 1]].double().abs() @ w[k, 0].double().abs().t().contiguous())
    additions = len(rules) * -(-cout // 32) + 3
    assert ((torch.as_tensor(got).cuda().double() - want).abs() <= (additions + 4) * 2.0 ** -24 * mag).all()


# left to k_conv_rows: large levels of 64 and more planes, wide inputs on small ones
BF16_ROWS = {("subm", 260001, 64, 64), ("subm", 40001, 64, 72), ("subm", 10001, 192, 112), ("subm", 2999, 256, 128)}


@pytest.mark.parametrize("kind,n,cin,cout", [
    ("subm", 1, 32, 16), ("subm", 17, 64, 32), ("subm", 7999, 96, 64), ("subm", 8001, 32, 40), ("subm", 19999, 32, 32),
    ("subm", 20001, 64, 24), ("subm", 300001, 32, 32), ("subm", 700001, 32, 20), ("subm", 2999, 256, 128), ("subm", 3001, 128, 100),
    ("subm", 39999, 96, 96), ("subm", 100001, 64, 128), ("subm", 259999, 32, 64), ("subm", 260001, 64, 64), ("subm", 40001, 64, 72),
    ("subm", 10001, 192, 112), ("down", 900, 64, 96), ("down", 60011, 96, 128), ("down", 500001, 32, 32), ("up", 301, 64, 64),
    ("up", 20011, 128, 96), ("up", 120011, 64, 32), ("nin", 77, 96, 128), ("nin", 44999, 32, 64), ("nin", 120001, 64, 32)])
@pytest.mark.parametrize("form", ["plain", "normalised"])
def test_bf16_operands(kind, n, cin, cout, form):
    """Operands rounded to bf16, products exact, added in fp32 by a unit that need not round to nearest: one result is off by at most
    an ulp, 2^-23, per addition of the sum of the products' magnitudes; a normalised row's value may be rounded from the neighbouring
    fp32 number, an ulp of bf16 (2^-7) away.  That needs a value within some 4 2^-24 of its terms of the middle between two bf16 numbers,
    which one in 2^13 is: the 2-norm of all results is off by 2^-8 / 2^6.5, twice that for values smaller than their terms."""
    import torch
    from test_conv_split_gpu import _table
    conv, rules, rows_in, rows_out, md = _table(kind, n, 8300 + n % 89)
    md.setBf16(True)
    g = torch.Generator().manual_seed(n + cout)
    x, w = torch.randn(rows_in, cin, generator=g).cuda(), (torch.randn(len(rules), 1, cin, cout, generator=g) * 0.1).cuda()
    bias = torch.randn(cout, generator=g).cuda()
    front = None
    f = x
    if form == "normalised" and kind != "nin":
        front = (torch.randn(cin, generator=g).cuda(), torch.rand(cin, generator=g).cuda() + 0.5, torch.rand(cin, generator=g).cuda() + 0.5,
                 torch.randn(cin, generator=g).cuda() + 1.0, 1e-4, 0.2)
        f = (x.double() - front[0]) * (front[2].double() / torch.sqrt(front[1].double() + front[4])) + front[3]
        f = torch.where(f > 0, f, 0.2 * f).float()
    f, wr = f.bfloat16().double(), w.bfloat16().double()
    want = bias.double().expand(rows_out, -1).clone()
    mag = want.abs()
    for k, r in enumerate(rules):
        r = torch.as_tensor(r).cuda().long()
        want.index_add_(0, r[:, 1], f[r[:, 0]] @ wr[k, 0])
        mag.index_add_(0, r[:, 1], f[r[:, 0]].abs() @ wr[k, 0].abs())
    got = conv(x, w, bias) if front is None else conv(x, w, bias, bn=front)
    bound = (len(rules) * cin + 8) * 2.0 ** -23 + (0 if front is None else 2.0 ** -7)
    assert ((got.double() - want).abs() <= bound * mag + 1e-30).all()
    if rows_out >= 1000:  # enough results for a share of them
        assert (got.double() - want).norm() <= 2.0 ** -13.5 * want.norm(), float((got.double() - want).norm() / want.norm())
    kernel = md._L.scn_md_last_conv_kernel(md._h).decode()
    assert ("rows-bf16" if (kind, n, cin, cout) in BF16_ROWS else "wave-bf16") in kernel, kernel


@pytest.mark.parametrize("n,cin,cout", [(1500, 128, 64), (3001, 128, 64), (6001, 128, 128), (12001, 128, 64), (12001, 64, 64)])
def test_bf16_sums_of_small_levels(n, cin, cout):
    """Four wavefronts take a row's R (tap, 32 channels) products in turn and add them up by fp32 adds, R / 4 each.  Of terms of either sign
    the partial sums grow like the square root of their number: off by sqrt(0.18 R / 8) 2^-24 of the result (2-norm; 0.18: the mean square of
    a rounding error over numbers whose logarithm is uniform), and by sqrt(1.5) 2^-24 from the 32 products of an instruction, which are not
    rounded to nearest.  The bound is 1.1 times that; one chain of instructions per wavefront is 1.25 to 1.4 times as far off."""
    import torch
    from test_conv_split_gpu import _table
    conv, rules, rows_in, rows_out, md = _table("subm", n, 8300 + n % 89)
    md.setBf16(True)
    g = torch.Generator().manual_seed(n + cin)
    x, w = torch.randn(rows_in, cin, generator=g).cuda(), (torch.randn(len(rules), 1, cin, cout, generator=g) * 0.1).cuda()
    got = conv(x, w, torch.zeros(cout).cuda())
    kernel = md._L.scn_md_last_conv_kernel(md._h).decode()
    assert "wave-bf16" in kernel, kernel
    want = torch.zeros(rows_out, cout, dtype=torch.float64, device="cuda")
    for k, r in enumerate(rules):
        r = torch.as_tensor(r).cuda().long()
        want.index_add_(0, r[:, 1], x[r[:, 0]].bfloat16().double() @ w[k, 0].bfloat16().double())
    products = sum(len(r) for r in rules) / rows_out * cin / 32
    limit = 1.1 * (0.18 * products / 8 + 1.5) ** 0.5 * 2.0 ** -24
    assert (got.double() - want).norm() <= limit * want.norm(), float((got.double() - want).norm() / want.norm()) / limit


@pytest.mark.parametrize("kind,n,cin,cout,says", [
    # many (tap, 32 channels) products per row on small levels: k_conv_rows deals them over workgroups
    ("subm", 64, 64, 64, "wave-bf16"), ("subm", 200, 96, 96, "rows-bf16"), ("subm", 501, 96, 24, "wave-bf16"),
    ("subm", 599, 128, 96, "rows-bf16"), ("subm", 601, 128, 96, "wave-bf16"), ("subm", 999, 160, 64, "rows-bf16"),
    ("subm", 1001, 160, 64, "wave-bf16"), ("subm", 4199, 256, 64, "rows-bf16"), ("subm", 4201, 256, 64, "wave-bf16"),
    ("subm", 4499, 320, 32, "rows-bf16"), ("down", 300, 320, 64, "rows-bf16"), ("up", 300, 320, 64, "wave-bf16"),
    ("nin", 27999, 64, 96, "wave-bf16"), ("nin", 28001, 64, 96, "rows-bf16"),
    # two granules per wavefront of k_conv_rows: not over tables of few iterations a tile, nor over most of the long tap lists
    ("up", 31001, 256, 128, "ss=2"), ("subm", 31001, 256, 128, "ss=4"), ("subm5", 61001, 64, 96, "ss=2"), ("subm5", 17001, 320, 128, "ss=4"),
    ("nin", 130001, 256, 128, "ss=2"), ("nin", 130001, 256, 96, "ss=4"), ("nin", 70001, 256, 96, "ss=2")])
def test_bf16_kernel_by_size(kind, n, cin, cout, says):
    import torch
    from test_conv_split_gpu import _table
    conv, rules, rows_in, rows_out, md = _table(kind, n, 8300 + n % 89)
    md.setBf16(True)
    g = torch.Generator().manual_seed(n + cin)
    x, w = torch.randn(rows_in, cin, generator=g).cuda(), (torch.randn(len(rules), 1, cin, cout, generator=g) * 0.1).cuda()
    got = conv(x, w, torch.zeros(cout).cuda())
    kernel = md._L.scn_md_last_conv_kernel(md._h).decode()
    assert says in kernel, kernel
    want = torch.zeros(rows_out, cout, dtype=torch.float64, device="cuda")
    mag = want.clone()
    for k, r in enumerate(rules):
        r = torch.as_tensor(r).cuda().long()
        f, v = x[r[:, 0]].bfloat16().double(), w[k, 0].bfloat16().double()
        want.index_add_(0, r[:, 1], f @ v)
        mag.index_add_(0, r[:, 1], f.abs() @ v.abs())
    assert ((got.double() - want).abs() <= (len(rules) * cin + 8) * 2.0 ** -23 * mag + 1e-30).all()


@pytest.mark.parametrize("kind,n,cin,cout,says", [
    ("subm", 1050, 224, 32, "split ncbw"), ("subm", 1999, 128, 32, "split ncbw"), ("subm", 2001, 128, 32, "split wave"),
    ("subm", 1499, 128, 16, "split ncbw"), ("subm", 1501, 128, 16, "split wave"), ("subm", 3699, 192, 24, "split ncbw"),
    ("subm", 3701, 192, 24, "split wave"), ("subm", 5499, 256, 20, "split ncbw"), ("subm", 5501, 256, 20, "split wave"),
    ("subm", 449, 100, 44, "split ncbw"), ("subm", 451, 100, 44, "split wave"), ("subm", 499, 160, 48, "split ncbw"),
    ("subm", 140, 96, 48, "split wave"), ("down", 100, 256, 17, "split ncbw"), ("down", 1500, 256, 17, "split wave"),
    ("down", 33001, 256, 48, "split ncbw")])
def test_kernel_by_length_of_the_chain(kind, n, cin, cout, says):
    """Many (tap, 32 channels) products per row on small levels: k_conv_split deals them over workgroups."""
    import torch
    from test_conv_split_gpu import _table
    conv, rules, rows_in, rows_out, md = _table(kind, n, 8100 + n % 89)
    g = torch.Generator().manual_seed(n + cout)
    x, w = torch.randn(rows_in, cin, generator=g).cuda(), (torch.randn(len(rules), 1, cin, cout, generator=g) * 0.1).cuda()
    got = conv(x, w, torch.zeros(cout).cuda())
    kernel = md._L.scn_md_last_conv_kernel(md._h).decode()
    assert says in kernel, kernel
    want = torch.zeros(rows_out, cout, dtype=torch.float64, device="cuda")
    mag = want.clone()
    for k, r in enumerate(rules):
        r = torch.as_tensor(r).cuda().long()
        want.index_add_(0, r[:, 1], x[r[:, 0]].double() @ w[k, 0].double())
        mag.index_add_(0, r[:, 1], x[r[:, 0]].double().abs() @ w[k, 0].double().abs())
    assert ((got.double() - want).abs() <= (len(rules) * -(-cin // 32) + 3 + 1 + 4) * 2.0 ** -24 * mag).all()


@pytest.mark.parametrize("cin", [12, 20, 36, 40, 44, 100, 132, 140])
@pytest.mark.parametrize("cout", [8, 32, 40, 96])
@pytest.mark.parametrize("kind", ["subm", "down", "up", "nin"])
def test_one_input_row(kind, cin, cout):
    """A level of one site, plane counts whose last 32 channels are mostly padding: the loads of steps past the last channel are further from the
    row's start than the input is long."""
    import torch
    from test_conv_split_gpu import _table
    conv, rules, rows_in, rows_out, md = _table(kind, 1, 8400)
    assert rows_in == rows_out == 1
    g = torch.Generator().manual_seed(cin + cout)
    x, w, bias = torch.randn(1, cin, generator=g).cuda(), torch.randn(len(rules), 1, cin, cout, generator=g).cuda(), torch.randn(cout, generator=g).cuda()
    got = conv(x, w, bias)
    want, mag = bias.double()[None].clone(), bias.double().abs()[None].clone()
    for k, r in enumerate(rules):
        if len(r):
            want += x.double() @ w[k, 0].double()
            mag += x.double().abs() @ w[k, 0].double().abs()
    assert ((got.double() - want).abs() <= (cin + 4) * 2.0 ** -24 * mag).all()
