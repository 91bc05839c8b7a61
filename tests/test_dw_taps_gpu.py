"""Weight gradients of up to 32 planes on both sides (all taps per workgroup): sizes around granules, blocks of 128 positions and one
block per workgroup, plane counts that are no multiple of anything, against sums in 64 bits over the exported rules.

Tolerance: a sum of R products in fp32, in any order, is off by at most R 2^-24 of the sum of their magnitudes; the partial sums of a
few hundred workgroups are part of those R."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 16, 127, 128, 129, 257, 299, 300, 5003, 32767, 32769, 70001])
@pytest.mark.parametrize("dim,size,planes", [(3, 3, (8, 8)), (3, 3, (32, 32)), (3, 3, (7, 9)), (2, 3, (16, 24)), (3, 1, (5, 32)), (2, 5, (20, 12))])
def test_weight_gradient(n, dim, size, planes):
    import torch
    import sparseconvnet_amd as scn
    n_a, n_b = planes
    g = torch.Generator().manual_seed(n + n_a)
    side = max(4, int((4.0 * n) ** (1.0 / dim)) + 1)
    cells = torch.randperm(side ** dim, generator=g)[:n]
    coords = torch.stack([cells // side ** d % side for d in range(dim)], 1)
    t = scn.InputLayer(dim, side, mode=0)([coords.cuda(), torch.zeros(n, 1).cuda()])
    conv = scn.SubmanifoldConvolution(dim, n_a, n_b, size, False).cuda()
    x = torch.randn(n, n_a, generator=g).cuda()
    dy = torch.randn(n, n_b, generator=g).cuda()
    y = conv(scn.SparseConvNetTensor(x.requires_grad_(True), t.metadata, t.spatial_size)).features
    y.backward(dy)
    got = conv.weight.grad.view(size ** dim, n_a, n_b)
    grid = torch.full((side + size,) * dim, -1, dtype=torch.long)
    half = size // 2
    grid[tuple((coords + half).T)] = torch.arange(n)
    for k in range(size ** dim):
        offset = torch.tensor([k // size ** (dim - 1 - d) % size for d in range(dim)])
        j = grid[tuple((coords + offset).T)].cuda()  # the neighbour each position reads through tap k
        at = (j >= 0).nonzero()[:, 0]
        a, b = x.detach()[j[at]].double(), dy[at].double()
        bound = (len(at) + 4) * 2.0 ** -24 * (a.abs().T @ b.abs()) + 1e-30
        assert ((got[k].double() - a.T @ b).abs() <= bound).all(), k


@pytest.mark.parametrize("kind,n,n_a,n_b", [("nin", 700001, 16, 32), ("subm", 700001, 32, 32)])
def test_sums_over_large_levels_are_cut_into_512_shares(kind, n, n_a, n_b):
    """Of products of either sign the partial sums grow like the square root of their number, and a sum of m additions in fp32 is off by
    sqrt(c m / 2) 2^-24 of its size (2-norm; c = 0.18, the mean square of a rounding error over numbers whose logarithm is uniform).
    A tap with R rules is summed in 512 shares, m = R / 512; 256 shares would be off by 1.41 times as much, the bound is 1.2 times.
    (Adding the shares up comes on top, in quadrature: a few percent where a share has as many rules as here.)"""
    import torch
    from test_conv_split_gpu import _table
    _, rules, rows_in, rows_out, md = _table(kind, n, 9900 + n % 79)
    g = torch.Generator().manual_seed(n + n_a)
    x, d = torch.randn(rows_in, n_a, generator=g).cuda(), torch.randn(rows_out, n_b, generator=g).cuda()
    w = torch.zeros(len(rules), 1, n_a, n_b).cuda()
    if kind == "nin":
        got = md.networkInNetworkBackward(x, d, w[0, 0], False)[1]
    else:
        got = md.submanifoldConvolutionBackward(torch.LongTensor([1022] * 3), torch.LongTensor([3] * 3), x, d, w, False)[1]
    got = got.reshape(len(rules), n_a, n_b).double()
    error = limit = 0.0
    for k, r in enumerate(rules):
        r = torch.as_tensor(r).cuda().long()
        want = x[r[:, 0]].double().t().contiguous() @ d[r[:, 1]].double()
        error += float((got[k] - want).norm()) ** 2
        limit += 0.18 * len(r) / 512 / 2 * 2.0 ** -48 * float(want.norm()) ** 2
    assert error <= 1.2 ** 2 * limit, (error / limit) ** 0.5
