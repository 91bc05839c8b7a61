"""A convolution whose output will be differentiated runs in the kernels that served it before k_conv_wave, for that one call."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,planes", [(3001, 16), (30001, 32), (2001, 48)])
def test_one_call_keeps_its_rounding(n, planes):
    import torch
    import sparseconvnet_amd as scn
    g = torch.Generator().manual_seed(n)
    side = 96
    cells = torch.randperm(side ** 3, generator=g)[:n]
    coords = torch.stack([cells // side ** 2, cells // side % side, cells % side], 1)
    t = scn.InputLayer(3, side, mode=0)([coords.cuda(), torch.zeros(n, 1).cuda()])
    x = scn.SparseConvNetTensor(torch.randn(n, planes, generator=g).cuda(), t.metadata, t.spatial_size)
    conv = scn.SubmanifoldConvolution(3, planes, planes, 3, False).cuda()

    def kernel():
        return t.metadata._L.scn_md_last_conv_kernel(t.metadata._h).decode()
    with torch.no_grad():
        a = conv(x).features
    assert "split wave" in kernel()
    b = conv(x).features
    assert "split wave" not in kernel()
    with torch.no_grad():
        c = conv(x).features
    assert "split wave" in kernel() and torch.equal(a, c)
    assert (a - b).norm() <= 1e-6 * a.norm()


@pytest.mark.parametrize("n,cin,cout", [(300001, 32, 32), (300001, 64, 24), (600001, 48, 32), (310001, 20, 20)])
def test_large_levels_have_one_rounding(n, cin, cout):
    """From 300 k sites on k_conv_wave adds in k_conv_split's order: the same bits, so that differentiated calls use it as well."""
    import torch
    from test_conv_split_gpu import _table
    conv, rules, rows_in, rows_out, md = _table("subm", n, 8400)
    g = torch.Generator().manual_seed(n + cin)
    x, w = torch.randn(rows_in, cin, generator=g).cuda(), torch.randn(len(rules), 1, cin, cout, generator=g).cuda() * 0.1
    bias = torch.randn(cout, generator=g).cuda()
    md.nextDifferentiated()
    got = conv(x, w, bias)
    assert "split wave" in md._L.scn_md_last_conv_kernel(md._h).decode()
    # 52 planes of which the first cout are these: k_conv_split, a tile's columns do not depend on one another
    wide = torch.zeros(len(rules), 1, cin, 52).cuda()
    wide[..., :cout] = w
    want = conv(x, wide, torch.cat([bias, torch.zeros(52 - cout).cuda()]))
    assert "split ncbw" in md._L.scn_md_last_conv_kernel(md._h).decode()
    assert torch.equal(got, want[:, :cout])
