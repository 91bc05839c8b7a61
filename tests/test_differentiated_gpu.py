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


@pytest.mark.parametrize("fails", ["operands", "call"])
def test_a_call_that_fails_leaves_nothing_behind(fails):
    import ctypes as C
    import torch
    import sparseconvnet_amd as scn
    g = torch.Generator().manual_seed(5)
    cells = torch.randperm(96 ** 3, generator=g)[:3001]
    coords = torch.stack([cells // 96 ** 2, cells // 96 % 96, cells % 96], 1)
    t = scn.InputLayer(3, 96, mode=0)([coords.cuda(), torch.zeros(3001, 1).cuda()])
    md = t.metadata
    conv = scn.SubmanifoldConvolution(3, 16, 16, 3, False).cuda()
    x = torch.randn(3001, 16, generator=g).cuda()
    if fails == "operands":  # refused in Python
        with pytest.raises(Exception):
            conv(scn.SparseConvNetTensor(x.double(), md, t.spatial_size))
    else:  # refused by the library in front of its kernel
        md.nextDifferentiated()
        assert md._L.scn_conv_bn_fwd(md._h, 9, None, None, None, None, None, None, None, None, 16, 16, 1, None, None, C.c_void_p(0), None) != 0
    with torch.no_grad():
        conv(scn.SparseConvNetTensor(x, md, t.spatial_size))
    assert "split wave" in md._L.scn_md_last_conv_kernel(md._h).decode()


def test_calls_without_granule_masks_and_without_scratch_do_not_take_the_kernel():
    """125 taps (tables of more than 32 keep no granule masks), differentiated and not, and the allocation-free entry."""
    import ctypes as C
    import torch
    import sparseconvnet_amd as scn
    from sparseconvnet_amd import _lib
    g = torch.Generator().manual_seed(6)
    cells = torch.randperm(64 ** 3, generator=g)[:3000]
    coords = torch.stack([cells // 64 ** 2, cells // 64 % 64, cells % 64], 1)
    t = scn.InputLayer(3, 64, mode=0)([coords.cuda(), torch.zeros(3000, 1).cuda()])
    md = t.metadata

    def kernel():
        return md._L.scn_md_last_conv_kernel(md._h).decode()
    for planes, out in ((64, 32), (64, 40), (16, 16)):
        x = scn.SparseConvNetTensor(torch.randn(3000, planes, generator=g).cuda(), md, t.spatial_size)
        conv = scn.SubmanifoldConvolution(3, planes, out, 5, False).cuda()
        y = conv(x).features
        assert "split wave" not in kernel(), kernel()
        y.sum().backward()
        with torch.no_grad():
            assert torch.equal(conv(x).features, y.detach())
        assert "split wave" not in kernel(), kernel()
    x, w = torch.randn(3000, 32, generator=g).cuda(), torch.randn(27, 1, 32, 32, generator=g).cuda()
    sp, fs = md._s(t.spatial_size), md._s(torch.LongTensor([3, 3, 3]))
    _lib.check(md._L.scn_md_submanifold_rules(md._h, sp, fs, C.c_void_p(0)))
    y = torch.empty(3000, 32).cuda()
    _lib.check(md._L.scn_subm_conv_fwd_noalloc(md._h, sp, fs, C.c_void_p(x.data_ptr()), C.c_void_p(y.data_ptr()), C.c_void_p(w.data_ptr()), None,
                                               32, 32, C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    assert "split wave" not in kernel(), kernel()
    torch.cuda.synchronize()
