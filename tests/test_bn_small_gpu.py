"""Training-mode batch normalisation of up to 1536 rows in one launch: to the bit what the launches for larger levels give, which
arrays that are not 16-byte aligned still take, around the ends of row blocks, column groups and the range; and what 64 bits give."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 2, 15, 17, 255, 256, 257, 513, 1279, 1535, 1536, 1537])
@pytest.mark.parametrize("planes", [4, 16, 20, 32, 36, 64, 100, 224])
@pytest.mark.parametrize("stride", [0, 8])
def test_one_launch_gives_what_three_give(rows, planes, stride):
    import torch
    from sparseconvnet_amd import _lib
    L = _lib.lib()
    g = torch.Generator().manual_seed(rows * 7 + planes)

    def normal(*shape):
        return torch.randn(*shape, generator=g).cuda()
    ld = planes + stride
    x, dy = normal(rows, ld), normal(rows, ld)
    gamma, beta = torch.rand(planes, generator=g).cuda() + 0.5, normal(planes)
    leak, eps = 0.1, 1e-4
    s = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    h = L.scn_md_create(3)

    def p(t):
        return C.c_void_p(t.data_ptr())
    got = []
    for offset in (0, 1):  # one float off: three launches
        flat = [torch.full((rows * ld + 4,), 7.0).cuda() for _ in range(2)]
        y, dx = (f[offset:offset + rows * ld].view(rows, ld) for f in flat)
        mean, invstd, rm, d_gamma, d_beta = (torch.zeros(planes).cuda() for _ in range(5))
        rv = torch.ones(planes).cuda()
        _lib.check(L.scn_bn_train_fwd(h, p(x), p(y), rows, planes, ld, ld, p(mean), p(invstd), p(rm), p(rv), p(gamma), p(beta), eps, 0.9,
                                      leak, s))
        # the gradient reads the aligned output on both sides: only where it is written differs
        out = y.clone() if offset == 0 else got[0][0]
        _lib.check(L.scn_bn_bwd(h, p(x), p(dx), p(out), p(dy), rows, planes, ld, ld, p(mean), p(invstd), p(gamma), p(d_gamma), p(d_beta), leak, s))
        got.append([y.clone(), dx.clone(), mean, invstd, rm, rv, d_gamma, d_beta])
        assert (y[:, planes:] == 7.0).all() and (dx[:, planes:] == 7.0).all()
        assert (flat[0][rows * ld + offset:] == 7.0).all() and (flat[1][rows * ld + offset:] == 7.0).all()
    L.scn_md_destroy(h)
    for a, b in zip(*got):
        assert torch.equal(a.nan_to_num(5.0), b.nan_to_num(5.0))  # (the unbiased variance of one row is not a number)
    if rows >= 256:  # sums of at most 16 + 64 terms in fp32, then 64 bits; the variance by a difference of sums: some 1e-5 of each value
        xd, g64 = x[:, :planes].double(), gamma.double()
        mu, var = xd.mean(0), xd.var(0, unbiased=False)
        want = (xd - mu) / torch.sqrt(var + eps) * g64 + beta.double()
        want = torch.where(want > 0, want, leak * want)
        assert (got[0][0][:, :planes].double() - want).abs().max() <= 2e-5 * want.abs().max()
