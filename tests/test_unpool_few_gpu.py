"""Unpooling over a halving rulebook (k_unpool_few): every fine site receives its parent's row, exactly, at sizes around a workgroup's
elements, to windows of 4096 positions and to the largest table made in one launch, with planes dropped, and where planes or strides do not
allow 16-byte loads (the general kernel)."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 255, 257, 1023, 1025, 4095, 4097, 8191, 40009, 65536, 65537])
@pytest.mark.parametrize("planes,drop", [(4, 0), (20, 0), (64, 0), (36, 4), (7, 0), (12, 3)])
def test_children_receive_their_parents_row(n, planes, drop):
    import torch
    import sparseconvnet_amd as scn
    g = torch.Generator().manual_seed(n + planes)
    side = 64
    cells = torch.randperm(side ** 3, generator=g)[:n]
    coords = torch.stack([cells // side ** 2, cells // side % side, cells % side], 1)
    t = scn.InputLayer(3, side, mode=0)([coords.cuda(), torch.zeros(n, 1).cuda()])
    with torch.no_grad():
        coarse = scn.MaxPooling(3, 2, 2)(t)
        x = torch.randn(coarse.features.size(0), planes, generator=g).cuda()
        x[0, -1] = -0.0
        y = scn.UnPooling(3, 2, 2, drop)(scn.SparseConvNetTensor(x, coarse.metadata, coarse.spatial_size)).features
    row = {tuple(c): i for i, c in enumerate(coarse.metadata.getSpatialLocations(coarse.spatial_size)[:, :3].tolist())}
    parent = torch.tensor([row[tuple(c)] for c in (coords // 2).tolist()]).cuda()
    assert torch.equal(y, x[parent, drop:])
