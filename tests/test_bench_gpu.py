"""bench.py's per-layer table puts itself between the layers and the library: it takes every call the layers make."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_the_table_of_layers_covers_a_whole_network():
    import bench
    import sparseconvnet_amd as scn
    g = torch.Generator().manual_seed(5)
    n = 600
    coords = torch.cat([torch.randint(0, 24, (n, 3), generator=g), torch.zeros(n, 1, dtype=torch.long)], 1)
    model = scn.Sequential().add(scn.SubmanifoldConvolution(3, 3, 16, 3, False)).add(
        scn.UNet(3, 1, [16, 32], False)).add(scn.BatchNormReLU(16)).cuda().eval()
    x = scn.InputLayer(3, 32, mode=4)([coords.cuda(), torch.randn(n, 3, generator=g).cuda()])
    with torch.no_grad():
        want = model(x).features
    rows = bench.unet_layer_table(torch, scn, model, x, reps=1)
    kinds = [r["op"] for r in rows]
    assert kinds.count("Convolution") == 1 and kinds.count("Deconvolution") == 1, kinds
    # the first layer, one block of one layer on each side of the down and up sampling, and one inside
    assert kinds.count("SubmanifoldConvolution") >= 4, kinds
    assert all(r["kernel"] and r["rules"] > 0 for r in rows)
    with torch.no_grad():  # and it is out of the way again
        assert torch.equal(model(x).features, want)
