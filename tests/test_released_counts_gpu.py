"""Multiply-adds of handles that died before anyone asked: the same number as from a live handle, also where tables are shared by
several convolutions, more than one launch's worth of tables is left behind, and earlier handles' counts are folded on the way."""
import gc

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("levels", [1, 7])
@pytest.mark.parametrize("handles", [1, 5])
def test_counts_left_behind_equal_those_taken(levels, handles):
    import numpy as np
    import torch
    import sparseconvnet_amd as scn
    from sparseconvnet_amd import synthetic
    from sparseconvnet_amd.metadata import mac_counter
    torch.manual_seed(levels)
    coords = torch.as_tensor(np.concatenate([synthetic.shells_and_planes(b, 64, 1500, b) for b in range(2)])).cuda()
    x = torch.randn(len(coords), 3).cuda()
    net = scn.Sequential().add(scn.SubmanifoldConvolution(3, 3, 8, 3, False)).add(
        scn.UNet(3, 2, [8 * (i + 1) for i in range(levels)], False)).add(scn.OutputLayer(3)).cuda().eval()
    layer = scn.InputLayer(3, 256, mode=4)

    def scene():
        t = layer([coords, x])
        with torch.no_grad():
            return t.metadata, net(t)
    gc.collect()
    torch.cuda.synchronize()
    mac_counter.reset(0)
    md, _ = scene()
    want = md.takeMacs()
    assert want > 0
    del md, _
    mac_counter.reset(0)
    for _ in range(handles):
        scene()
        torch.cuda.synchronize()
    gc.collect()
    assert mac_counter.read() == handles * want
