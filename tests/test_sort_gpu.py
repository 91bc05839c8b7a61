"""The rulebook builders' radix sort through the C ABI against numpy's stable argsort: sizes around
the one-workgroup limit and the tile size, ragged tails, 1 to 64 key bits, repeated keys (stability
is what makes the input layer's first-occurrence row numbers come out)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,bits", [(1, 8), (63, 3), (4096, 16), (4097, 16), (2048 * 3 + 5, 24), (100003, 36),
                                    (1 << 20, 40), (300000, 64), (70000, 1), (5000, 9), (2500000, 33),
                                    (1000, 27), (4095, 35), (3001, 64), (2, 1),
                                    # two launches per digit: odd tiles, one, two and four digit values per thread, the ends of the range
                                    (6144, 27), (6145, 27), (8191, 7), (8192, 27), (8193, 27), (9001, 8), (16385, 18), (20001, 10), (32767, 40), (32768, 29),
                                    (32769, 29)])
def test_sort_pairs(n, bits):
    import torch
    from sparseconvnet_amd import _lib
    L = _lib.lib()
    rng = np.random.default_rng(n + bits)
    span = min(bits, 12) if n % 2 else bits  # odd sizes: few distinct keys, many repeats
    keys = rng.integers(0, 1 << min(span, 63), size=n, dtype=np.uint64)
    if bits == 64:
        keys |= rng.integers(0, 2, size=n, dtype=np.uint64) << np.uint64(63)
    junk = rng.integers(0, 1 << 20, size=n, dtype=np.uint64) << np.uint64(bits) if bits < 44 else np.zeros(n, np.uint64)
    keys_all = keys | junk  # bits above end_bit must not matter
    vals = np.arange(n, dtype=np.int32)
    kin = torch.as_tensor(keys_all.view(np.int64)).cuda()
    vin = torch.as_tensor(vals).cuda()
    kout, vout = torch.empty_like(kin), torch.empty_like(vin)
    h = L.scn_md_create(3)
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(L.scn_sort_pairs(h, C.c_void_p(kin.data_ptr()), C.c_void_p(kout.data_ptr()), C.c_void_p(vin.data_ptr()),
                                C.c_void_p(vout.data_ptr()), n, bits, stream))
    torch.cuda.synchronize()
    mask = np.uint64((1 << bits) - 1) if bits < 64 else np.uint64(0xFFFFFFFFFFFFFFFF)
    order = np.argsort(keys_all & mask, kind="stable")
    assert (vout.cpu().numpy() == vals[order]).all()
    assert (kout.cpu().numpy().view(np.uint64) == keys_all[order]).all()
    assert (kin.cpu().numpy().view(np.uint64) == keys_all).all(), "the input arrays must not be written"
    L.scn_md_destroy(h)


@pytest.mark.parametrize("n", [4096, 4097, 6145, 20001, 32768, 32769])
@pytest.mark.parametrize("side,batch", [(500, 1), (1024, 3), (4096, 2)])
def test_input_layers_whichever_sort_they_take(n, side, batch):
    """Keys of up to three digits and more: rows in the order of their sites' first points, each the sum of its points' vectors."""
    import torch
    import sparseconvnet_amd as scn
    rng = np.random.default_rng(n + side)
    first = rng.integers(0, side, size=(n - n // 4, 3))
    coords = np.concatenate([first, first[rng.integers(0, len(first), n // 4)]])  # a quarter of the points repeat a site
    coords = np.concatenate([coords, rng.integers(0, batch, size=(n, 1))], 1)[rng.permutation(n)]
    coords[0, 3] = batch - 1
    x = rng.integers(-8, 9, size=(n, 2)).astype(np.float32)  # sums are exact
    t = scn.InputLayer(3, side, mode=3)([torch.as_tensor(coords).cuda(), torch.as_tensor(x).cuda()])
    sites, at, inverse = np.unique(coords, axis=0, return_index=True, return_inverse=True)
    order = np.argsort(at)
    want = np.zeros((len(sites), 2), np.float32)
    np.add.at(want, inverse.reshape(-1), x)
    assert (t.metadata.getSpatialLocations(t.spatial_size).cpu().numpy() == sites[order]).all()
    assert (t.features.cpu().numpy() == want[order]).all()
