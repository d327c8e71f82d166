"""GPU tests of the tiled permutation kernel (transpose_kernel: 64x64 or 32x32 tiles through
LDS) and of the rule that picks it: every permutation of ragged 2-D, 3-D and 4-D shapes around the tile
edges, sources off 16-byte boundaries, merged and size-1 axes. Bytes must be those of
torch.permute."""
import itertools

import pytest
import torch

from my_pytchon_opencl_lib_amd import _native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 65), (64, 64), (63, 129), (200, 3), (5, 64, 65),
                                   (70, 1, 130), (2200, 70), (129, 3, 66), (2, 127, 40), (3, 65, 2, 70),
                                   (40, 33, 31), (600, 32), (9, 24, 24), (3, 100, 20),
                                   (7, 5, 64, 33), (66, 4, 3, 5), (2, 3, 4, 5, 130)])
def test_every_permutation(nncl, shape):
    n = 1
    for s in shape:
        n *= s
    buf = torch.randn(n + 1, device="cuda:0")
    for off in (0, 1):
        x = buf[off:off + n].view(shape)
        for axes in itertools.permutations(range(len(shape))):
            got = nncl.Permute(x, axes)
            assert torch.equal(got, x.permute(axes).contiguous()), (axes, off)


@pytest.mark.parametrize("shape,axes,kernel", [
    ((640, 500), (1, 0), "transpose tile=64x64"), ((30, 20, 10), (2, 1, 0), "transpose tile=32x32"),
    # both sides of each line: 32x32 tiles for 32 or fewer contiguous elements ...
    ((9, 32, 32), (0, 2, 1), "transpose tile=32x32"), ((9, 32, 33), (0, 2, 1), "transpose tile=64x64"),
    # ... unless over a quarter of several tiles is empty
    ((9, 48, 32), (0, 2, 1), "transpose tile=32x32"), ((9, 47, 32), (0, 2, 1), "transpose tile=64x64"),
    # no tiles with fewer than 320, 256 (33-128 rows), 224 (more) or 512 (64x64) elements
    ((9, 16, 20), (0, 2, 1), "transpose tile=32x32"), ((9, 16, 19), (0, 2, 1), "permute_gather"),
    ((9, 64, 8), (0, 2, 1), "transpose tile=32x32"), ((9, 64, 7), (0, 2, 1), "permute_gather"),
    ((9, 160, 7), (0, 2, 1), "transpose tile=32x32"), ((9, 160, 6), (0, 2, 1), "permute_gather"),
    ((9, 8, 64), (0, 2, 1), "transpose tile=64x64"), ((9, 8, 63), (0, 2, 1), "permute_gather"),
    ((100000, 3), (1, 0), "permute_gather"), ((3, 100000), (1, 0), "permute_gather"),
    ((70000, 20, 60), (0, 2, 1), "transpose tile=64x64"),
    ((8, 30, 4, 16), (0, 2, 1, 3), "permute_gather")])
def test_kernel_choice(nncl, shape, axes, kernel):
    x = torch.randn(shape, device="cuda:0")
    assert torch.equal(nncl.Permute(x, axes), x.permute(axes).contiguous())
    assert _native.last_plan().startswith(kernel + " "), _native.last_plan()


@pytest.mark.parametrize("outer,kernel", [((1 << 23) - 1, "transpose"),
                                          (1 << 23, "permute_gather")])
def test_more_tiles_than_one_launch_holds(nncl, outer, kernel):
    """64 x 8 elements per batch entry are 2 tiles: 2^23 entries would need 2^24 work-groups of
    256 threads, one more than a grid holds, and run through the gather kernel (17 GB)."""
    print("tiles of one launch", outer, flush=True)
    part = 1 << 18
    x = torch.randn(part, 64, 8, device="cuda:0").repeat((outer - 1) // part + 1, 1, 1)[:outer]
    got = nncl.Permute(x, (0, 2, 1))
    assert _native.last_plan().startswith(kernel + " "), _native.last_plan()
    for i in range(0, outer, part):
        assert torch.equal(got[i:i + part], x[i:i + part].transpose(1, 2))
    del x, got
    torch.cuda.empty_cache()
