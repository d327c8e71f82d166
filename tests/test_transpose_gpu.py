"""GPU tests of the tiled permutation kernel (transpose_kernel: 64x64 tiles through LDS) and
of the rule that picks it: every permutation of ragged 2-D, 3-D and 4-D shapes around the tile
edges, sources off 16-byte boundaries, merged and size-1 axes. Bytes must be those of
torch.permute."""
import itertools

import pytest
import torch

from my_pytchon_opencl_lib_amd import _native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 65), (64, 64), (63, 129), (200, 3), (5, 64, 65),
                                   (70, 1, 130), (2200, 70), (129, 3, 66), (2, 127, 40), (3, 65, 2, 70),
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
    ((640, 500), (1, 0), "transpose"), ((9, 32, 32), (0, 2, 1), "transpose"),
    ((9, 31, 33), (0, 2, 1), "permute_gather"), ((30, 20, 10), (2, 1, 0), "transpose"),
    ((70000, 20, 60), (0, 2, 1), "transpose"), ((8, 30, 4, 16), (0, 2, 1, 3), "permute_gather")])
def test_kernel_choice(nncl, shape, axes, kernel):
    x = torch.randn(shape, device="cuda:0")
    assert torch.equal(nncl.Permute(x, axes), x.permute(axes).contiguous())
    assert _native.last_plan().startswith(kernel + " "), _native.last_plan()


@pytest.mark.parametrize("outer,kernel", [((1 << 21) - 1, "transpose"),
                                          (1 << 21, "permute_gather")])
def test_more_tiles_than_one_launch_holds(nncl, outer, kernel):
    """2 x 512 elements per batch entry are 8 tiles: 2^21 entries would need 2^24 work-groups of
    256 threads, one more than a grid holds, and run through the gather kernel."""
    print("tiles of one launch", outer, flush=True)
    x = torch.randn(1 << 20, device="cuda:0").repeat(outer // 1024 + 1)[:outer * 1024]
    x = x.view(outer, 2, 512)
    got = nncl.Permute(x, (0, 2, 1))
    assert _native.last_plan().startswith(kernel + " "), _native.last_plan()
    for i in range(0, outer, 1 << 18):
        assert torch.equal(got[i:i + (1 << 18)], x[i:i + (1 << 18)].transpose(1, 2))
    del x, got
    torch.cuda.empty_cache()
