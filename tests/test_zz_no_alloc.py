"""The allocation-free TV prox (qh_hip_tv_prox_dev_noalloc: device pointers, the dual in the
library's fixed device array) against the allocating entry point qh_hip_tv_prox on the same
inputs, bit for bit, over consecutive calls whose volumes shrink (the fixed array keeps the
previous call's dual, which each call must clear), and its refusal of volumes above the limit."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MAX_VOXELS = 2097152  # QH_TV_NOALLOC_MAX_VOXELS


def _prox_allocating(lib, native, b, lam, inner, fused):
    x = np.empty_like(b)
    nz, ny, nx = b.shape
    native.check(lib.qh_hip_tv_prox(native.ptr(b), nz, ny, nx, lam, inner, fused, native.ptr(x)))
    return x


# Passes are of up to four steps now: 5 steps are 3 + 2, and 4 steps of a small volume 2 + 2.
def test_noalloc_prox_equals_allocating_prox(device):
    import torch
    from qoraholo_amd import _native

    lib = _native.lib()
    rng = np.random.default_rng(11)
    stream = torch.cuda.current_stream()
    # Consecutive calls, each volume smaller than the one before: two FGP steps per pass with
    # an odd last step, x tiles of a 384-wide row, single steps only.
    cases = [((40, 48, 56), 0.03, 5, 1), ((8, 20, 384), 0.02, 4, 1), ((24, 20, 32), 0.05, 3, 0)]
    for shape, lam, inner, fused in cases:
        print(f"noalloc prox {shape} inner {inner} fused {fused}", flush=True)
        b = (rng.standard_normal(shape) * 0.2 + 0.3).astype(np.float32)
        want = _prox_allocating(lib, _native, b, lam, inner, fused)
        bd = torch.from_numpy(b).cuda()
        xd = torch.full(shape, float("nan"), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        _native.check(lib.qh_hip_tv_prox_dev_noalloc(
            _native.ptr(bd.data_ptr()), *shape, lam, inner, fused, _native.ptr(xd.data_ptr()),
            _native.ptr(stream.cuda_stream)))
        torch.cuda.synchronize()
        got = xd.cpu().numpy()
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), shape
        assert np.all(got >= 0)


def test_noalloc_prox_in_place(device):
    """The output may be the input: tiles read b beyond their own points while others write."""
    import torch
    from qoraholo_amd import _native

    lib = _native.lib()
    rng = np.random.default_rng(12)
    stream = torch.cuda.current_stream()
    for shape, inner in [((20, 70, 130), 10), ((9, 33, 65), 3), ((4, 8, 16), 0)]:
        b = (rng.standard_normal(shape) * 0.2 + 0.3).astype(np.float32)
        want = _prox_allocating(lib, _native, b, 0.03, inner, 1)
        bd = torch.from_numpy(b).cuda()
        _native.check(lib.qh_hip_tv_prox_dev_noalloc(
            _native.ptr(bd.data_ptr()), *shape, 0.03, inner, 1, _native.ptr(bd.data_ptr()),
            _native.ptr(stream.cuda_stream)))
        torch.cuda.synchronize()
        assert np.array_equal(bd.cpu().numpy().view(np.uint32), want.view(np.uint32)), shape


@pytest.mark.parametrize("shape,inner", [((128, 127, 129), 10), ((3000, 1, 500), 3), ((700, 5, 450), 4)])
def test_noalloc_prox_without_room_for_whole_groups_of_rows(device, shape, inner):
    """Volumes near the limit whose row count is no multiple of four: the fixed array holds their
    dual only without the rows that would fill the last group. The allocating call has that room."""
    import torch
    from qoraholo_amd import _native

    lib = _native.lib()
    rows = -(-shape[1] // 4) * 4
    assert np.prod(shape) <= MAX_VOXELS < shape[0] * rows * shape[2]
    rng = np.random.default_rng(shape[1])
    b = (rng.standard_normal(shape) * 0.2 + 0.3).astype(np.float32)
    want = _prox_allocating(lib, _native, b, 0.05, inner, 1)
    bd = torch.from_numpy(b).cuda()
    xd = torch.empty_like(bd)
    _native.check(lib.qh_hip_tv_prox_dev_noalloc(
        _native.ptr(bd.data_ptr()), *shape, 0.05, inner, 1, _native.ptr(xd.data_ptr()),
        _native.ptr(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    assert np.array_equal(xd.cpu().numpy(), want)


def test_noalloc_prox_refuses_volumes_above_the_limit(device):
    import torch
    from qoraholo_amd import _native

    lib = _native.lib()
    bd = torch.zeros(16, device="cuda")
    for shape in [(129, 128, 128), (2, 1024, 1025)]:
        assert shape[0] * shape[1] * shape[2] > MAX_VOXELS
        with pytest.raises(ValueError, match="exceeds the fixed dual buffer"):
            _native.check(lib.qh_hip_tv_prox_dev_noalloc(
                _native.ptr(bd.data_ptr()), *shape, 0.01, 2, 1, _native.ptr(bd.data_ptr()),
                _native.ptr(0)))
