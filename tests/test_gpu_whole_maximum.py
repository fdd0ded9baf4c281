"""Small tensors, whose quantizer's blocks each take the maximum of the whole: scale, history and codes are the definition's at any offset and
size, and with infinities and NaN in any place."""

import pytest
import torch

import oracle.tensor as ot

pytestmark = pytest.mark.gpu


def _encode(x, limit, index=0, delayed=0, work=None):
    from viola_amd import _lib
    rows, cols = x.shape
    pitch_t = -(-rows // 128) * 128
    history, scale = torch.zeros(4, device="cuda"), torch.empty(1, device="cuda")
    q, qt = torch.empty(rows, cols, dtype=torch.uint8, device="cuda"), torch.empty(cols, pitch_t, dtype=torch.uint8, device="cuda")
    code = {torch.float32: _lib.F32, torch.bfloat16: _lib.BF16, torch.float16: _lib.F16}[x.dtype]
    work = torch.full((1024,), float("nan"), device="cuda") if work is None else work
    _lib.call("viola_tensor_encode", _lib.ptr(x), code, rows, cols, _lib.ptr(work), 1024, _lib.ptr(history), 4, index, delayed, limit, _lib.ptr(scale), _lib.ptr(q),
              cols, _lib.ptr(qt), pitch_t, _lib.E4M3, None, _lib.F32)
    return history.cpu(), scale.cpu(), q.cpu(), qt.cpu()


def _check(x, history, scale, q, qt):
    amax = torch.nan_to_num(x.float().abs(), nan=0.0, posinf=float("inf")).max()
    assert torch.equal(history, torch.tensor([amax, 0, 0, 0])) and torch.equal(scale, torch.clamp_min(amax, 1e-30).reshape(1) / 448.0)
    codes = ot.quantize(x, scale, torch.float8_e4m3fn).view(torch.uint8)
    nan = torch.isnan(codes.view(torch.float8_e4m3fn).float())
    for got in (q, qt[:, :x.shape[0]].T):
        assert torch.equal(got[~nan], codes[~nan]) and torch.isnan(got.contiguous().view(torch.float8_e4m3fn).float()[nan]).all()
    assert (qt[:, x.shape[0]:] == 0).all()


# fewer values than a load, a thread's, a turn's and one more; the largest of the range and the first beyond it, in bytes and in tiles
@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 5), (1, 2049), (129, 255), (512, 64), (513, 64), (128, 512), (256, 512), (257, 512), (8, 8192), (8, 8256)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("offset", [0, 3])
def test_maximum_of_a_small_tensor(rows, cols, dtype, offset):
    torch.manual_seed(rows + cols)
    for place in (0, rows * cols - 1, rows * cols // 2):
        flat = torch.randn(rows * cols + offset).to(dtype)
        flat[offset + place] = -7.5
        x = flat[offset:].view(rows, cols)
        _check(x, *_encode(flat.cuda()[offset:].view(rows, cols), 448.0))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("place", [0, 1, 2047, 6000, 12287])
def test_nan_is_no_maximum(dtype, place):
    torch.manual_seed(place)
    for bad in (float("nan"), -float("nan")):
        x = torch.randn(96, 128).to(dtype)
        x.view(-1)[place] = bad
        _check(x, *_encode(x.cuda(), 448.0))
    _check(torch.full((96, 128), float("nan")).to(dtype), *_encode(torch.full((96, 128), float("nan")).to(dtype).cuda(), 448.0))
    x = torch.randn(96, 128).to(dtype)
    x.view(-1)[place] = -float("inf")
    history, scale, _, _ = _encode(x.cuda(), 448.0)
    assert history[0] == float("inf") and scale[0] == float("inf")


@pytest.mark.parametrize("dtype,kilobytes,whole", [(torch.bfloat16, 256, True), (torch.float16, 256, True), (torch.float32, 192, True), (torch.bfloat16, 260, False),
                                                    (torch.float16, 260, False), (torch.float32, 196, False)])
def test_beyond_its_limit_the_maximum_is_a_pass_of_its_own(dtype, kilobytes, whole):
    """There the blocks' walks over the whole tensor take longer than the launch that they save, over an x that no cache holds most of all. Only the pass
    leaves maxima in the workspace. The largest value lies in each of a walk's turns of 64 KB, wherever a block begins."""
    n = (kilobytes << 10) // torch.finfo(dtype).bits * 8
    for place in range(n // 8, n, n // 4):
        x = torch.randn(n).to(dtype).view(-1, 256)
        x.view(-1)[place] = 30.0
        work = torch.full((1024,), float("nan"), device="cuda")
        _check(x, *_encode(x.cuda(), 448.0, work=work))
        assert torch.isnan(work).all().item() == whole
