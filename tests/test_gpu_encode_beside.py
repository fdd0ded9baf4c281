"""A gradient's per-tensor codes with another matrix's codes turned in the same launch equal the two calls apart."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _buffers(rows, cols, slices):
    pitch, pitch_t = -(-cols // 128) * 128, -(-rows // 128) * 128
    full = lambda *shape: torch.full(shape, 0x55, dtype=torch.uint8, device="cuda")
    return (torch.empty(1024 + slices * cols, device="cuda"), torch.zeros(4, device="cuda"), torch.empty(1, device="cuda"), full(rows, pitch),
            full(cols, pitch_t), torch.empty(cols, device="cuda"))


def _encode(name, x, buffers, index, delayed, sums, *codes):
    from viola_amd import _lib
    work, history, scale, q, qt, total = buffers
    _lib.call(name, _lib.ptr(x), _lib.BF16, *x.shape, _lib.ptr(work), work.numel(), _lib.ptr(history), 4, index, delayed, 57344.0, _lib.ptr(scale), _lib.ptr(q),
              q.shape[1], _lib.ptr(qt), qt.shape[1], _lib.E5M2, _lib.ptr(total) if sums else None, _lib.F32, *codes)
    return history, scale, q, qt, *((total,) if sums else ())


# one block's tile, its edges, several tiles with rows of zeros behind them, more blocks than the quantizer has; the last gradient has too many
# maxima for the quantizer's blocks, whose scale is then a launch of its own, as a delayed one is
@pytest.mark.parametrize("rows,cols,code_rows,code_cols,code_pitch", [(1, 8, 4, 4, 4), (3, 8, 64, 64, 64), (100, 264, 68, 60, 128), (65, 64, 2048, 512, 2048),
                                                                      (256, 128, 300, 1028, 384), (8192, 4096, 132, 128, 256)])
def test_codes_turned_beside_a_quantizer(rows, cols, code_rows, code_cols, code_pitch):
    from viola_amd import _lib
    torch.manual_seed(rows + code_rows)
    x = torch.randn(rows, cols).bfloat16().cuda()
    codes = torch.randint(0, 256, (code_rows, code_cols), dtype=torch.uint8).cuda()
    slices = _lib.library().viola_tensor_encode_slices(_lib.BF16, rows, cols)
    for index, delayed, sums in ((0, 0, False), (2, 1, False), (3, 0, True)):
        turned = torch.full((code_cols, code_pitch), 0x55, dtype=torch.uint8, device="cuda")
        apart = _encode("viola_tensor_encode", x, _buffers(rows, cols, slices), index, delayed, sums)
        beside = _encode("viola_tensor_encode_beside", x, _buffers(rows, cols, slices), index, delayed, sums, _lib.ptr(codes), _lib.ptr(turned), code_rows,
                         code_cols, code_pitch)
        assert all(torch.equal(a, b) for a, b in zip(apart, beside))
        assert torch.equal(turned[:, :code_rows], codes.T) and (turned[:, code_rows:] == 0).all()


@pytest.mark.parametrize("code_rows,code_cols,code_pitch,offset", [(6, 8, 8, 0), (8, 6, 8, 0), (8, 8, 10, 0), (8, 8, 8, 1)])
def test_codes_that_are_no_whole_words_are_refused(code_rows, code_cols, code_pitch, offset):
    from viola_amd import _lib
    x = torch.randn(16, 16).bfloat16().cuda()
    codes, turned = torch.zeros(128, dtype=torch.uint8, device="cuda"), torch.zeros(256, dtype=torch.uint8, device="cuda")
    buffers = _buffers(16, 16, _lib.library().viola_tensor_encode_slices(_lib.BF16, 16, 16))
    with pytest.raises(RuntimeError):
        _encode("viola_tensor_encode_beside", x, buffers, 0, 0, False, _lib.ptr(codes[offset:]), _lib.ptr(turned), code_rows, code_cols, code_pitch)
    torch.cuda.synchronize()
    assert (buffers[3] == 0x55).all() and (buffers[4] == 0x55).all()


@pytest.mark.parametrize("out_features,in_features", [(96, 64), (70, 64), (2048, 512)])
def test_linear_backward_turns_the_weight_in_the_quantizer(out_features, in_features):
    from viola_amd import _lib, nn
    torch.manual_seed(3)
    layer = nn.Linear(in_features, out_features, device="cuda", dtype=torch.bfloat16, scaling="current", mode="memory", weight_dtype="fp8")
    x = torch.randn(128, in_features).bfloat16().cuda().requires_grad_()
    y = layer(x)
    _lib.timeline = []
    try:
        y.backward(torch.randn_like(y))
        torch.cuda.synchronize()
        names = [row[0] for row in _lib.timeline]
    finally:
        _lib.timeline = None
    assert "viola_tensor_encode_beside" in names
    assert ("viola_codes_transpose_pitched" in names) == (out_features % 4 != 0)
