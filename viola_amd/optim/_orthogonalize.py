"""Quintic Newton-Schulz orthogonalization entry points (viola/optim/_orthogonalize.py:10-57).
Both methods run the HIP GEMM chain, enqueued by the native host path (csrc/host_optim.cpp); `_orthogonalize_kernels.run`
is the same chain product by product. The reference's default instead traces the same recurrences with torch.compile."""

from .. import _lib


def _chain(matrix, steps, gram):
    assert matrix.is_cuda, "viola_amd kernels run on the GPU only"
    return _lib.host().newton_schulz(matrix, steps, gram)


def standard(matrix, steps=5):
    return _chain(matrix, steps, False)


def gram(matrix, steps=5):
    return _chain(matrix, steps, True)


METHODS = {"standard": standard, "gram": gram}
