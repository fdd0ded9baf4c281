"""What an optimizer step holds and allocates on the way."""

import gc

import pytest
import torch

import viola_amd

pytestmark = pytest.mark.gpu


def _optimizer(shapes, **options):
    torch.manual_seed(0)
    params = [torch.nn.Parameter(torch.randn(*s, device="cuda") * .05) for s in shapes]
    opt = viola_amd.optim.FP8Muon(params, lr=2e-3, **options)
    for p in params:
        p.grad = torch.randn_like(p) * 1e-2
    opt.step()                                                                # state and pointer tables
    torch.cuda.synchronize()
    return params, opt


def _peak(opt):
    """Bytes that a step holds at once beyond what is there before it (optimizers that are no longer in use are not: they would go on the way)."""
    gc.collect()
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    opt.step()
    torch.cuda.synchronize()
    return torch.cuda.max_memory_allocated() - before


@pytest.mark.parametrize("method", ["standard", "gram"])
def test_a_step_holds_no_more_than_its_lanes_may(method):
    """Buckets of one matrix, one at a time: what one of them needs, not four. Per element 2 bytes of updates, 2 of the result, 4 for the two sides of
    the chain and 1 for each of its two squares of 512 x 512 (six in the Gram recurrence); sums, tables and the allocator's rounding to
    pieces of 2 MB."""
    shapes, elements = [(512, 1024)] * 4, 512 * 1024
    params, opt = _optimizer(shapes, ns_method=method)
    together = _peak(opt)
    opt._LANES, opt._BATCH_ELEMENTS = 1, elements
    opt.step()
    one = _peak(opt)
    assert one <= (10 if method == "standard" else 14) * elements + (2 << 20) and together > 2 * one


def _allocated(opt):
    """Bytes that a step asks the allocator for, freed on the way or not."""
    torch.cuda.synchronize()
    before = torch.cuda.memory_stats()["allocated_bytes.all.allocated"]
    opt.step()
    torch.cuda.synchronize()
    return torch.cuda.memory_stats()["allocated_bytes.all.allocated"] - before


@pytest.mark.parametrize("shapes", [[(1024, 1024), (1024, 3072), (2048, 1024)], [(1024, 1024)]])
def test_a_chain_that_ends_in_the_weights_has_no_result(shapes):
    """Per element 2 bytes of updates and 4 for the two sides of the chain, and two squares of the smaller extent; sums, tables, rounding."""
    params, opt = _optimizer(shapes)
    assert _allocated(opt) <= sum(6 * p.numel() + 4 * min(p.shape) ** 2 for p in params) + (2 << 20)


@pytest.mark.parametrize("options", [dict(tile_size=128), dict(tile_size=64), dict(granularity="block")])
def test_what_cannot_go_together_is_refused_before_it_is_prepared(options):
    """A gradient that is no row-major matrix is copied once: per element 4 bytes of it, 2 of updates, 2 of the result, 4 for the two sides of the
    chain, 4 for its two squares."""
    params, opt = _optimizer([(1024, 1024)], **options)
    params[0].grad = (torch.randn(1024, 1024, device="cuda") * 1e-2).t()
    opt.step()
    assert _allocated(opt) <= 16 * (1 << 20) + (1 << 18)
