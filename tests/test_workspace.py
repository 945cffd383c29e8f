"""The backward's single workspace: every buffer aligned, inside the allocation
and apart from the others."""
import torch

from pack3d_amd import _lib


def test_workspace_buffers_are_aligned_and_disjoint():
    work, sizes = _lib.Workspace(), {"a": (3, 2), "empty": (0, 4), "b": (64, 4), "c": (1, 4), "d": (1000, 2)}
    for name, (count, itemsize) in sizes.items():
        work.take(name, count, itemsize)
    at = work.allocate(torch.device("cpu"))
    base, end = work.memory.data_ptr(), work.memory.data_ptr() + work.memory.numel()
    spans = sorted((at[n] - base, at[n] - base + c * s) for n, (c, s) in sizes.items())
    assert all(lo % 256 == 0 and base + hi <= end for lo, hi in spans)
    assert all(hi <= lo for (_, hi), (lo, _) in zip(spans, spans[1:]))
