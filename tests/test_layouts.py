"""Layout plans of the host layer (CPU): which calls read an array as it lies,
and that the plan addresses the elements the general path would."""

from __future__ import annotations

import itertools

import torch

from numbagg_amd.decorators import _inner_split


def _gather(t, plan):
    """(outer * cols, n) of the elements the plan addresses."""
    outer, n, cols, ld_outer, ld_row = plan
    return torch.as_strided(t, (outer, n, cols), (ld_outer, ld_row, 1), t.storage_offset()).movedim(1, -1).reshape(-1, n)


def test_inner_split_matches_the_general_path():
    base = torch.arange(4 * 12 * 5 * 60).view(4, 12, 5, 60)
    views = [base, base[:, ::2], base[..., 3:], base[:, :, 1], base.transpose(1, 2), base.permute(3, 0, 1, 2),
             base.permute(2, 3, 0, 1), base[:1], base[:, :, :1], base[:, 3:4].expand(4, 7, 5, 60), base[0].t() if
             base[0].dim() == 2 else base[0, 0].t(), base[0, :, 2], base[0, :, 2].t()]
    planned = 0
    for t in views:
        for r in range(1, t.dim() + 1):
            for axes in itertools.permutations(range(t.dim()), r):
                plan = _inner_split(t, axes)
                if plan is None:
                    continue
                planned += 1
                moved = t.movedim(axes, tuple(range(t.dim() - r, t.dim())))
                n = 1
                for a in axes:
                    n *= t.shape[a]
                assert plan[1] == n
                assert torch.equal(_gather(t, plan), moved.reshape(-1, n)), (t.shape, t.stride(), axes)
    assert planned > 30
    # the innermost axis, a broadcast axis, an empty array and a scalar stay on the general path
    assert _inner_split(base, (3,)) is None
    assert _inner_split(base[:, 3:4].expand(4, 7, 5, 60), (1,)) is None
    assert _inner_split(base[:0], (1,)) is None
    assert _inner_split(torch.zeros(()), ()) is None
    assert _inner_split(base, (1,)) == (4, 12, 300, 3600, 300)
