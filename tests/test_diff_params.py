"""The material records a differentiable render writes from its parameters (no GPU)."""
from __future__ import annotations

import pytest
import torch

import gknextengine_amd as gk
from gknextengine_amd import diff
from gknextengine_amd.scenes import material


@pytest.mark.parametrize("n", [0, 1, 4, 257])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_records_equal_field_by_field_writes(n, dtype):
    g = torch.Generator().manual_seed(n)
    base = [material(tuple(torch.rand(3, generator=g).tolist())) for _ in range(n)]
    for i, m in enumerate(base):
        m.refraction_index, m.diffuse_texture_id, m.diffuse[3] = 1.0 + i, i - 1, 0.25 * i
    before = [bytes(m) for m in base]
    p = torch.randn(n + 2, 5, generator=g, dtype=dtype)  # rows past the materials are not read
    if n:
        p[0, 0], p[0, 4] = float("inf"), float("nan")
    got = diff._materials(base, p)
    assert len(got) == n and [bytes(m) for m in base] == before
    q = p.to(torch.float32)
    for i in range(n):
        want = gk.Material.from_buffer_copy(base[i])
        for k in range(3):
            want.diffuse[k] = float(q[i, k])
        want.fuzziness, want.metalness = float(q[i, 3]), float(q[i, 4])
        assert bytes(got[i]) == bytes(want), i
    if n:
        with pytest.raises(IndexError):
            diff._materials(base, p[:n - 1])
