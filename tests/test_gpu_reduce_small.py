"""The one-launch reduce of small inputs and its edges with the two-launch one: whole-number values, so
that sums are exact in any order, at aligned and odd elements, in a workspace of the returned size."""
import pytest
import torch

import cdna4
from gpu_util import DEV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset", [0, 1, 2, 5])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.int32, torch.int64, torch.float16, torch.bfloat16])
def test_edges_of_the_small_reduce(dtype, offset):
    vec = 16 // dtype.itemsize
    wide = 1024 * vec
    sizes = [1, vec - 1, vec + 1, 1000, wide - 1, wide + vec + 1] + [wide * k + d for k in (8, 16) for d in (-1, 0, 1)]
    ws = torch.full((cdna4.reduce_workspace_size(0, cdna4.F32) + 64,), 0x5A, dtype=torch.uint8, device=DEV)
    for i, n in enumerate(n for n in sizes if n > 0):
        g = torch.Generator(device=DEV).manual_seed(i)
        buf = torch.full((n + offset + 16,), 100, device=DEV, dtype=dtype)   # a value outside must not count
        x = buf[offset:offset + n]
        x.copy_(torch.randint(-9, 10, (n,), device=DEV, generator=g))
        ref = x.to(torch.float64)
        for op, want in (("sum", ref.sum()), ("max", ref.max()), ("min", ref.min())):
            got = cdna4.reduce(x, op, workspace=ws[:-64])
            assert float(got) == float(want), (dtype, n, offset, op)
        assert (ws[-64:] == 0x5A).all()
