"""The scan's forms by size (scan_layout::spread_u, large_tiles) against exact prefix sums: sizes at
the edges between the forms and of their tiles, inputs at any element, in a workspace of exactly the
returned size, and replays of a captured call on new values."""
import pytest
import torch

import cdna4
from gpu_util import DEV

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.float64, torch.int32, torch.int64, torch.float16, torch.bfloat16]


def values(n, dtype, seed):
    """Values of -1, 0 and 1: every prefix sum below 2^24 is exact in fp32, whatever the order."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randint(-1, 2, (n,), device=DEV, generator=g).to(dtype)


def want(x):
    acc = torch.float32 if x.element_size() == 2 else x.dtype
    return torch.cumsum(x.to(torch.int64), 0).to(acc)


def sizes(dtype):
    vec = 2 if dtype.itemsize == 8 else 4
    group = 64 * vec * (64 if dtype.itemsize == 2 else 32) * (8 if dtype.itemsize == 8 else 4)   # a large one
    line = 256 if dtype.itemsize == 2 else 384
    out = []
    for u, tiles in ((2, 256), (4, 256), (8, 512), (16, 512)):          # the last size of each single-wave form
        out += [64 * vec * u * tiles + d for d in (-vec - 1, 0, 1)]
    if dtype.itemsize == 8:   # the large tiles' range of one round of groups
        out += [group * t + d for t in (128, 256) for d in (-1, 0, 1)]
    return out + [64 * vec * 16 * 1000 + 5, group * (line - 1) - 1, group * (line - 1), group * (line - 1) + 1,
                  group * (line + 7) + vec + 1]


@pytest.mark.parametrize("offset", [0, 1, 3])
@pytest.mark.parametrize("dtype", DTYPES)
def test_edges_between_the_forms(dtype, offset):
    for i, n in enumerate([1, 3, 511, 513] + sizes(dtype)):
        x = values(n + offset, dtype, 40 + i)[offset:]
        need = cdna4.scan_workspace_size(n, {torch.float32: cdna4.F32, torch.float64: cdna4.F64, torch.int32: cdna4.I32,
                                             torch.int64: cdna4.I64, torch.float16: cdna4.F16,
                                             torch.bfloat16: cdna4.BF16}[dtype])
        store = torch.full((need + 256,), 0x5A, dtype=torch.uint8, device=DEV)
        ref = want(x)
        out = torch.full((n + offset + 8,), 77, dtype=ref.dtype, device=DEV)
        got = cdna4.scan_inclusive(x, "sum", out=out[offset:offset + n], workspace=store[:need])
        assert torch.equal(got, ref), (dtype, n, offset)
        assert (out[:offset] == 77).all() and (out[offset + n:] == 77).all() and (store[need:] == 0x5A).all()
        if x.element_size() != 2:
            for op, f in (("max", torch.cummax), ("min", torch.cummin)):
                assert torch.equal(cdna4.scan_inclusive(x, op), f(x, 0)[0]), (dtype, n, offset, op)


@pytest.mark.parametrize("dtype", [torch.float32, torch.int64, torch.float16])
def test_replays_of_a_captured_scan_see_new_values(dtype):
    for n in (700, 30001, 500009, 3000007):
        x, y = values(n, dtype, 1), values(n, dtype, 2)
        ws = torch.zeros(cdna4.scan_workspace_size(n, {torch.float32: cdna4.F32, torch.int64: cdna4.I64,
                                                       torch.float16: cdna4.F16}[dtype]), dtype=torch.uint8, device=DEV)
        buf = x.clone()
        out = cdna4.scan_inclusive(buf, "sum", workspace=ws)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            cdna4.scan_inclusive(buf, "sum", out=out, workspace=ws, check=False)
        for k in range(6):
            src = (x, y)[k % 2]
            buf.copy_(src)
            graph.replay()
            torch.cuda.synchronize()
            assert cdna4.scan_status(ws) == 0
            assert torch.equal(out, want(src)), (dtype, n, k)
            cdna4.scan_inclusive(y, "sum", workspace=ws, check=k % 2 == 0)   # an eager call between replays
