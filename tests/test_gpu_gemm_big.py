"""The 256 x 256 and 256 x 128 tiles of the large products (csrc/gemm.hip) against torch fp32 products.

Shapes at the edges of the tiles (one row and one 4-column group past a whole tile, one short of it,
fewer rows than a tile beside whole ones), the shortest K each form takes, odd and even stage counts,
every output form; bounds as in test_gpu_gemm.py."""
import pytest
import torch

import cdna4
from gpu_util import DEV

pytestmark = pytest.mark.gpu


def _operands(M, N, K, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(M, K, device=DEV, generator=g).half(),
            (torch.randn(N, K, device=DEV, generator=g) * K ** -0.5).half())


@pytest.mark.parametrize("M,N,K,out_dtype,accum,tile", [
    (2048, 4096, 4096, torch.float16, False, (256, 128)),
    (4096, 4096, 320, torch.float32, False, (256, 256)),
    (4097, 4100, 384, torch.float32, True, (256, 256)),
    (3839, 4092, 448, torch.float16, True, (256, 256)),
    (2100, 6148, 1024, torch.float16, False, (256, 256)),
    (3000, 2304, 768, torch.float32, True, (256, 128)),
    (2047, 2308, 832, torch.float16, True, (256, 128)),
    (1540, 4100, 320, torch.float32, False, (256, 128)),
])
def test_gemm_big_tiles(M, N, K, out_dtype, accum, tile):
    if torch.cuda.get_device_properties(DEV).multi_processor_count == 256:
        assert cdna4.gemm_f16_nt_tile(M, N, K) == tile
    X, W = _operands(M, N, K, M + N + K)
    ref = X.float() @ W.float().t()
    buf = torch.randn(M + 1, N + 8, device=DEV).to(out_dtype)   # a guard row and guard columns
    Y0 = buf.clone()
    out = buf[:M, :N]
    if accum:
        ref = ref + Y0[:M, :N].float()
    cdna4.gemm_f16_nt(X, W, out=out, accum=accum, out_dtype=out_dtype)
    torch.cuda.synchronize()
    scale = max(1.0, ref.abs().max().item())
    tol = 1e-5 * scale if out_dtype == torch.float32 else 1e-5 * scale + 2.0 ** -11 * scale
    assert (out.float() - ref).abs().max().item() <= tol
    assert torch.equal(buf[M:], Y0[M:]) and torch.equal(buf[:, N:], Y0[:, N:])


@pytest.mark.parametrize("M,F,K,tile", [
    (4096, 2052, 128, (256, 256)), (1025, 8196, 128, (256, 256)), (2047, 3068, 192, (256, 256)),
    (1024, 3072, 768, (256, 128)), (700, 4100, 1024, (256, 128)), (511, 7748, 256, (256, 128)),
])
def test_gemm_silu_big_tiles(M, F, K, tile):
    if torch.cuda.get_device_properties(DEV).multi_processor_count == 256:
        assert cdna4.gemm_f16_nt_silu_tile(M, F, K) == tile
    X, W = _operands(M, 2 * F, K, M + F + K)
    g, u = X.float() @ W[:F].float().t(), X.float() @ W[F:].float().t()
    ref = g / (1 + torch.exp(-g)) * u
    got = cdna4.gemm_f16_nt_silu(X, W)
    torch.cuda.synchronize()
    s = max(1.0, g.abs().max().item() * max(1.0, u.abs().max().item()))
    assert ((got.float() - ref).abs() - 2.0 ** -11 * ref.abs()).max().item() <= 1e-5 * s
