"""The GEMM of up to 16 rows (gemm_rows) against fp64 and at the edges of its rule: rows 1 to 17, ragged
columns, K of four stages and more than the waves divide evenly, strided outputs and accumulation."""
import pytest
import torch

import cdna4
from gpu_util import DEV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["f16", "f16_accum", "f32", "f32_accum", "silu"])
@pytest.mark.parametrize("M,N,K", [(1, 4, 256), (16, 20, 256), (3, 100, 320), (7, 1028, 832), (16, 4096, 2112),
                                   (15, 768, 3072), (17, 100, 320), (16, 100, 192), (16, 4100, 256)])
def test_few_rows(M, N, K, kind):
    g = torch.Generator(device=DEV).manual_seed(M * 31 + N + K)
    X = torch.randn(M, K, device=DEV, generator=g).half()
    W = (torch.randn((2 if kind == "silu" else 1) * N, K, device=DEV, generator=g) / K ** 0.5).half()
    dt = torch.float32 if kind.startswith("f32") else torch.float16
    buf = torch.randn(M, N + 8, device=DEV, generator=g).to(dt)
    before, out = buf.clone(), buf[:, :N]
    rows = M <= 16 and K >= 256 and N <= 4096
    P = X.double() @ W.double().t().contiguous()
    if kind == "silu":
        if torch.cuda.get_device_properties(0).multi_processor_count == 256:
            assert (cdna4.gemm_f16_nt_silu_tile(M, N, K) == (16, 32)) == rows
        cdna4.gemm_f16_nt_silu(X, W, out=out)
        ref = torch.nn.functional.silu(P[:, :N]) * P[:, N:]
    else:
        if torch.cuda.get_device_properties(0).multi_processor_count == 256:
            assert (cdna4.gemm_f16_nt_tile(M, N, K) == (16, 16)) == rows
        cdna4.gemm_f16_nt(X, W, out=out, accum="accum" in kind)
        ref = P + (before[:, :N].double() if "accum" in kind else 0)
    # Products of order one summed in fp32 (K eps at most, far less met), silu's product of two such sums;
    # then one rounding to fp16.
    mag = float(ref.abs().max()) + float(P.abs().max()) ** (2 if kind == "silu" else 1)
    tol = K * 2.0 ** -24 * mag + (0 if dt == torch.float32 else 2.0 ** -11 * float(ref.abs().max()))
    assert float((out.double() - ref).abs().max()) <= tol
    assert torch.equal(buf[:, N:], before[:, N:])
