"""The decode step's Q|K|V GEMV rotates Q and K bit for bit as the prompt's RoPE + append kernel does, so
that a cache row does not depend on which of them wrote it. The GEMV is the library's own function
(no entry point of the C ABI launches it alone)."""
import ctypes

import pytest
import torch

import cdna4
from gpu_util import DEV, ptr, stream

pytestmark = pytest.mark.gpu


def _gemv_qkv():
    fn = cdna4.lib()["_ZN5cdna412llm_gemv_qkvEbPKfPKvS3_fS3_S3_iiiiS1_S1_PvS4_S4_iiP12ihipStream_tPKi"]
    vp, i = ctypes.c_void_p, ctypes.c_int
    fn.restype = i
    fn.argtypes = [ctypes.c_bool, vp, vp, vp, ctypes.c_float, vp, vp, i, i, i, i, vp, vp, vp, vp, vp, i, i, vp, vp]
    return fn


@pytest.mark.parametrize("norm_bias", [False, True])
@pytest.mark.parametrize("H,D,nH,nKV", [(768, 64, 12, 12), (1024, 128, 8, 2)])
def test_step_rotation_equals_the_appends(H, D, nH, nKV, norm_bias):
    g = torch.Generator(device=DEV).manual_seed(H)
    x = torch.randn(H, device=DEV, generator=g)
    gain = (1 + 0.1 * torch.randn(H, device=DEV, generator=g)).half()
    beta = (0.1 * torch.randn(H, device=DEV, generator=g)).half()
    W = (torch.randn((nH + 2 * nKV) * D, H, device=DEV, generator=g) * H ** -0.5).half()
    max_seq, positions = 64, list(range(1, 64, 3))
    cos, sin = cdna4.rope_table_f32(0, max_seq, D, 10000.0)
    gemv = _gemv_qkv()

    def step(cos_t, sin_t, pos):
        q = torch.zeros(nH * D, device=DEV, dtype=torch.float16)
        Kc, Vc = (torch.zeros(nKV, max_seq, D, device=DEV, dtype=torch.float16) for _ in range(2))
        rc = gemv(False, ptr(x), ptr(gain), ptr(beta) if norm_bias else None, 1e-6, ptr(W), None, H, D, nH, nKV,
                  ptr(cos_t[pos]), ptr(sin_t[pos]), ptr(q), ptr(Kc), ptr(Vc), pos, max_seq, stream(), None)
        assert rc == 0
        return q, Kc, Vc

    ones, zeros = torch.ones_like(cos), torch.zeros_like(sin)
    for pos in positions:
        q0, K0, V0 = step(ones, zeros, pos)   # cos 1, sin 0: the projections before the rotation
        q1, K1, V1 = step(cos, sin, pos)
        qa, Ka, Va = torch.zeros_like(q0), torch.zeros_like(K0), torch.zeros_like(V0)
        k, v = K0[:, pos].contiguous(), V0[:, pos].contiguous()
        cdna4.rope_append_kv_f16(q0, k, v, qa, Ka, Va, cos[pos:pos + 1], sin[pos:pos + 1], 1, nH, nKV, D, pos, max_seq)
        torch.cuda.synchronize()
        assert torch.equal(q1, qa) and torch.equal(K1, Ka) and torch.equal(V1, Va), pos
