"""Dequantisation kernels (rwkv-infer-next_amd/csrc/w6a16.hip) at their edges, equal to s q rounded once: ragged columns,
one chunk, chunks that do not fill a workgroup, batches, a zero scale and, through the C ABI, an output address that
allows no vector stores."""
import ctypes

import numpy as np
import pytest

from gpu_util import say

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from test_gpu_int6 import DEV, R, _dev, _weights  # noqa: E402


def _expected(lo, hi, sc, g, dtype):
    q = torch.from_numpy(R.unpack_codes(np.asarray(lo), np.asarray(hi)).astype(np.float32) - 32)
    s = torch.from_numpy(np.asarray(sc).astype(np.float32)).repeat_interleave(g, dim=-2)
    return (s * q).to(dtype)


@pytest.mark.parametrize("B,K,N,g", [(1, 64, 16, 64), (1, 192, 144, 64), (2, 320, 2064, 64), (1, 256, 400, 256)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_dequantise_bits(B, K, N, g, dtype):
    from rwkv_next_amd import _lib
    from rwkv_next_amd.kernels import int6_gemm as I6
    say("dequantise", dict(B=B, K=K, N=N, g=g, dtype=str(dtype)))
    rng = np.random.default_rng(500 + K + N)
    lo, hi, sc = _weights(rng, B, K, N, g)
    sc[:, 0, 5] = 0
    want = _expected(lo, hi, sc, g, dtype)
    Ld, Hd, Sd = _dev(lo, hi, sc)
    pk = I6.prepack_int6(Ld, Hd, Sd, g)
    off = torch.zeros(B * K * N + 3, dtype=dtype, device=DEV)
    code = {torch.bfloat16: _lib.W6A16_OUT_BF16, torch.float16: _lib.W6A16_OUT_F16, torch.float32: _lib.W6A16_OUT_F32}[dtype]
    _lib.check(_lib.load().w6a16_dequantize_packed(
        ctypes.c_void_p(pk.weight.data_ptr()), ctypes.c_void_p(pk.scales.data_ptr()),
        ctypes.c_void_p(off.data_ptr() + want.element_size()), B, K, N, g, K * N, code,
        torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    for got in (I6.dequantize_int6(Ld, Hd, Sd, g, dtype=dtype), I6.dequantize_int6_packed(pk, dtype=dtype),
                off[1:-2].view(B, K, N)):
        got = got.reshape(B, K, N).cpu().contiguous()
        assert torch.equal(got, want)
    assert float(off[0]) == 0 and float(off[-1]) == 0 and float(off[-2]) == 0
