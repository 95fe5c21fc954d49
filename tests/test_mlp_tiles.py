"""The tiled GEMM at the edges of its tiles, chunks and load widths, in every
operand layout it takes: against the BF16 oracle, and bit for bit against the
kernel for arbitrary strides (the same products in the same order).

Tolerance against the oracle: FP32 accumulation of K products, as for the
layouts of test_mlp.py (1e-5 sqrt(K) of the largest entry)."""
import numpy as np
import pytest

from oracle import mlp_oracle as MO

gpu = pytest.mark.gpu

# 32 x 32 tiles (few of them), 64 x 64 tiles (at least as many as compute units), 128 x 64 tiles (twice as many)
SIZES = [(1, 1, 1), (31, 33, 7), (32, 32, 128), (33, 65, 129), (65, 30, 263), (5, 130, 1031), (130, 5443, 67),
         (1030, 3713, 9)]


@gpu
@pytest.mark.parametrize('M,N,K', SIZES)
def test_gemm_tiles(M, N, K):
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    from vulcan_amd import _lib
    from vulcan_amd.device import dptr, stream_handle
    from vulcan_amd.mlp import to_bf16
    lib = _lib.load()
    rng = np.random.default_rng(M + N + K)
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = rng.standard_normal((K, N)).astype(np.float32)
    bias = torch.as_tensor(rng.standard_normal(N).astype(np.float32), device='cuda')
    start = torch.as_tensor(rng.standard_normal((M, N + 3)).astype(np.float32), device='cuda')
    ref = MO.bf16(A) @ MO.bf16(B) + bias.cpu().numpy() + start.cpu().numpy()[:, :N]

    def gemm(Ad, sa, Bd, sb):
        C = start.clone()                           # accumulated into, row stride N + 3
        Y = torch.zeros((M, N + 1), dtype=torch.int16, device='cuda')
        _lib.check(lib.vk_mlp_gemm(M, N, K, dptr(Ad), sa[0], sa[1], dptr(Bd), sb[0], sb[1], dptr(C), N + 3, dptr(bias),
                                   1, dptr(Y), N + 1, stream_handle()), 'vk_mlp_gemm')
        return C, Y

    def up(x):
        return to_bf16(torch.as_tensor(np.ascontiguousarray(x), device='cuda'))
    # every second entry of wider arrays: no unit stride on either side
    C0, Y0 = gemm(up(np.repeat(A, 2, axis=1)), (2 * K, 2), up(np.repeat(B, 2, axis=1)), (2 * N, 2))
    assert np.abs(C0.cpu().numpy()[:, :N] - ref).max() <= 1e-5 * np.sqrt(K) * np.abs(ref).max()
    assert torch.equal(C0[:, N:], start[:, N:]) and not Y0[:, N:].any()
    for Ad, sa in ((up(A), (K, 1)), (up(A.T), (1, M))):
        for Bd, sb in ((up(B), (N, 1)), (up(B.T), (1, K))):
            C, Y = gemm(Ad, sa, Bd, sb)
            assert torch.equal(C, C0) and torch.equal(Y, Y0), (sa, sb)
