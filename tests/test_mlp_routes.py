"""The GEMM where its shape moves it to another kernel or tile: products less
deep than a chunk, with many outputs or few rows, and tiles of 128 rows where
few or many of them lie past the last row.  Checked as in test_mlp_tiles.py."""
import pytest

from test_mlp_tiles import test_gemm_tiles as _check

gpu = pytest.mark.gpu


@gpu
@pytest.mark.parametrize('M,N,K', [(1030, 3713, k) for k in (63, 64, 79, 80, 129)] + [(40, 130, 33), (63, 200, 81),
                         (64, 33001, 81), (66, 33001, 130), (1900, 1100, 65), (1920, 1100, 97), (190, 16500, 100)])
def test_gemm_routes(M, N, K):
    _check(M, N, K)
