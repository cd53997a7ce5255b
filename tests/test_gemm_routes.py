"""Which fp32 products with few rows and which LSTM layers go to the bf16 matrix pipes."""
import pytest
import torch

from pipedream_amd import ops


@pytest.mark.parametrize("M,N,K,rows_of_k,columns_of_k", [
    (1, 2048, 2056, True, True), (64, 2048, 2056, True, True), (96, 2048, 2056, True, True), (97, 2048, 2056, False, True),
    (128, 3072, 2048, False, True), (97, 4096, 2048, True, True), (128, 4096, 2048, True, True), (129, 4096, 4096, False, False),
    (8, 2048, 2048, False, False), (128, 1024, 1024, False, False), (8, 4096, 2052, False, False), (8, 10, 1024, False, False)])
def test_rows_and_weights(M, N, K, rows_of_k, columns_of_k):
    a, b = torch.empty(M, K), torch.empty(N, K)
    assert ops._use_skinny_x6(M, N, K, False, True, a, b, K, K) == rows_of_k
    assert ops._use_skinny_x6(M, N, K, False, False, a, b.t().contiguous(), K, N) == columns_of_k
    assert not ops._use_skinny_x6(M, N, K, True, True, a, b, K, K)


@pytest.mark.parametrize("T,B,H,takes", [(1, 8, 64, False), (2, 8, 64, True), (2, 128, 256, True), (2, 8, 512, False), (3, 8, 512, True),
                                         (4, 40, 1024, False), (5, 40, 1024, True), (5, 129, 1024, False), (5, 40, 1000, False)])
def test_lstm_steps(T, B, H, takes):
    w = torch.empty(4 * H, H)
    assert ops._lstm_x6(T, B, H, w) == takes
    assert not ops._lstm_x6(T, B, H, torch.empty(4 * H, 2 * H)[:, :H])
