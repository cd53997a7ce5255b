"""Which fp32 products with few rows and which LSTM layers go to the bf16 matrix pipes."""
import pytest
import torch

from pipedream_amd import ops


@pytest.mark.parametrize("M,N,K,rows_of_k,columns_of_k", [
    (1, 2048, 2056, True, True), (64, 2048, 2056, True, True), (96, 2048, 2056, True, True), (97, 2048, 2056, False, True),
    (128, 3072, 2048, False, True), (97, 4096, 2048, True, True), (128, 4104, 1024, True, True), (128, 4096, 1032, False, True), (128, 6000, 1000, True, True), (128, 4096, 2048, True, True), (129, 4096, 4096, False, False),
    (8, 2048, 2048, False, False), (128, 1024, 1024, False, False), (8, 4096, 2052, False, False), (8, 10, 1024, False, False)])
def test_rows_and_weights(M, N, K, rows_of_k, columns_of_k):
    a, b = torch.empty(M, K), torch.empty(N, K)
    assert ops._use_skinny_x6(M, N, K, False, True, a, b, K, K) == rows_of_k
    assert ops._use_skinny_x6(M, N, K, False, False, a, b.t().contiguous(), K, N) == columns_of_k
    assert not ops._use_skinny_x6(M, N, K, True, True, a, b, K, K)


@pytest.mark.parametrize("M,k_of_rows,k_of_columns", [(1, 64, 64), (16, 64, 64), (17, 128, 128), (64, 128, 128), (65, 384, 256),
                                                      (96, 384, 256), (97, 768, 256), (128, 768, 256)])
def test_short_reductions(M, k_of_rows, k_of_columns):
    """The shortest reduction, whatever the number of weights."""
    for trans_b, least in ((True, k_of_rows), (False, k_of_columns)):
        for K in (least - 8, least):
            N = (1 << 24) // K // 8 * 8
            a, b = torch.empty(M, K, device="meta"), torch.empty(*((N, K) if trans_b else (K, N)), device="meta")
            assert ops._use_skinny_x6(M, N, K, False, trans_b, a, b, K, b.stride(0)) == (K == least)


@pytest.mark.parametrize("T,B,H,takes", [(1, 8, 64, False), (2, 8, 64, True), (2, 128, 256, True), (2, 8, 512, False), (3, 8, 512, True), (2, 8, 768, False), (3, 8, 768, True), (3, 8, 800, False),
                                         (3, 40, 1024, False), (4, 40, 1024, True), (4, 40, 1056, False), (5, 40, 1056, True), (5, 129, 1024, False), (5, 40, 1000, False)])
def test_lstm_steps(T, B, H, takes):
    w = torch.empty(4 * H, H)
    assert ops._lstm_x6(T, B, H, w) == takes
    assert not ops._lstm_x6(T, B, H, torch.empty(4 * H, 2 * H)[:, :H])
