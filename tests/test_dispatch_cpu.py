"""Dispatch rules of the layers that are plain arithmetic on sizes, on the CPU."""
import pytest

import _lib
import bgemm_linear as bl

F32, F16, BITS_F32 = _lib.OUT_F32_SCALED, _lib.OUT_F16_SCALED, _lib.OUT_BITS_F32


@pytest.mark.parametrize("batch, N, M, D, ahead", [
    (1, 1, 1, 32, True), (64, 2048, 2048, 64, True), (1, 2049, 8, 32, False), (1, 8, 2049, 32, False), (1, 2048, 2048, 128, True),
    # measured on both sides of the limit on D > 96, which D = 96 does not know
    (16, 1536, 1536, 128, True), (64, 1024, 1024, 128, False), (16, 2048, 2048, 128, False), (64, 1536, 1536, 96, True), (64, 1536, 1536, 128, False),
    (11, 2048, 2048, 128, True), (12, 2048, 2048, 128, False), (12, 2047, 2048, 128, True)])
def test_scores_gradients_go_where_they_are_ahead(batch, N, M, D, ahead):
    assert bl._scores_grad_ahead(batch, N, M, D) is ahead


@pytest.mark.parametrize("N, M, K, kind, ahead", [
    # columns, K-tiles and rows of the lines; numbers of which there are more than the caches hold, on rows that share lines and on others
    (1, 4096, 512, F32, True), (32, 4096, 513, F32, False), (33, 4096, 1024, F16, True), (511, 4096, 1536, F16, False), (2048, 4096, 2048, F32, True),
    (2047, 4096, 2048, F32, False), (1024, 16384, 256, F16, True), (1024, 16385, 256, F16, False), (255, 16385, 256, F16, True),
    (16384, 3000, 768, F32, False), (16384, 3000, 769, F32, True), (16384, 6000, 512, F32, False), (16384, 6000, 513, F32, True), (8192, 4100, 128, F32, True),
    (10240, 4096, 256, F32, True), (10240, 4100, 256, F32, False), (16384, 8192, 128, F32, True), (16384, 3000, 128, F16, True), (16384, 3000, 128, BITS_F32, True)])
def test_one_launch_layers_go_where_they_are_ahead(N, M, K, kind, ahead):
    assert _lib.lib().bgemm_linear_rows_supported(N, M, K, 1, kind) == (2 if ahead else 1)
