"""Rules by size: the forms that measuring found faster, on both sides of the lines."""
import importlib

import pytest

from llmctl.ops import functional as F
from llmctl.ops import hybrid as H


@pytest.mark.parametrize("T,H,V,pays", [(8192, 64, 256, True), (16384, 64, 256, True), (24576, 64, 32000, False), (24576, 4096, 32000, True), (32768, 128, 50304, False),
                                        (32768, 1024, 32000, True), (50000, 1024, 50304, False), (50000, 2048, 50304, True), (65536, 64, 32000, False),
                                        (65536, 4096, 32000, True), (65537, 4096, 32000, False)])
def test_embedding_gradients(T, H, V, pays):
    assert F.embed_grad_pays(T, H, V) == pays


@pytest.mark.parametrize("M,N,K,stream", [(32, 12288, 256, False), (32, 12288, 512, True), (32, 12288, 1280, False), (24, 12288, 2048, True), (17, 28672, 768, False), (24, 32000, 1024, True),
                                          (32, 128256, 2304, False), (32, 152064, 3072, True), (32, 102400, 256, False), (17, 102400, 256, True), (16, 1024, 5120, False),
                                          (14, 1024, 5120, True), (16, 6144, 7168, False), (16, 6912, 11008, True), (12, 29696, 11008, False), (4, 16384, 8192, True), (5, 16384, 8192, True),
                                          (4, 12288, 8192, False), (8, 3072, 14336, False), (8, 4096, 14336, True), (4, 50304, 11008, False), (4, 24576, 20480, False), (4, 29696, 11008, False),
                                          (1, 2048, 2048, True)])
def test_weight_streams(M, N, K, stream):
    assert F.stream_pays(M, N, K) == stream


@pytest.mark.parametrize("M,N,K,form", [(16, 5120, 512, "stream"), (16, 5152, 512, "skinny"), (8, 4608, 256, "stream"), (8, 512, 768, "skinny"), (8, 768, 768, "stream"), (16, 1536, 10240, "skinny"),
                                        (8, 1280, 11008, "skinny"), (8, 1536, 11008, "stream"), (16, 9248, 384, "skinny"), (16, 9248, 512, "stream"), (8, 9248, 896, "skinny"),
                                        (4, 3648, 1280, "skinny"), (4, 2048, 1280, "stream"), (5, 16384, 8192, "stream"), (16, 2048, 14336, "skinny"), (1, 2304, 768, "skinny")])
def test_forms_of_a_few_rows(M, N, K, form):
    assert F.decode_form(M, N, K) == form


@pytest.mark.parametrize("M,N,K,pays", [(16, 2048, 512, True), (16, 2048, 256, False), (32, 4096, 2048, True), (32, 4096, 1024, False), (32, 2048, 1024, True), (8, 4096, 16384, False),
                                        (17, 4096, 16384, True), (4, 4096, 16384, True), (33, 2048, 2048, False), (16, 4100, 2048, False)])
def test_partial_sums(M, N, K, pays):
    assert H.parts_pay(M, N, K) == pays


@pytest.mark.parametrize("T,N,K,pays", [(2300, 4240, 2048, True), (2300, 4240, 4096, False), (1331, 8256, 4096, False), (1331, 8256, 2048, True), (1800, 10504, 3072, False), (3379, 6200, 2048, False),
                                        (4090, 12008, 2048, True), (1331, 4240, 2048, False), (3379, 6144, 2048, False), (3379, 4240, 1000, False)])
def test_odd_products(T, N, K, pays):
    assert F.odd_pays(T, N, K) == pays


@pytest.mark.parametrize("T,F_,pays", [(1331, 11008, True), (1331, 8192, False), (2911, 8192, True), (300, 28672, False), (500, 11008, False), (700, 11008, True), (1500, 4096, True), (1023, 4096, False),
                                       (1331, 8200, False)])
def test_gated_products(T, F_, pays):
    assert F.ragged_swiglu_pays(T, F_) == pays


@pytest.mark.parametrize("M,N,K,pays", [(50304, 768, 8192, True), (50304, 512, 3072, True), (50304, 768, 2048, False), (50304, 256, 6144, True), (40008, 256, 8192, False), (12008, 512, 3072, False),
                                        (32136, 768, 3072, False), (8200, 2048, 4096, True), (8200, 768, 6144, False), (5000, 4096, 16384, False)])
def test_weight_gradients_of_a_vocabulary(M, N, K, pays):
    assert importlib.import_module("llmctl.exec.linear")._whole_pays(M, N, K) == pays
