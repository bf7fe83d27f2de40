"""Rules by size: the forms that measuring found faster, on both sides of the lines."""
import pytest

from llmctl.ops import functional as F


@pytest.mark.parametrize("T,H,V,pays", [(8192, 64, 256, True), (16384, 64, 256, True), (24576, 64, 32000, False), (24576, 4096, 32000, True), (32768, 128, 50304, False),
                                        (32768, 1024, 32000, True), (50000, 1024, 50304, False), (50000, 2048, 50304, True), (65536, 64, 32000, False),
                                        (65536, 4096, 32000, True), (65537, 4096, 32000, False)])
def test_embedding_gradients(T, H, V, pays):
    assert F.embed_grad_pays(T, H, V) == pays
