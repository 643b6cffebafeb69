"""The rules by which sizes choose a kernel, at the sizes where both sides were measured; no GPU."""
import pytest
import torch

from infinilm_amd import kernels as K

DEV = torch.device("cuda", 0)


@pytest.fixture(autouse=True)
def chip(monkeypatch):
    monkeypatch.setattr(K, "_num_cus", lambda device: 256)


@pytest.mark.parametrize("M,N,k,span", [(8, 1024, 4096, 1024), (16, 8192, 8192, 1024), (1, 4096, 4608, 1024), (8, 1023, 8192, 4096), (8, 4096, 8200, 4096),
                                        (17, 4096, 4096, 4096), (8, 8200, 4096, 4096), (1, 12288, 2048, 4096), (8, 12288, 8192, 4096),
                                        (16, 32768, 5120, 4096)])
def test_parts_of_a_few_rows_product(M, N, k, span):
    assert K._few_span(M, N, k) == span
