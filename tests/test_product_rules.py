"""Rules that choose a product's kernel by the number of rows, on the CPU."""
import pytest
import torch

from microllm_rocm_amd.ops import kernels
from microllm_rocm_amd.parts.linear import Weight, takes_tiled


@pytest.mark.parametrize("from_float", [False, True])
@pytest.mark.parametrize("k", [32, 896, 1024, 1056, 2048, 2080, 3584, 18944])
def test_a_padded_step_takes_the_kernel_of_its_own_rows(k, from_float):
    """Steps are padded to multiples of 64 rows, above 1024 of 256: both counts of every step lie on one side of every line."""
    for rows in range(1, 8193):
        multiple = 64 if rows <= 1024 else 256
        padded = -(-rows // multiple) * multiple
        assert kernels.tiled_gated_pays(rows, k, from_float) == kernels.tiled_gated_pays(padded, k, from_float), rows
    assert not kernels.tiled_gated_pays(2048, k + 8, from_float)       # the tiled kernel's steps of 32


@pytest.mark.parametrize("from_float", [False, True])
@pytest.mark.parametrize("n", [64, 1408, 4096, 9728, 37888, 59136])
@pytest.mark.parametrize("k", [512, 1024, 2048, 2560, 3584, 8192])
def test_a_padded_step_takes_the_kernel_of_its_own_rows_for_every_weight(n, k, from_float):
    for rows in range(1, 8193, 7):
        multiple = 64 if rows <= 1024 else 256
        assert kernels.tiled_gated_pays(rows, k, from_float, n) == kernels.tiled_gated_pays(-(-rows // multiple) * multiple, k, from_float, n), rows


@pytest.mark.parametrize("rows,n,k,pays,clamped", [(2048, 1408, 2048, False, False), (4096, 512, 512, True, True), (512, 512, 512, False, False),
                                                   (2048, 37888, 3584, True, True), (1536, 37888, 3584, True, True), (2048, 59136, 8192, False, True),
                                                   (512, 9728, 896, True, True), (1024, 16384, 2048, True, True), (2048, 17920, 2560, False, True)])
def test_where_the_tiled_kernel_takes_gated_products(rows, n, k, pays, clamped):
    """Weights of few rows and of the longest reductions stay with the library, and clamped gates of those go to the tiled kernel where there are many."""
    assert kernels.tiled_gated_pays(rows, k, False, n) == pays
    assert kernels.tiled_gated_pays(rows, k, True, n) == clamped


@pytest.mark.parametrize("rows,n,k,pays", [(4096, 9728, 896, True), (16384, 9728, 896, True), (4096, 16384, 2048, True), (3200, 37888, 3584, True),
                                           (16301, 37888, 3584, True), (4096, 17920, 2560, True), (4096, 1408, 4096, False), (8192, 59136, 8192, False)])
def test_many_rows_of_gated_products(rows, n, k, pays):
    assert kernels.tiled_gated_pays(rows, k, False, n) == pays


@pytest.mark.parametrize("rows,n,k,pays", [(16301, 37888, 3584, True), (3200, 37888, 3584, True), (500, 37888, 3584, True), (256, 37888, 3584, False), (255, 27648, 5120, True),
                                           (192, 27648, 5120, False), (2560, 14336, 4096, False), (1024, 22016, 4096, False), (2048, 1408, 4096, False),
                                           (4096, 37888, 2080, True), (4096, 28672, 7168, False), (384, 13824, 4096, True),
                                           # few columns leave units idle up to 768 rows: 0.78, 0.95, 1.06; 0.86, 1.00, 1.02; 0.97, 1.05 of the library's time
                                           (384, 8192, 4096, False), (640, 8192, 4096, False), (704, 8192, 4096, True), (384, 9728, 4096, False),
                                           (512, 9728, 4096, False), (576, 9728, 4096, True), (384, 11008, 6144, False), (448, 11008, 6144, True),
                                           (2048, 4096, 4096, True), (2048, 4096, 3072, False), (4096, 4096, 4096, False)])
def test_where_the_tiled_kernel_takes_long_reductions(rows, n, k, pays):
    """By how full its rounds are; a padded step takes the kernel of its own rows."""
    assert kernels.tiled_gated_pays(rows, k, False, n) == pays
    assert not kernels.tiled_gated_pays(rows, k + 8, False, n)
    for count in range(1, 8193, 13):
        multiple = 64 if count <= 1024 else 256
        padded = -(-count // multiple) * multiple
        assert kernels.tiled_gated_pays(count, k, False, n) == kernels.tiled_gated_pays(padded, k, False, n), count


@pytest.mark.parametrize("rows,n,clamped_alone", [(512, 13824, False), (512, 8192, False), (1024, 4096, True)])
def test_a_gated_linear_takes_the_tiled_kernel_by_rule_address_and_library(rows, n, clamped_alone, monkeypatch):
    """What ``takes_tiled`` says, which is what a gated linear asks: the rule, rows at a 16-byte boundary, no tuned library."""
    k = 2304
    weight = Weight(torch.zeros((16, k), dtype=torch.bfloat16), pack=False, gated=True)
    flat = torch.zeros(rows * k + 8, dtype=torch.bfloat16)
    x, apart = (flat[first:first + rows * k].view(rows, k) for first in (0, 1))
    assert not takes_tiled(x, weight)                       # nothing is packed
    weight.packed, weight.out_features = torch.zeros((1, k // 32, 4, 16, 8), dtype=torch.bfloat16), n
    for from_float in (False, True):
        pays = kernels.tiled_gated_pays(rows, k, from_float, n)
        assert pays == (n == 13824 or (clamped_alone and from_float))
        assert takes_tiled(x, weight, from_float) == pays
        assert not takes_tiled(apart, weight, from_float) and not takes_tiled(x.float(), weight, from_float)
        monkeypatch.setattr(kernels, "library_tuning", lambda: True)
        assert not takes_tiled(x, weight, from_float)
        monkeypatch.undo()
