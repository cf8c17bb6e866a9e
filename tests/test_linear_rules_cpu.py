"""Which products of prompts and fine-tunes run in own tiles (ops/linear.py): the
sizes that were measured to be faster there, and those that were not."""
import pytest

from runbooks_amd.ops import linear


@pytest.mark.parametrize("m,n,k,tiles", [
    (129, 12288, 4096, True), (256, 12288, 3072, True),
    (320, 12288, 4096, True), (256, 15360, 5120, True),
    (192, 18432, 2048, True),
    (320, 12288, 1024, False), (320, 15360, 5120, False),
    (320, 24576, 1024, False), (129, 24576, 8192, False),
    (257, 32768, 4096, False), (321, 12288, 4096, False),
    (200, 6144, 4096, False)])
def test_wide_products(m, n, k, tiles):
    assert linear._wide_in_tiles(m, n, k) is tiles


@pytest.mark.parametrize("m,n,k,parts", [
    (129, 4096, 4096, True), (512, 4096, 11008, True),
    (300, 3584, 3584, True), (400, 2048, 5632, True),
    (129, 2048, 2048, False), (400, 2048, 2048, False),
    (1021, 1024, 1024, False), (129, 1024, 2816, False),
    (768, 4096, 4096, False), (4096, 4096, 14336, False)])
def test_sums_in_parts(m, n, k, parts):
    pytest.importorskip("runbooks_amd.ops._hip_core")
    assert linear._sums_in_parts(m, n, k) is parts


@pytest.mark.parametrize("m,n,k,tiles", [
    (129, 12288, 4096, True), (2048, 22016, 4096, True),
    (256, 6144, 4096, True), (2048, 4096, 4096, True),
    (1800, 2048, 2048, True), (2048, 4096, 11008, True),
    (3001, 4096, 14336, True), (1024, 8192, 8192, True),
    (3001, 28672, 4096, False), (512, 4096, 4096, False),
    (1024, 2048, 5632, False), (1280, 4096, 11008, False),
    (1536, 4096, 14336, False), (1800, 768, 3072, False),
    (700, 8192, 28672, False), (2048, 8192, 8192, False),
    (128, 22016, 4096, False)])
def test_products_with_adapters(m, n, k, tiles):
    assert linear._lora_in_tiles(m, n, k) is tiles


@pytest.mark.parametrize("m,n,k,tiles", [
    # one round of 256 x 256: columns that are a multiple of 256 and others
    (1021, 12288, 3072, True), (512, 12288, 4096, True), (400, 10240, 4096, True),
    (900, 4096, 4096, True), (1280, 4096, 4096, False), (640, 8192, 3072, False),
    (330, 8192, 4096, False), (2048, 6144, 4096, True), (640, 8256, 3072, True),
    (1280, 4160, 4096, True),
    # small tiles of short sums
    (1280, 2048, 2048, True), (330, 5120, 4096, False),
    # more rounds
    (900, 18432, 8192, True), (7931, 6144, 4096, False), (7931, 6208, 4096, True),
    (2048, 8192, 2560, False), (2500, 12288, 6144, True),
    (2500, 12288, 6208, False), (2048, 9216, 4096, False),
    # narrow, short, and past what was measured
    (10300, 256, 1024, True), (10300, 248, 1024, False), (16384, 16, 256, False),
    (24576, 12288, 512, True), (24577, 12288, 512, False),
    (2048, 20480, 256, True), (2048, 20736, 256, False), (2048, 12288, 192, False)])
def test_wide_products_of_many_rows(m, n, k, tiles):
    pytest.importorskip("runbooks_amd.ops._hip_core")
    assert linear._many_in_tiles(m, n, k) is tiles


@pytest.mark.parametrize("m,n,k,tiles", [
    (2048, 4096, 22016, True), (512, 4096, 22016, True), (300, 4096, 12288, True),
    (2048, 11008, 4096, True), (3001, 14336, 4096, True),
    # a few rows, narrow columns
    (32, 4096, 4096, False), (33, 4096, 4096, True), (33, 768, 8192, False),
    (129, 256, 4096, False), (2048, 16, 4096, False), (2048, 64, 4096, True),
    # small results of short sums
    (300, 1024, 1024, False), (300, 1024, 512, True), (400, 2048, 2048, False),
    (700, 2048, 2048, True),
    # few tiles, and enough
    (1100, 4096, 4096, False), (2304, 4096, 17408, False),
    (3001, 4096, 28672, True),
    # past what was measured
    (24577, 4096, 4096, False), (2048, 4096, 57408, False)])
def test_gradients_of_inputs(m, n, k, tiles):
    ext = pytest.importorskip("runbooks_amd.ops._hip_core")
    assert ext.tile_gemm_down_pays(m, n, k) is tiles
