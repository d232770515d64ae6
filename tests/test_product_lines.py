"""Where prompts' products take this repository's kernel: the line is a function of
their sizes, and sides of it were measured with weights in turn from memory."""
import pytest

ext = pytest.importorskip("polyrl_amd._hip")


@pytest.mark.parametrize("m,n,k", [
    # (tiles of 96 rows whose weights come from memory)
    (1024, 4096, 14336), (600, 8192, 28672), (560, 8192, 8192), (3072, 1536, 8960),
    (768, 6144, 4096), (3072, 2048, 8192),
    # (few of 128 rows, three rounds of them, rounds that they leave empty)
    (1024, 6144, 4096), (1024, 8192, 28672), (4096, 6144, 4096), (16384, 1536, 8960),
    (4096, 1536, 8960),
    # (whole tiles of 256 rows)
    (4096, 4096, 4096), (8192, 3584, 3584), (16384, 3584, 3584)])
def test_library(m, n, k):
    assert not ext.linear_rows_pays(m, n, k)


@pytest.mark.parametrize("m,n,k", [
    (5135, 1024, 4096), (2300, 2048, 2048), (1800, 3072, 2048), (2048, 4096, 4096),
    (5135, 1536, 8960), (4096, 2048, 8192), (1400, 8192, 28672), (4096, 3584, 18944),
    (5135, 4096, 14336), (6145, 2048, 2048)])
def test_kernel(m, n, k):
    assert ext.linear_rows_pays(m, n, k)


def test_row_parts():
    """Tiles of as many rows as end the last round of 256 earliest."""
    for parts in range(3, 9):
        rows, cost = ext.product_rows(8192 * parts - 17, 1, 4096, 3)
        assert rows == parts and cost > 0
    for bad in ((0, 1, 64, 3), (1, 0, 64, 3), (1, 1, 0, 3), (1, 1, 64, 9)):
        with pytest.raises(RuntimeError):
            ext.product_rows(*bad)
