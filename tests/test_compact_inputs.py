"""Retained indices of every integer width, and page ids of every size, as the compaction takes them (CPU)."""
import pytest
import torch

from unifiedkv_amd import compaction


@pytest.mark.parametrize("dtype", [torch.uint8, torch.int8, torch.int16, torch.int32, torch.int64])
@pytest.mark.parametrize("n_pages", [101, 300, 100000])
def test_indices_are_checked_wider_than_their_type(dtype, n_pages):
    keep = torch.tensor([[0, 50, 100]] * 2, dtype=dtype)  # inside every list, whatever the type wraps to
    got = compaction._keep_ids(keep, n_pages, torch.device("cpu"), "t")
    assert got.dtype == torch.int32 and torch.equal(got, keep.to(torch.int32))


@pytest.mark.parametrize("value", [-1, 300, 2 ** 32, 2 ** 32 + 5])
def test_wide_indices_are_refused_before_they_are_narrowed(value):
    with pytest.raises(ValueError, match=r"outside \[0, 300\)"):
        compaction._keep_ids(torch.tensor([[0, value]]), 300, torch.device("cpu"), "t")


@pytest.mark.parametrize("bad", [-1, 10, 2 ** 31, 2 ** 40, 2 ** 63, 2 ** 70, -2 ** 70])
def test_page_ids_of_any_size_are_refused_alike(bad):
    class Pool:
        N_total = 10

    with pytest.raises(ValueError, match="outside the pool"):
        compaction._check_pool_ids(Pool, [1, bad, 2], "t")
    assert [int(x) for x in compaction._check_pool_ids(Pool, [1.0, 9], "t")] == [1, 9]
