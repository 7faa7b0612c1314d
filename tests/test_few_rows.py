"""Which dense products go through the streaming kernel for few rows, on the CPU."""
import pytest
import torch

from inferx_amd.engine.runtime import Runtime


@pytest.mark.parametrize("dtype,rows,features,reduction,off,streamed", [
    (torch.float32, 1, 8, 8, 0, True), (torch.float32, 32, 8, 8, 0, True), (torch.float32, 33, 8, 8, 0, False),
    (torch.float32, 4, 8, 6, 0, False), (torch.float32, 4, 8, 8, 1, False), (torch.float32, 4, 8, 8, 4, True),
    (torch.float32, 4, 0, 8, 0, False), (torch.float32, 4, 8, 0, 0, False), (torch.float32, 0, 8, 8, 0, False),
    (torch.bfloat16, 9, 8, 8, 0, True), (torch.bfloat16, 32, 8, 16, 0, True), (torch.bfloat16, 33, 8, 16, 0, False),
    (torch.bfloat16, 4, 8, 12, 0, False)])
def test_products_of_few_rows(dtype, rows, features, reduction, off, streamed):
    rt = Runtime.__new__(Runtime)  # (a whole one needs the HIP library)
    x = torch.zeros(off + rows * reduction, dtype=dtype)[off:].view(rows, reduction)
    w = torch.zeros(features, reduction, dtype=dtype)
    assert rt._skinny_ok(x, w) == streamed
    assert not rt._skinny_ok(x, w.to(torch.float64))
