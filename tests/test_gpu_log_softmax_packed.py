"""The resident schedule for many rows of 16-bit logits (two rows per CU) against the two-launch schedule: same bits."""
import pytest
import torch

from llm_reproducibility_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("cols", [4, 1000, 4096, 4100, 114684, 114688, 114692, 151936, 154624])
def test_widths_around_the_register_and_lds_parts(dev, dtype, cols):
    """Less than a segment, whole segments, a ragged one, the end of the register part (28 segments), the longest row."""
    print("case packed log_softmax", dtype, cols, flush=True)
    rows = 259
    x = (torch.randn((rows, cols), generator=torch.Generator(device=dev).manual_seed(cols), device=dev) * 3).to(dtype)
    x[1] = -7.0                                               # a constant row: -log(cols)
    for softmax, to_float in ((False, False), (False, True), (True, False)):
        big = ops.bi_log_softmax(x, softmax, to_float)
        for r0 in (0, 128, rows - 3):
            assert torch.equal(ops.bi_log_softmax(x[r0:r0 + 3], softmax, to_float), big[r0:r0 + 3]), (softmax, to_float, r0)
    got = ops.bi_log_softmax(x, False, True)[:4].cpu().double()
    assert (got - torch.log_softmax(x[:4].cpu().double(), -1)).abs().max() < 2e-5     # the tolerance of the other widths' tests
