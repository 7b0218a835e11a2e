"""Device memory of a solver: state blocks (16 bytes per element of main_size)."""
import pytest
import torch

import libheom_amd as H
from libheom_amd import configs

pytestmark = pytest.mark.gpu


# complex128: y, y_new, two stage inputs, k_2..k_5 (the error sum in k_2's place), D of
# y and of y_new.  complex64: half blocks but for y, y_new and the error sum, and FP32
# copies of y and y_new.  The margin of 0.3 blocks (37 MB) holds the 2 MB of partials
# and the rounding of each of the 12 allocations to 2 MB.
@pytest.mark.parametrize("dtype,blocks", [("complex128", 10.0), ("complex64", 7.5)])
def test_rkdp_state_blocks(dtype, blocks):
    m = configs.random_model(12, 3, 5, 6, seed=1, dense_v=False)
    eng = H.hip(0)
    q = H.heom_hilb(6, dtype=dtype).load(m, eng)
    block = 16 * q.main_size()
    assert block > 120e6
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    s = H.qme_solver(eng, q, H.rkdp())
    used = before - torch.cuda.mem_get_info()[0]
    assert blocks - 0.1 <= used / block <= blocks + 0.3
    del s
