"""The forward's assignment of query rows to workgroups (blocks of rows go to
the XCDs in turn, last rows first) at the row counts where it can go wrong:
below one row per XCD, counts that are no multiple of eight, and both sides of
the block size and of the 256-row rule.  Tolerances as in test_sfa_fwd_gpu."""
import numpy as np
import pytest
import torch

from oracle.sfa import sfa_fwd_bsnd
from tests.helpers import assert_close, dev, sfa_inputs, sparse_indices

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,N1", [(128, 4), (512, 16), (512, 128)])
@pytest.mark.parametrize("S1", [1, 7, 8, 33, 48, 255, 256, 257, 300, 521])
def test_every_row_is_computed_once(S1, D, N1):
    import dsa_triton_ascend_amd as dsa
    print(f"[row order] S1={S1} D={D} N1={N1}", flush=True)
    dtype, K = torch.bfloat16, 8
    q, k, qr, kr = sfa_inputs(1, S1, S1, N1, D, dtype)
    si = sparse_indices(1, S1, S1, K, 1, 3)
    scale = 1.0 / np.sqrt(D + 64)
    got = dsa.sparse_flash_attention_triton(
        dev(q, dtype), dev(k, dtype), None, dev(si, torch.int32), scale_value=scale, query_rope=dev(qr, dtype),
        key_rope=dev(kr, dtype), sparse_mode=3, return_softmax_lse=True)
    torch.cuda.synchronize()
    ref = sfa_fwd_bsnd(q, k, si, qr, kr, scale, [S1], [S1], 1, 3, True, "float32", positions="kernel")
    for g, e, name in zip(got, ref, ("out", "softmax_max", "softmax_sum")):
        assert_close(g.float().cpu().numpy(), e, 2e-2, 2e-3, name)


@pytest.mark.parametrize("S1", [264, 400, 513, 600, 800])
def test_every_row_is_computed_once_in_smaller_blocks(S1):
    """Counts whose blocks of rows are smaller than 32, to keep the XCDs even."""
    test_every_row_is_computed_once(S1, 512, 128)
    test_every_row_is_computed_once(S1, 128, 4)
