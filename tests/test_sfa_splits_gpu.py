"""The forward's token splits in bf16.  Launches with one workgroup per CU round
the split count down; the softmax numerators keep their lo part wherever the
rounded-up count's ranges hold fewer than 256 tokens, as they did in those
ranges.

With hi + lo numerators (16 bits) the output is the exact value but for the
split partials' rounding to fp16, at most 2^-11 of their magnitude, before its
own rounding to bf16, whose steps are 2^-8 to 2^-7 of the value: at most one
value in eight is moved across the middle of a step.  With the hi part alone
each numerator is off by up to 2^-9, and about three in ten are."""
import numpy as np
import pytest
import torch

from oracle.sfa import sfa_fwd_bsnd
from tests.helpers import dev, sfa_inputs, sparse_indices

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,N1,D,K,up", [
    (70, 64, 512, 1000, 0),    # three splits of 334 for four of 250
    (48, 16, 512, 2048, 6),    # five of 410 for six of 342, 200 tokens in each of the six
    (20, 128, 512, 2048, 7),   # seven of 293: six would take an XCD two rounds as well
    (48, 128, 512, 2048, 3),   # two of 1024 for three of 683
    (100, 16, 256, 2048, 3),   # two of 1024 for three of 683
    (70, 128, 256, 1000, 0),
    (70, 16, 128, 1000, 0),    # four of 250: D = 128 rounds up
    (100, 16, 512, 6000, 3),   # two of 3000 for three of 2000, in chunks of 2048 positions
])
def test_numerators_keep_their_lo_part(rows, N1, D, K, up):
    import dsa_triton_ascend_amd as dsa
    print(f"[splits] rows={rows} N1={N1} D={D} K={K}", flush=True)
    dt, S2 = torch.bfloat16, max(3000, K)
    q, k, qr, kr = sfa_inputs(1, rows, S2, N1, D, dt)
    si = sparse_indices(1, rows, S2, K, 1, 0)
    if up:  # 200 tokens in each range of the rounded-up count
        si[..., np.arange(K) % -(-K // up) >= 200] = -1
    scale = 1.0 / np.sqrt(D + 64)
    out, _, _ = dsa.sparse_flash_attention_triton(
        dev(q, dt), dev(k, dt), None, dev(si, torch.int32), scale_value=scale, query_rope=dev(qr, dt),
        key_rope=dev(kr, dt), sparse_mode=0)
    some = [0, rows // 3, rows - 1]
    ref = sfa_fwd_bsnd(q, k, si, qr, kr, scale, [rows], [S2], 1, 0, True, positions="kernel",
                       rows=[(0, r) for r in some], compute_dtype=np.float64)[0]
    got = out.float().cpu().numpy()[0, some]
    exp = torch.from_numpy(ref[0, some]).to(dt).float().numpy()
    differ = float((got != exp).mean())
    print(f"[splits] {differ:.3g} of the outputs differ from the exact value's rounding", flush=True)
    assert differ < 0.125
