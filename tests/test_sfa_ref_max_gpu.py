"""Scores far above a row's first tokens, whose maximum is the reference of its
softmax numerators, in every kernel of the forward: 20 and 60 binades pass
fp16's range (2^16) and stay below the bf16 limit of 64.  The large token lies in
the second or a later tile, or there is one in the first tile too.

One token holds nearly all of the softmax, so the numerators' rounding (2^-9 in
bf16) does not average out: it bounds the output's error by 2^-9 max |v| (its
own rounding is inside rtol), and the sums are fp32."""
import numpy as np
import pytest
import torch

from oracle.sfa import sfa_fwd_bsnd
from tests.helpers import assert_close, dev, sfa_inputs

pytestmark = pytest.mark.gpu

# rows, heads, D, selected tokens, test flags
ROUTES = {"few4": (130, 32, 512, 1024, 0), "few4_16": (130, 16, 512, 1024, 0), "few1": (800, 32, 512, 1024, 0),
          "few1_16": (800, 8, 512, 1024, 0), "split64": (8, 128, 512, 1024, 0), "whole64": (140, 64, 512, 1024, 0),
          "whole128": (140, 128, 512, 1024, 0), "wide": (140, 32, 512, 1024, 8), "wide_split": (8, 128, 512, 1024, 8),
          "d256": (140, 16, 256, 1024, 0), "d128_split": (8, 16, 128, 1024, 0), "d128_chunks": (140, 16, 128, 2100, 0)}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("level", [20, 60])
@pytest.mark.parametrize("at", [(40,), (900,), (0, 40, 900)])
@pytest.mark.parametrize("route", list(ROUTES))
def test_scores_far_above_the_reference(route, at, level, dtype):
    import dsa_triton_ascend_amd as dsa
    from dsa_triton_ascend_amd import _lib
    S1, N1, D, K, flags = ROUTES[route]
    print(f"[ref max] {route} at={at} level={level} {dtype}", flush=True)
    q, k, qr, kr = sfa_inputs(1, S1, K, N1, D, dtype, scale_qk=0.25, seed=11)
    scale = 1.0 / np.sqrt(D + 64)
    qr[..., 0] = 8.0
    kr[0, :, 0, 0] = 0.0
    for i, t in enumerate(at):  # the later the larger, by a binade
        kr[0, t, 0, 0] = (level + i) / (8.0 * scale * 1.4426950408889634)
    kr = torch.from_numpy(kr).to(dtype).float().numpy()
    si = np.broadcast_to(np.arange(K, dtype=np.int32), (1, S1, 1, K)).copy()
    lib = _lib.load()
    if flags:
        lib.dsa_set_test_flags(flags)
    try:
        got = dsa.sparse_flash_attention_triton(
            dev(q, dtype), dev(k, dtype), None, dev(si, torch.int32), scale_value=scale, query_rope=dev(qr, dtype),
            key_rope=dev(kr, dtype), sparse_mode=0, return_softmax_lse=True)
        torch.cuda.synchronize()
    finally:
        if flags:
            lib.dsa_set_test_flags(0)
    rows = [0, S1 - 1]
    ref = sfa_fwd_bsnd(q, k, si, qr, kr, scale, [S1], [K], 1, 0, True, "float32", positions="kernel",
                       rows=[(0, r) for r in rows])
    for g, e, name in zip(got, ref, ("out", "softmax_max", "softmax_sum")):
        ax = 1 if name == "out" else 2
        atol = 2.0 ** -9 * float(np.abs(k).max()) if name == "out" else 2e-3
        assert_close(np.take(g.float().cpu().numpy(), rows, ax), np.take(e, rows, ax), 2e-2, atol, name)
