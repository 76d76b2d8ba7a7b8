"""The D_idx = 128 kernels of the dense stage at the edges of their 64-row
tiles, 128-key workgroups and query-row chunks: lengths around the tile sizes,
several rows per workgroup, more keys than queries and the reverse, batches
with hidden rows, 16-bit weights at an odd element offset.  Oracle, tolerances
and their reasons: test_dense_kl_gpu."""
import math

import numpy as np
import pytest
import torch

from oracle.dense_kl import dense_index_lse, dense_kl_bwd
from tests.test_dense_kl_gpu import _case, _check, _dev, _np, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("Ni", [32, 64, 128])
@pytest.mark.parametrize("S1,S2", [(1, 1), (5, 63), (64, 64), (65, 129), (130, 193), (200, 70)])
def test_tile_edges(S1, S2, Ni, dtype):
    print(f"[dense tiles] S1={S1} S2={S2} Ni={Ni} {dtype}", flush=True)
    c = _case(1, S1, S2, 32, 1, 128, Ni, 128, dtype, torch.float32)
    got = _run(c, dtype, torch.float32, given_lse=False)
    q, k, qr, kr, qi, ki, w, smax, ssum, scale = c
    exp = dense_kl_bwd(q, k, qr, kr, qi, ki, w, smax, ssum, scale)
    _check(got, exp, f"{S1}x{S2} Ni={Ni}", torch.float32)


@pytest.mark.parametrize("Ni", [32, 128])
def test_lengths_over_batches(Ni):
    B, S1, S2 = 3, 70, 150
    aq, ak = [70, 33, 1], [150, 20, 131]
    print(f"[dense tiles] lengths Ni={Ni}", flush=True)
    c = _case(B, S1, S2, 32, 1, 128, Ni, 128, torch.bfloat16, torch.bfloat16, aq, ak)
    got = _run(c, torch.bfloat16, torch.bfloat16, given_lse=True, act_q=aq, act_k=ak)
    q, k, qr, kr, qi, ki, w, smax, ssum, scale = c
    exp = dense_kl_bwd(q, k, qr, kr, qi, ki, w, smax, ssum, scale, act_q=aq, act_k=ak)
    _check(got, exp, f"lengths Ni={Ni}", torch.bfloat16)
    for b in range(B):
        assert np.all(got[0][b, aq[b]:] == 0) and np.all(got[2][b, aq[b]:] == 0) and np.all(got[1][b, ak[b]:] == 0)


@pytest.mark.parametrize("w_dtype", [torch.bfloat16, torch.float16])
def test_weights_at_an_odd_offset(w_dtype):
    """16-bit weights that start two bytes past a word boundary."""
    import dsa_triton_ascend_amd as dsa
    print(f"[dense tiles] odd offset {w_dtype}", flush=True)
    c = _case(1, 66, 140, 32, 1, 128, 64, 128, w_dtype, w_dtype)
    q, k, qr, kr, qi, ki, w, smax, ssum, scale = c
    d = [_dev(x, w_dtype) for x in (q, k, qi, ki)]
    buf = torch.empty(w.size + 1, dtype=w_dtype, device="cuda")
    odd = buf[1:].view(w.shape)
    odd.copy_(_dev(w, w_dtype))
    assert odd.is_contiguous() and odd.data_ptr() % 4 == 2
    kw = dict(scale_value=scale, query_rope=_dev(qr, w_dtype), key_rope=_dev(kr, w_dtype))
    st = (_dev(smax, torch.float32), _dev(ssum, torch.float32))
    a = dsa.dense_loss_backward_triton(d[0], d[1], d[2], d[3], odd, *st, **kw)
    b = dsa.dense_loss_backward_triton(d[0], d[1], d[2], d[3], _dev(w, w_dtype), *st, **kw)
    for x, y in zip(a, b):
        assert np.array_equal(_np(x), _np(y))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("Ni,Di", [(32, 128), (64, 128), (128, 128), (64, 256)])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), -float("inf")])
def test_key_rows_that_no_row_sees_are_not_read(bad, Ni, Di, dtype):
    """Non-finite index keys past the key lengths (padding that nobody wrote)
    change nothing: every output is bit for bit that of finite padding."""
    print(f"[dense tiles] padding {bad} Ni={Ni} Di={Di} {dtype}", flush=True)
    B, S1, S2 = 3, 70, 200
    aq, ak = [70, 33, 5], [150, 20, 131]
    c = list(_case(B, S1, S2, 32, 1, 128, Ni, Di, dtype, torch.float32, aq, ak))
    want = _run(c, dtype, torch.float32, given_lse=False, act_q=aq, act_k=ak)
    c[5] = c[5].copy()
    for b in range(B):
        c[5][b, ak[b]:] = bad
    got = _run(c, dtype, torch.float32, given_lse=False, act_q=aq, act_k=ak)
    for x, y in zip(got, want):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("Ni", [32, 64, 128])
@pytest.mark.parametrize("at", [64, 97, 129])
def test_key_rows_behind_the_causal_diagonal(at, Ni, dtype):
    """A NaN index key reaches the query rows that see it and no others (the
    rows before it share its tile)."""
    print(f"[dense tiles] diagonal at={at} Ni={Ni} {dtype}", flush=True)
    S = 150
    c = list(_case(1, S, S, 32, 1, 128, Ni, 128, dtype, torch.float32))
    want = _run(c, dtype, torch.float32, given_lse=False)
    c[5] = c[5].copy()
    c[5][0, at] = float("nan")
    got = _run(c, dtype, torch.float32, given_lse=False)
    for i in (0, 2):  # dQueryIndex, dWeights
        assert np.array_equal(got[i][0, :at], want[i][0, :at])


def test_index_lse_is_as_exact_as_its_scores():
    """The LSE's sum is off by the scores' absolute error.  Scores of 32 heads
    with weights in [0, 1) are about 72; rounded once to fp32 from sums of a
    quarter each they are off by 3.1e-8 of that (2.4e-8 from the last rounding,
    the rest from the quarters), 2.25e-6."""
    import dsa_triton_ascend_amd as dsa
    print("[dense tiles] LSE error", flush=True)
    S, Ni, dt = 3001, 32, torch.float16
    g = torch.Generator(device="cuda").manual_seed(7)
    qi = torch.randn(1, S, Ni, 128, generator=g, device="cuda", dtype=dt)
    ki = torch.randn(1, S, 1, 128, generator=g, device="cuda", dtype=dt)
    w = torch.rand(1, S, Ni, generator=g, device="cuda")
    mx, sm = dsa.dense_lightning_indexer_softmax_lse_triton(qi, ki, w)
    kt = ki[0, :, 0].double().t().contiguous()
    exp = torch.empty(S, dtype=torch.float64, device="cuda")
    for a in range(0, S, 128):
        b = min(S, a + 128)
        relu = (qi[0, a:b].double().reshape(-1, 128) @ kt).reshape(b - a, Ni, S).clamp_(min=0)
        score = (relu * w[0, a:b].double()[..., None]).sum(1)
        score.masked_fill_(torch.arange(S, device="cuda")[None] > torch.arange(a, b, device="cuda")[:, None], -math.inf)
        exp[a:b] = (score - score.max(1, keepdim=True).values).exp().sum(1)
    err = ((sm.double().reshape(-1) - exp).norm() / exp.norm()).item()
    print(f"[dense tiles] sum off by {err:.3g}", flush=True)
    assert err < 2.25e-6


@pytest.mark.parametrize("which", ["query_index", "key_index"])
def test_index_rows_at_an_odd_offset(which):
    """Index rows that start two bytes past a 16-byte boundary."""
    import dsa_triton_ascend_amd as dsa
    print(f"[dense tiles] odd offset {which}", flush=True)
    dt = torch.bfloat16
    c = _case(1, 66, 140, 32, 1, 128, 64, 128, dt, torch.float32)
    q, k, qr, kr, qi, ki, w, smax, ssum, scale = c
    t = {"query_index": _dev(qi, dt), "key_index": _dev(ki, dt)}
    buf = torch.empty(t[which].numel() + 1, dtype=dt, device="cuda")
    odd = buf[1:].view(t[which].shape)
    odd.copy_(t[which])
    t[which] = odd
    assert odd.is_contiguous() and odd.data_ptr() % 16 == 2
    got = dsa.dense_loss_backward_triton(
        _dev(q, dt), _dev(k, dt), t["query_index"], t["key_index"], _dev(w, torch.float32), _dev(smax, torch.float32),
        _dev(ssum, torch.float32), scale_value=scale, query_rope=_dev(qr, dt), key_rope=_dev(kr, dt))
    _check([_np(x) for x in got], dense_kl_bwd(q, k, qr, kr, qi, ki, w, smax, ssum, scale), which, torch.float32)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("Ni", [1, 48, 100])
def test_head_counts_of_the_c_interface(Ni, dtype):
    """Index head counts that the library takes and the Python API does not:
    partly filled head tiles of the scores, and the per-row gradient kernels."""
    from dsa_triton_ascend_amd import _lib
    print(f"[dense tiles] C interface Ni={Ni} {dtype}", flush=True)
    B, S1, S2, N1, D = 2, 40, 150, 32, 128
    aq, ak = [40, 17], [150, 77]
    c = _case(B, S1, S2, N1, 1, D, Ni, 128, dtype, torch.float32, aq, ak)
    q, k, qr, kr, qi, ki, w, smax, ssum, scale = c
    d = [_dev(x, dtype) for x in (q, k, qr, kr, qi, ki)] + [_dev(x, torch.float32) for x in (w, smax, ssum)]
    seq = [torch.tensor(x, dtype=torch.int32, device="cuda") for x in (aq, ak)]
    outs = [torch.empty_like(d[4]), torch.empty_like(d[5]), torch.empty_like(d[6]), torch.empty(1, device="cuda")]
    imax, isum = torch.empty(B, S1, device="cuda"), torch.empty(B, S1, device="cuda")
    lib, stream = _lib.load(), _lib.stream_handle(torch.device("cuda", torch.cuda.current_device()))
    n = lib.dsa_dense_kl_bwd_workspace_size(B, S1, S2, 128)
    ws = torch.empty(n, dtype=torch.uint8, device="cuda")
    code, f32 = _lib.dtype_code(dtype), _lib.dtype_code(torch.float32)
    p = [t.data_ptr() for t in d]
    _lib.check(lib.dsa_dense_li_softmax_lse(p[4], p[5], p[6], seq[0].data_ptr(), seq[1].data_ptr(), imax.data_ptr(),
                                            isum.data_ptr(), B, S1, S2, Ni, 128, code, f32, stream), "lse")
    _lib.check(lib.dsa_dense_kl_bwd(
        p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], p[8], imax.data_ptr(), isum.data_ptr(), seq[0].data_ptr(),
        seq[1].data_ptr(), *[t.data_ptr() for t in outs], B, S1, S2, N1, 1, D, 64, Ni, 128, code, f32, scale,
        ws.data_ptr(), n, stream), "bwd")
    torch.cuda.synchronize()
    em, es = dense_index_lse(qi, ki, w, act_q=aq, act_k=ak)
    rows = es.reshape(B, S1) > 0
    np.testing.assert_allclose(_np(imax)[rows], em.reshape(B, S1)[rows], rtol=1e-5, atol=1e-4)
    np.testing.assert_allclose(_np(isum), es.reshape(B, S1), rtol=1e-4, atol=1e-2)
    exp = dense_kl_bwd(q, k, qr, kr, qi, ki, w, smax, ssum, scale, act_q=aq, act_k=ak)
    _check([_np(x) for x in outs], exp, f"Ni={Ni}", torch.float32)
