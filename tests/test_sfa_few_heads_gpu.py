"""The D = 512 forward for few heads (sfa_fwd_few.hip) against the oracle:
four waves per row and one wave per row, at the edges of its 16-token tiles
and 512-position chunks, over every layout it takes.

Tolerances are those of test_sfa_fwd_gpu (rtol 2e-2 / atol 2e-3 against the
fp32 golden).  Inputs scaled up spread the scores over hundreds of binades,
which sends waves through their second pass, and leave the softmax one or two
tokens: the rounding errors of P no longer average out, and the bound is that
of one rounding of P to bf16, |dO| <= 2^-9 sum p |v| <= 2^-9 max |v| (the
output's own rounding is inside rtol)."""
import numpy as np
import pytest
import torch

from oracle.common import expand_block_indices
from oracle.sfa import sfa_fwd_bsnd
from tests.helpers import assert_close, dev, sfa_inputs, sparse_indices

pytestmark = pytest.mark.gpu

D = 512


def _check(S1, S2, N1, K, mode, dtype, bs=1, mul=1.0, flags=0, act_k=None, punch=False, holes=(), seed=5):
    import dsa_triton_ascend_amd as dsa
    from dsa_triton_ascend_amd import _lib
    print(f"[few heads] S1={S1} S2={S2} N1={N1} K={K} mode={mode} bs={bs} {dtype} x{mul} flags={flags}", flush=True)
    q, k, qr, kr = sfa_inputs(1, S1, S2, N1, D, dtype, scale_qk=mul, seed=seed)
    act_k = act_k or S2
    si = sparse_indices(1, S1, S2, K, bs, mode, [S1], [act_k])
    if punch:  # -1 inside the rows, and rows that are all -1
        rng = np.random.RandomState(3)
        si[rng.rand(*si.shape) < 0.4] = -1
        si[:, ::7] = -1
    for h in holes:
        si[..., h] = -1
    scale = 1.0 / np.sqrt(D + 64)
    lib = _lib.load()
    if flags:
        lib.dsa_set_test_flags(flags)
    try:
        got = dsa.sparse_flash_attention_triton(
            dev(q, dtype), dev(k, dtype), None, dev(si, torch.int32), scale_value=scale,
            actual_seq_lengths_kv=[act_k], query_rope=dev(qr, dtype), key_rope=dev(kr, dtype), sparse_block_size=bs,
            sparse_mode=mode, return_softmax_lse=True)
        torch.cuda.synchronize()
    finally:
        if flags:
            lib.dsa_set_test_flags(0)
    rows = sorted(set([0, 1, S1 // 2, S1 - 1] + list(np.random.RandomState(1).randint(0, S1, 12))))
    ref = sfa_fwd_bsnd(q, k, expand_block_indices(si, bs), qr, kr, scale, [S1], [act_k], 1, mode, True, "float32",
                       positions="kernel", rows=[(0, int(r)) for r in rows])
    for g, e, name in zip(got, ref, ("out", "softmax_max", "softmax_sum")):
        ax = 1 if name == "out" else 2
        atol = 2e-3 if mul == 1 or name != "out" else 2.0 ** -9 * float(np.abs(k).max())
        assert_close(np.take(g.float().cpu().numpy(), rows, ax), np.take(e, rows, ax), 2e-2, atol, name)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("N1", [1, 16, 32])
@pytest.mark.parametrize("S1,K", [(130, 520), (130, 2048), (200, 1000), (800, 513), (800, 1041), (1100, 2048)])
def test_rows_and_lengths(S1, K, N1, dtype):
    _check(S1, S1 + 1500, N1, K, 3, dtype)


@pytest.mark.parametrize("S1", [130, 800])
@pytest.mark.parametrize("N1", [16, 32])
def test_holes_short_rows_and_causal_start(S1, N1):
    _check(S1, S1, N1, 600, 3, torch.bfloat16, punch=True)


@pytest.mark.parametrize("S1,K,holes", [(800, 1024, (0,)), (130, 4096, (0, 1024, 2048, 3072))])
@pytest.mark.parametrize("N1", [16, 32])
def test_list_full_to_its_last_entry(S1, K, holes, N1):
    """One hole in a wave's first 512 positions leaves 15 entries for the next
    chunk, whose 512 then fill the list: the pad must stay inside it (the next
    wave's list follows)."""
    _check(S1, K + 100, N1, K, 0, torch.bfloat16, holes=holes)


@pytest.mark.parametrize("S1", [130, 800])
@pytest.mark.parametrize("N1", [8, 32])
def test_second_pass(S1, N1):
    _check(S1, S1 + 900, N1, 700, 0, torch.bfloat16, mul=6.0)


@pytest.mark.parametrize("S1", [130, 800])
@pytest.mark.parametrize("N1", [16, 32])
def test_blocks_lengths_and_64bit_gather(S1, N1):
    _check(S1, S1 + 700, N1, 300, 3, torch.bfloat16, bs=4)
    _check(S1, S1 + 700, N1, 600, 3, torch.float16, act_k=S1 + 333)
    _check(S1, S1 + 700, N1, 600, 3, torch.bfloat16, flags=1)


@pytest.mark.parametrize("B,S1", [(50, 3), (300, 3)])
@pytest.mark.parametrize("N1", [16, 32])
def test_paged_equals_dense(B, S1, N1):
    """A paged cache with shuffled pages gives the dense cache's results bit for bit."""
    import dsa_triton_ascend_amd as dsa
    print(f"[few heads] paged B={B} S1={S1} N1={N1}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(9)
    S2, page, K, dt = 704, 64, 600, torch.bfloat16
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dt)  # noqa: E731
    q, qr, k, kr = rn(B, S1, N1, D), rn(B, S1, N1, 64), rn(B, S2, 1, D), rn(B, S2, 1, 64)
    si = torch.argsort(torch.rand(B * S1, S2, generator=g, device="cuda"), 1)[:, :K].to(torch.int32).reshape(B, S1, 1, K)
    n = B * S2 // page
    bt = torch.randperm(n, generator=g, device="cuda").to(torch.int32).reshape(B, S2 // page)
    cache = torch.empty(n, page, 1, D, device="cuda", dtype=dt)
    cache[bt.flatten().long()] = k.reshape(n, page, 1, D)
    cache_r = torch.empty(n, page, 1, 64, device="cuda", dtype=dt)
    cache_r[bt.flatten().long()] = kr.reshape(n, page, 1, 64)
    kw = dict(scale_value=0.04, query_rope=qr, sparse_mode=3, return_softmax_lse=True)
    a = dsa.sparse_flash_attention_triton(q, k, None, si, key_rope=kr, **kw)
    b = dsa.sparse_flash_attention_triton(q, cache, None, si, key_rope=cache_r, block_table=bt, layout_kv="PA_BSND",
                                          actual_seq_lengths_kv=[S2] * B, **kw)
    for x, y in zip(a, b):
        assert torch.equal(x, y)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("N1", [16, 32])
@pytest.mark.parametrize("S1", [130, 800])
def test_numerators_round_as_on_the_wide_kernel(S1, N1, dtype):
    """The softmax numerators are rounded relative to the same reference as on
    the 128-head kernels (the max of the row's first 32 tokens), so the outputs
    agree but for the order of the fp32 sums.  Those leave the scores (|s| < 16
    log2 units) and sums within about 1e-6 of each other: at most some 1 % of
    the numerators and outputs land on another 16-bit value.  With another
    reference every numerator rounds anew, and a quarter of the outputs differ."""
    import dsa_triton_ascend_amd as dsa
    from dsa_triton_ascend_amd import _lib
    print(f"[few heads] wide kernel S1={S1} N1={N1} {dtype}", flush=True)
    K = 1024
    q, k, qr, kr = sfa_inputs(1, S1, 1500, N1, D, dtype)
    si = sparse_indices(1, S1, 1500, K, 1, 0)
    args = (dev(q, dtype), dev(k, dtype), None, dev(si, torch.int32))
    kw = dict(scale_value=1.0 / np.sqrt(D + 64), query_rope=dev(qr, dtype), key_rope=dev(kr, dtype), sparse_mode=0,
              return_softmax_lse=True)
    a = dsa.sparse_flash_attention_triton(*args, **kw)
    lib = _lib.load()
    lib.dsa_set_test_flags(8)
    try:
        b = dsa.sparse_flash_attention_triton(*args, **kw)
        torch.cuda.synchronize()
    finally:
        lib.dsa_set_test_flags(0)
    differ = (a[0] != b[0]).float().mean().item()
    print(f"[few heads] {differ:.2g} of the outputs differ", flush=True)
    assert differ < 0.08
    torch.testing.assert_close(a[1], b[1], rtol=1e-6, atol=1e-6)
    torch.testing.assert_close(a[2], b[2], rtol=1e-5, atol=0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("S1", [130, 800])
@pytest.mark.parametrize("N1", [16, 32])
def test_large_first_token_is_the_reference_of_every_wave(N1, S1, dtype):
    """A first token 24 binades above the rest (an attention sink), and one
    token 20 binades above the rest in each later quarter of the positions:
    relative to the first token no numerator passes 1, relative to a later
    quarter's own first tokens the fp16 one of its large token is infinite.
    One token dominates, so the output is bounded by one rounding of P."""
    import dsa_triton_ascend_amd as dsa
    print(f"[few heads] sink N1={N1} S1={S1} {dtype}", flush=True)
    K = 1024
    level = np.zeros(K, np.float32)
    level[0] = 24
    level[[300, 600, 1000]] = 20
    q, k, qr, kr = sfa_inputs(1, S1, K, N1, D, dtype, scale_qk=0.25, seed=11)
    qr[..., 0] = 8.0
    scale = 1.0 / np.sqrt(D + 64)
    kr[0, :, 0, 0] = torch.from_numpy(level / (8.0 * scale * 1.4426950408889634)).to(dtype).float().numpy()
    si = np.broadcast_to(np.arange(K, dtype=np.int32), (1, S1, 1, K)).copy()
    got = dsa.sparse_flash_attention_triton(
        dev(q, dtype), dev(k, dtype), None, dev(si, torch.int32), scale_value=scale, query_rope=dev(qr, dtype),
        key_rope=dev(kr, dtype), sparse_mode=0, return_softmax_lse=True)
    torch.cuda.synchronize()
    rows = [0, S1 // 2, S1 - 1]
    ref = sfa_fwd_bsnd(q, k, si, qr, kr, scale, [S1], [K], 1, 0, True, "float32", positions="kernel",
                       rows=[(0, r) for r in rows])
    for g, e, name in zip(got, ref, ("out", "softmax_max", "softmax_sum")):
        ax = 1 if name == "out" else 2
        atol = 2.0 ** -9 * float(np.abs(k).max()) if name == "out" else 2e-3
        assert_close(np.take(g.float().cpu().numpy(), rows, ax), np.take(e, rows, ax), 2e-2, atol, name)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("S1,N1,K", [(140, 64, 1000), (600, 64, 300), (130, 32, 640), (260, 32, 768)])
def test_whole_rows_on_the_64_head_kernel(S1, N1, K, dtype):
    """Unsplit rows of 64 heads, and of 32 heads with few tokens each."""
    _check(S1, S1 + 1500, N1, K, 3, dtype)
