"""Inputs whose memory is in another order than their shape (dense, transposed):
every output equals the contiguous call's bit for bit."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _perm(t):
    """The same values, laid out with the first two dimensions swapped in memory."""
    return t.transpose(0, 1).contiguous().transpose(0, 1)


def _rn(g, *s, dtype=torch.bfloat16):
    return torch.randn(*s, generator=g, device="cuda").to(dtype)


def _sfa(g, B=2, S1=6, S2=40, N=16, D=128, K=24):
    q, qr, k, kr = _rn(g, B, S1, N, D), _rn(g, B, S1, N, 64), _rn(g, B, S2, 1, D), _rn(g, B, S2, 1, 64)
    si = torch.argsort(torch.rand(B, S1, 1, S2, generator=g, device="cuda"), -1)[..., :K].to(torch.int32)
    return q, qr, k, kr, si


def _same(fn, tensors):
    for i in range(-1, len(tensors)):  # all of them, then each alone
        moved = [_perm(t) if i in (-1, j) else t for j, t in enumerate(tensors)]
        assert i == -1 or not moved[i].is_contiguous()
        for a, b in zip(fn(*moved), fn(*tensors)):
            assert torch.equal(a, b)


def test_sfa_forward_and_grad():
    import dsa_triton_ascend_amd as dsa
    print("[strided] sfa", flush=True)
    q, qr, k, kr, si = _sfa(torch.Generator(device="cuda").manual_seed(1))
    kw = dict(scale_value=0.07, sparse_mode=0)
    fwd = lambda q, qr, k, kr, si: dsa.sparse_flash_attention_triton(  # noqa: E731
        q, k, k, si, query_rope=qr, key_rope=kr, return_softmax_lse=True, **kw)
    out, mx, sm = fwd(q, qr, k, kr, si)
    do = torch.randn_like(out)
    _same(fwd, [q, qr, k, kr, si])
    _same(lambda q, qr, k, kr, si, do, out: dsa.sparse_flash_attention_grad_triton(
        q, k, k, si, do, out, mx, sm, query_rope=qr, key_rope=kr, **kw), [q, qr, k, kr, si, do, out])


def test_sfa_train():
    import dsa_triton_ascend_amd as dsa
    print("[strided] train", flush=True)
    q, qr, k, kr, si = _sfa(torch.Generator(device="cuda").manual_seed(2))

    def step(*leaves):
        leaves = [t.detach().requires_grad_() for t in leaves]
        out, _, _ = dsa.sparse_flash_attention_train(leaves[0], leaves[2], si, scale_value=0.07, query_rope=leaves[1],
                                                     key_rope=leaves[3])
        return torch.autograd.grad(out, leaves, torch.ones_like(out))
    _same(step, [q, qr, k, kr])


@pytest.mark.parametrize("w_dtype", [torch.float32, torch.bfloat16])
def test_indexer_losses(w_dtype):
    import dsa_triton_ascend_amd as dsa
    print(f"[strided] losses {w_dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(3)
    q, qr, k, kr, si = _sfa(g, N=32)
    B, S1, S2, N = 2, 6, 40, 32
    qi, ki = _rn(g, B, S1, 32, 128), _rn(g, B, S2, 1, 128)
    w = torch.rand(B, S1, 32, generator=g, device="cuda").to(w_dtype)
    mx = torch.full((B, 1, S1, N), 3.0, device="cuda")
    sm = torch.full((B, 1, S1, N), 20.0, device="cuda")
    scale = 1 / math.sqrt(192)
    si = torch.where(si <= S2 - S1, si, -1)
    _same(lambda qi, ki, w, q, k, qr, kr: dsa.sparse_lightning_indexer_grad_kl_loss_triton(
        q, k, qi, ki, w, si, mx, sm, query_rope=qr, key_rope=kr, scale_value=scale), [qi, ki, w, q, k, qr, kr])
    _same(lambda qi, ki, w, q, k, qr, kr: dsa.dense_loss_backward_triton(
        q, k, qi, ki, w, mx, sm, scale_value=scale, query_rope=qr, key_rope=kr), [qi, ki, w, q, k, qr, kr])
    _same(lambda qi, ki, w: dsa.dense_lightning_indexer_softmax_lse_triton(qi, ki, w), [qi, ki, w])
