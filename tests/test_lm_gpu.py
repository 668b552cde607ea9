"""Embedding and cross-entropy kernels on the GPU against the oracle."""
import numpy as np
import pytest
import torch

from helpers import announce, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,V,D", [(1000, 300, 1024), (77, 50, 100), (5, 7, 8)])
def test_embedding(oracle, N, V, D):
    from ceo_amd.nn import embedding_backward, embedding_forward

    announce(f"embedding N={N} V={V} D={D}")
    rng = np.random.default_rng(N + V)
    w = torch.randn(V, D, generator=torch.Generator().manual_seed(N)).to(torch.bfloat16)
    idx = rng.integers(0, V, N).astype(np.int32)
    idx[1] = V + 3  # out of range: zero row (checked entry), skipped in the backward
    idx[2] = -1
    idd = torch.from_numpy(idx).cuda()
    out = embedding_forward(idd, w.cuda())
    torch.cuda.synchronize()
    ref = oracle.embedding_fwd(idx, w.float().numpy())
    assert np.array_equal(out.float().cpu().numpy(), ref)
    # the unchecked reference entry on valid indices only
    good = torch.from_numpy(np.clip(idx, 0, V - 1)).cuda()
    out2 = embedding_forward(good, w.cuda(), checked=False)
    assert torch.equal(out2.cpu(), w[np.clip(idx, 0, V - 1)])
    dy = torch.randn(N, D, generator=torch.Generator().manual_seed(7)).to(torch.bfloat16)
    dw = torch.full((V, D), 0.5, device="cuda")  # accumulated into
    embedding_backward(dy.cuda(), idd, dw)
    torch.cuda.synchronize()
    rdw = oracle.embedding_bwd(dy.float().numpy(), idx, V) + 0.5
    e = rel_l2(dw, rdw)
    print(f"  dW rel-L2={e:.2e}", flush=True)
    assert e <= 1e-6


@pytest.mark.parametrize("B,V,eps", [(64, 32000, 0.0), (37, 32000, 0.1), (16, 50257, 0.0),
                                     (9, 1000, 0.0), (5, 77, 0.2), (3, 70000, 0.0)])
def test_cross_entropy(oracle, B, V, eps):
    from ceo_amd.nn import cross_entropy_backward, cross_entropy_forward

    announce(f"cross_entropy B={B} V={V} eps={eps}")
    g = torch.Generator().manual_seed(B * V)
    z = (torch.randn(B, V, generator=g) * 4).to(torch.bfloat16)
    t = torch.randint(0, V, (B,), generator=g, dtype=torch.int32)
    t[0] = V  # invalid target -> NaN loss, zero gradient row
    gl = torch.rand(B, generator=g) + 0.5
    zd, td = z.cuda(), t.cuda()
    loss = cross_entropy_forward(zd, td, eps)
    grad = cross_entropy_backward(gl.cuda(), zd, td, eps)
    torch.cuda.synchronize()
    rl = oracle.cross_entropy_fwd(z.float().numpy(), t.numpy(), eps)
    rg = oracle.cross_entropy_bwd(gl.numpy(), z.float().numpy(), t.numpy(), eps)
    ln = loss.cpu().numpy()
    assert np.isnan(ln[0]) and not grad[0].any()
    err = np.abs(ln[1:] - rl[1:]).max() / np.abs(rl[1:]).max()
    eg = rel_l2(grad[1:], rg[1:])
    print(f"  loss max rel {err:.2e}, grad rel-L2 {eg:.2e}", flush=True)
    assert err <= 1e-5 and eg <= 1e-2


@pytest.mark.parametrize("B,V,eps", [(37, 32000, 0.1), (9, 1000, 0.0), (3, 70000, 0.0)])
def test_cross_entropy_forward_backward_fused(B, V, eps):
    """The one-pass entry gives the two entries' results bit for bit: with a
    per-row grad_loss, with grad_loss NULL (= ones) and in place over the
    logits (the row-in-registers path and the looped path for V = 70000)."""
    from ceo_amd.nn import (cross_entropy_backward, cross_entropy_forward,
                            cross_entropy_forward_backward)

    announce(f"cross_entropy fused fwd+bwd B={B} V={V} eps={eps}")
    g = torch.Generator().manual_seed(B + V)
    z = (torch.randn(B, V, generator=g) * 4).to(torch.bfloat16).cuda()
    t = torch.randint(0, V, (B,), generator=g, dtype=torch.int32)
    t[1] = -1  # invalid target: NaN loss, zero gradient row
    t = t.cuda()
    gl = (torch.rand(B, generator=g) + 0.5).cuda()
    loss_ref = cross_entropy_forward(z, t, eps)
    grad_ref = cross_entropy_backward(gl, z, t, eps)
    ones_ref = cross_entropy_backward(torch.ones(B, device="cuda"), z, t, eps)
    loss, grad = cross_entropy_forward_backward(z, t, eps, grad_loss=gl)
    assert torch.equal(loss.nan_to_num(), loss_ref.nan_to_num()) and torch.isnan(loss[1])
    assert torch.equal(grad, grad_ref)
    zc = z.clone()
    loss2, grad2 = cross_entropy_forward_backward(zc, t, eps, in_place=True)
    assert grad2.data_ptr() == zc.data_ptr()
    assert torch.equal(loss2.nan_to_num(), loss_ref.nan_to_num())
    assert torch.equal(grad2, ones_ref)


def test_cross_entropy_uniform_logits():
    from ceo_amd.nn import cross_entropy_forward

    announce("cross_entropy uniform logits")
    B, V = 8, 32000
    loss = cross_entropy_forward(torch.zeros(B, V, dtype=torch.bfloat16, device="cuda"),
                                 torch.arange(B, dtype=torch.int32, device="cuda"), 0.3)
    assert abs(loss.sum().item() - np.log(V)) < 1e-5


# Masked and extreme logits in the row-in-registers path: every kind of piece
# count, threads whose whole part is masked (-inf) or holds bf16's lowest
# value, a target at a piece's first and last element, a row with one finite
# logit.  Loss: fp32 sums of V terms, 1e-5 as above; the gradient is rounded
# to bf16 (2^-8) after fp32 exponentials of differences up to 60 (60 2^-22).
@pytest.mark.parametrize("V", [8, 1000, 8192, 8200, 32000, 65536])
def test_cross_entropy_masked_and_extreme(V):
    from ceo_amd.nn import cross_entropy_forward, cross_entropy_forward_backward

    announce(f"cross_entropy masked V={V}")
    g = torch.Generator().manual_seed(V)
    z = (torch.randn(6, V, generator=g) * 6).to(torch.bfloat16)
    t = torch.tensor([0, V - 1, 7, V // 2, 3, 5], dtype=torch.int32)
    z[0, V // 2:] = float("-inf")
    z[1, :V - 8] = float("-inf")
    z[2, 1::2] = torch.finfo(torch.bfloat16).min
    z[3] = float("-inf")
    z[3, V // 2] = 2.0
    z[4, :] = -3.0
    loss, grad = cross_entropy_forward_backward(z.cuda(), t.cuda())
    assert torch.equal(loss, cross_entropy_forward(z.cuda(), t.cuda()))
    torch.cuda.synchronize()
    lp = torch.log_softmax(z.double(), -1)
    ref = -lp.gather(1, t.long()[:, None])[:, 0] / 6
    rg = lp.exp()
    rg[torch.arange(6), t.long()] -= 1
    loss, grad = loss.cpu().double(), grad.cpu().double() * 6
    # lp[t] near 0 is the difference of two numbers of about 20
    both = torch.isfinite(ref)
    assert torch.equal(torch.isinf(loss), ~both)
    err = ((loss - ref).abs() / ref.abs().clamp(min=1))[both].max().item()
    eg = ((grad - rg).abs() - (2.0 ** -8 + 60 * 2.0 ** -22) * rg.abs()).max().item()
    print(f"  loss {err:.2e} grad beyond the bound {eg:.2e}", flush=True)
    assert err <= 1e-5 and eg <= 1e-5  # p_t - 1: fp32's 2^-22 of 1


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_cross_entropy_row_with_inf_or_nan(bad):
    from ceo_amd.nn import cross_entropy_forward_backward

    z = torch.zeros(3, 1000, dtype=torch.bfloat16)
    z[1, 500] = bad
    t = torch.tensor([1, 1, 1], dtype=torch.int32)
    loss, grad = cross_entropy_forward_backward(z.cuda(), t.cuda())
    assert loss.isnan().tolist() == [False, True, False]
    assert grad.isnan().all(1).tolist() == [False, True, False] and not grad[0].isnan().any()


# The three entries agree with each other and in both paths (rows of whole 16-byte
# pieces up to 65536 logits in registers, others looped): ordinary rows to the bounds
# above, and a row with +inf or NaN gives NaN for its loss and its whole gradient.
@pytest.mark.parametrize("V", [1000, 1001, 32000, 32001, 40000, 65536, 65544])
def test_cross_entropy_entries_and_paths_agree(V):
    from ceo_amd.nn import (cross_entropy_backward, cross_entropy_forward,
                            cross_entropy_forward_backward)

    announce(f"cross_entropy entries V={V}")
    g = torch.Generator().manual_seed(V)
    z = (torch.randn(4, V, generator=g) * 3).to(torch.bfloat16)
    z[2, V // 3], z[3, V - 1] = float("inf"), float("nan")
    t = torch.tensor([V - 1, 5, 1, 2], dtype=torch.int32).cuda()
    zc, gl = z.cuda(), torch.ones(4, device="cuda")
    loss, grad = cross_entropy_forward_backward(zc, t)
    alone = cross_entropy_forward(zc, t), cross_entropy_backward(gl, zc, t)
    lp = torch.log_softmax(z[:2].double(), -1)
    rg = lp.exp()
    rg[torch.arange(2), t[:2].long().cpu()] -= 1
    ref = -lp.gather(1, t[:2].long().cpu()[:, None])[:, 0] / 4
    for lo, gr in ((loss, grad), alone):
        assert lo.isnan().tolist() == [False, False, True, True]
        assert gr[2:].isnan().all() and not gr[:2].isnan().any()
        assert ((lo[:2].double().cpu() - ref).abs() / ref.abs().clamp(min=1)).max() <= 1e-5
        d = (gr[:2].double().cpu() * 4 - rg).abs() - (2.0 ** -8 + 60 * 2.0 ** -22) * rg.abs()
        assert d.max() <= 1e-5
