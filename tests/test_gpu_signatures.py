"""Signatures of many keys (the bulk kernels) against the oracle's MLP, at the edges of their tiles of 32 vectors and of a
workgroup's share of them."""
import pytest
import torch

from oracle import reference_path as O

pytestmark = pytest.mark.gpu


def _masker(wts, bits, hidden, act, layers=3):
    from sparse_attention_hub_amd.sparse_attention import HashAttentionTopKMaskerConfig
    from sparse_attention_hub_amd.sparse_attention.research_attention.maskers.fixed.implementations.hashattention_top_k import (
        HashAttentionTopKMasker,
    )

    return HashAttentionTopKMasker(HashAttentionTopKMaskerConfig(
        heavy_size=8, hat_bits=bits, hat_mlp_layers=layers, hat_mlp_hidden_size=hidden, hat_mlp_activation=act, hat_weights=wts))


def _codes(masker, x, heads, pitch, offset):
    codes = torch.full((x.shape[0], heads, pitch, 2), -7, dtype=torch.int32, device=x.device)
    masker._hash(x, x.shape[1], heads, 0, x.shape[2], 0, "key", codes, pitch, offset)
    return codes.cpu()


def _signs(codes, bits):
    shifts = torch.arange(bits)
    c = codes.to(torch.int64) & 0xFFFFFFFF
    return ((((c[..., :1] >> shifts) & 1) * 2 - 1) * ((c[..., 1:] >> shifts) & 1)).float()


@pytest.mark.parametrize("shape", [(128, 128, 32), (64, 128, 32), (128, 64, 16)])  # head_dim, hidden width, bits
@pytest.mark.parametrize("act", ["silu", "relu", "tanh", "gelu"])
@pytest.mark.parametrize("dtype,L", [(torch.bfloat16, 128), (torch.bfloat16, 257), (torch.bfloat16, 3001), (torch.float16, 287)])
def test_bulk_signatures(cuda, shape, act, dtype, L):
    from sparse_attention_hub_amd.sparse_attention.utils.hashattention_utils import random_hat_weights

    D, hidden, bits = shape
    B, Hkv, G = 2, 2, 3
    wts = random_hat_weights(1, Hkv * G, D, bits, 3, hidden, dtype=dtype, seed=1)
    gen = torch.Generator().manual_seed(L)
    x = torch.randn(B, L, Hkv, D, generator=gen).to(dtype)  # a transposed view, as a model hands its keys over
    pitch, offset = L + 9, 5
    codes = _codes(_masker(wts, bits, hidden, act), x.to(cuda).transpose(1, 2), Hkv * G, pitch, offset)
    assert (codes[:, :, :offset] == -7).all() and (codes[:, :, offset + L:] == -7).all()
    sig = O.hash_signatures(O.repeat_kv(x.transpose(1, 2), G), wts[0]["key_matrix"], wts[0]["key_bias"], act)
    # sums in another order: a value within rounding of 0 (or of a rounding border of an activation) may land on the other side
    agree = (_signs(codes[:, :, offset:offset + L], bits) == sig.float()).float().mean(dim=(0, 1, 3))
    assert agree.mean().item() >= 0.9995
    assert agree.min().item() >= 0.9  # a vector in another's place agrees in half of its bits


def test_a_key_that_is_not_finite_reaches_no_other_key(cuda):
    from sparse_attention_hub_amd.sparse_attention.utils.hashattention_utils import random_hat_weights

    wts = random_hat_weights(1, 4, 128, 32, 3, 128, dtype=torch.bfloat16, seed=2)
    x = torch.randn(1, 2, 300, 128, generator=torch.Generator().manual_seed(3)).to(torch.bfloat16).to(cuda)
    y = x.clone()
    bad = torch.tensor([0, 31, 32, 170, 299], device=cuda)
    y[:, :, bad[0::2], 5] = float("inf")
    y[:, :, bad[1::2], 77] = float("nan")
    m = _masker(wts, 32, 128, "silu")
    a, b = _codes(m, x, 4, 300, 0), _codes(m, y, 4, 300, 0)
    keep = torch.ones(300, dtype=torch.bool)
    keep[bad.cpu()] = False
    assert torch.equal(a[:, :, keep], b[:, :, keep])
    # not a number is neither positive nor zero
    assert (b[:, :, bad[1::2].cpu(), 0] == 0).all() and (b[:, :, bad[1::2].cpu(), 1] == -1).all()


@pytest.mark.parametrize("L", [129, 3001, 9000])  # weights that leave room for one workgroup a CU
def test_bulk_signatures_of_four_layers(cuda, L):
    from sparse_attention_hub_amd.sparse_attention.utils.hashattention_utils import random_hat_weights

    wts = random_hat_weights(1, 4, 128, 32, 4, 128, dtype=torch.bfloat16, seed=1)
    x = torch.randn(1, 2, L, 128, generator=torch.Generator().manual_seed(L)).to(torch.bfloat16)
    codes = _codes(_masker(wts, 32, 128, "silu", layers=4), x.to(cuda), 4, L, 0)
    sig = O.hash_signatures(O.repeat_kv(x, 2), wts[0]["key_matrix"], wts[0]["key_bias"], "silu")
    agree = (_signs(codes, 32) == sig.float()).float().mean(dim=(0, 1, 3))  # (as above)
    assert agree.mean().item() >= 0.9995 and agree.min().item() >= 0.9
