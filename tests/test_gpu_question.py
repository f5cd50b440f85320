"""Several queries per row (a question pass): the matrix-core forms of the scoring pass, the selection and the attention
at the edges of their tiles, against fp64 and against the forms they stand beside."""
import pytest
import torch

from _util import make_qkv

pytestmark = pytest.mark.gpu


def question_mask(B, Lq, Lk, dtype, device, kind):
    """None, the causal mask of the last Lq positions, or that with a finite bias on every third column ('general')."""
    if kind is None:
        return None
    last = torch.arange(Lk - Lq, Lk).view(-1, 1)
    m = torch.where(torch.arange(Lk).view(1, -1) > last, float(torch.finfo(dtype).min), 0.0)
    m = m.expand(B, 1, Lq, Lk).clone()
    if kind == "general":
        m[..., ::3] -= 1.5
        m.clamp_(min=float(torch.finfo(dtype).min))
    return m.to(dtype).to(device)


def score_keys(N, q, k, amask, resid=False):
    """(scores of the 16-bit keys, remainders or None), both (rows, Lk) on the host, and the raw key tensor."""
    B, Hq, Lq, D = q.shape
    Hkv, Lk = k.shape[1], k.shape[2]
    pitch = (Lk + 63) // 64 * 64
    keys = torch.zeros((B * Hq * Lq, pitch), dtype=torch.int16, device=q.device)
    rem = torch.zeros_like(keys) if resid else None
    ms = (0, 0, 0) if amask is None else (amask.stride(0), 0, amask.stride(2))
    N.call("sah_qk_scores", N.QkScoresArgs(
        q.data_ptr(), q.stride(0), q.stride(1), q.stride(2), k.data_ptr(), k.stride(0), k.stride(1), k.stride(2),
        None if amask is None else amask.data_ptr(), *ms, N.dtype_code(q.dtype), B, Hq, Hkv, Lq, Lk, D,
        keys.data_ptr(), pitch, N.stream_ptr(q.device), None if rem is None else rem.data_ptr()))
    torch.cuda.synchronize()
    u = keys.cpu().to(torch.int32) & 0xFFFF
    assert bool((u[:, Lk:] == 0).all())  # nothing is written beyond the row's keys
    bits = torch.where((u & 0x8000) != 0, u & 0x7FFF, (~u) & 0xFFFF).to(torch.int16)
    s = bits.view(q.dtype)[:, :Lk].float()
    return s, None if rem is None else rem[:, :Lk].cpu().view(q.dtype).float(), keys


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind", [None, "causal", "general"])
@pytest.mark.parametrize("shape", [  # vectors per KV head on either side of 32 and 64, keys on either side of 64 and 256
    (1, 14, 2, 1, 255, 128), (1, 8, 2, 8, 257, 128), (2, 4, 4, 33, 64, 64), (1, 8, 2, 17, 1000, 64), (1, 2, 1, 66, 129, 128)])
def test_scores_of_many_query_vectors(cuda, dtype, kind, shape):
    """Keys are the scores rounded to the tensor type where torch rounds them: after the product, and again after the mask
    is added. Bound: half a unit of the type per rounding, plus fp32 accumulation of D products (D 2^-24 of sum |q k|)."""
    from sparse_attention_hub_amd import _native as N

    B, Hq, Hkv, Lq, Lk, D = shape
    q, k, _ = make_qkv(B, Hq, Hkv, Lq, Lk, D, dtype, seed=7, outliers=True, device=cuda)
    q = q.transpose(1, 2).contiguous().transpose(1, 2)  # the layout HuggingFace hands over
    am = question_mask(B, Lq, Lk, dtype, cuda, kind)
    s, rem, keys = score_keys(N, q, k, am, resid=kind is None)
    kk = k.double().cpu().repeat_interleave(Hq // Hkv, dim=1)
    exact = (q.double().cpu() @ kk.transpose(-1, -2)).reshape(-1, Lk)
    mass = (q.double().cpu().abs() @ kk.abs().transpose(-1, -2)).reshape(-1, Lk)
    unit = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    bound = unit * exact.abs() + D * 2.0 ** -24 * mass + 2.0 ** -24
    if kind is not None:
        m = am.double().cpu().expand(B, Hq, Lq, Lk).reshape(-1, Lk)
        exact = (exact + m).clamp(min=-torch.finfo(dtype).max if dtype == torch.bfloat16 else -float("inf"))
        if dtype == torch.float16:  # minus a large score may leave the type's range
            exact = exact.masked_fill(exact < -65520.0, -float("inf"))
        bound = bound + unit * exact.abs().nan_to_num(posinf=0.0)
    hidden = torch.zeros_like(exact, dtype=torch.bool) if kind is None else m < -1e4
    assert bool(((s.double() - exact).abs() <= bound)[~hidden].all())
    assert bool((s[hidden] < -6e4).all())
    if kind is None:
        assert bool(((s.double() + rem.double() - exact).abs() <= 2.0 ** -15 * exact.abs() + D * 2.0 ** -24 * mass + 2.0 ** -24).all())
        s2, _, keys2 = score_keys(N, q, k, None)
        assert torch.equal(keys, keys2)  # the remainders change nothing about the keys
