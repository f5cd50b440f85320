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
@pytest.mark.parametrize("shape,form", [  # vectors per KV head on either side of 32 and 64, keys on either side of 64 and 256
    ((1, 14, 2, 1, 255, 128), "k_qk_scores"), ((1, 8, 2, 8, 257, 128), "k_qk_scores"), ((2, 4, 4, 33, 64, 64), "k_qk_scores"),
    ((1, 8, 2, 17, 1000, 64), "k_qk_scores"), ((1, 2, 1, 66, 129, 128), "k_qk_scores"),
    # ... and batches that make them key rows enough for the matrix cores
    ((40, 14, 2, 1, 1255, 128), "k_qk_scores_mfma"), ((25, 8, 2, 8, 511, 128), "k_qk_scores_mfma"),
    ((26, 4, 4, 33, 513, 64), "k_qk_scores_mfma"), ((40, 8, 2, 17, 641, 64), "k_qk_scores_mfma"),
    ((96, 2, 1, 66, 257, 128), "k_qk_scores_mfma")])
def test_scores_of_many_query_vectors(cuda, dtype, kind, shape, form):
    """Keys are the scores rounded to the tensor type where torch rounds them: after the product, and again after the mask
    is added. Bound: half a unit of the type per rounding, plus fp32 accumulation of D products (D 2^-24 of sum |q k|)."""
    from sparse_attention_hub_amd import _native as N

    B, Hq, Hkv, Lq, Lk, D = shape
    q, k, _ = make_qkv(B, Hq, Hkv, Lq, Lk, D, dtype, seed=7, outliers=True, device=cuda)
    q = q.transpose(1, 2).contiguous().transpose(1, 2)  # the layout HuggingFace hands over
    am = question_mask(B, Lq, Lk, dtype, cuda, kind)
    N.timing_enable(True)
    s, rem, keys = score_keys(N, q, k, am, resid=kind is None)
    assert launched(N) == {form}
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


def launched(N):
    names = set(N.timing_collect())
    N.timing_enable(False)
    return names


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind", [None, "causal", "general"])
@pytest.mark.parametrize("shape,density", [  # rows per KV head around 32, 64 and 128; keys around a 32-key tile and a 64-key
    # stage; batches that make these small calls rows enough for the matrix-core form (256 rows are one round of the gather)
    ((12, 8, 2, 8, 257, 128), 0.3), ((14, 14, 2, 5, 300, 64), 0.5), ((8, 4, 1, 40, 130, 128), 0.2), ((1, 8, 2, 33, 1000, 64), 0.3),
    ((4, 8, 2, 32, 1025, 128), 0.1), ((160, 2, 2, 2, 31, 128), 1.0), ((64, 4, 2, 3, 96, 64), None)])
def test_attention_of_many_query_vectors(cuda, dtype, kind, shape, density):
    """Against fp64. Bound per element: half a unit of the output type, the weights' exponentials and sums in fp32 (2^-19 of
    sum p |v|), and the logit's error (fp32 products and the mask's addition: D 2^-23 of the largest |q||k|) in the weights.
    density None: no mask at all (dense attention)."""
    import sparse_attention_hub_amd.sparse_attention as sa
    from sparse_attention_hub_amd import _native as N
    from sparse_attention_hub_amd.sparse_attention.utils.mask_attention_utils import get_masked_attention_output

    B, Hq, Hkv, Lq, Lk, D = shape
    q, k, v = make_qkv(B, Hq, Hkv, Lq, Lk, D, dtype, seed=3, device=cuda)
    am = question_mask(B, Lq, Lk, dtype, cuda, kind)
    sinks = torch.linspace(-1.0, 2.0, Hq) if kind == "causal" else None
    if density is None:
        member = torch.ones(B, Hq, Lq, Lk, dtype=torch.bool)
        mask = sa.Mask.create_full_mask((B, Hq, Lq, Lk), dtype=dtype, device=cuda)
    else:
        g = torch.Generator().manual_seed(1)
        member = torch.rand(B, Hq, Lq, Lk, generator=g) < density
        member[..., 0] = True           # no empty row
        member[0, 0, 0, 1:] = False     # a row of one entry
        member[0, -1, -1, :] = True     # and one of all
        mask = sa.Mask.create_mask_from_dense_mask((B, Hq, Lq, Lk), member.to(dtype).to(cuda), dtype)
    N.timing_enable(True)
    out = get_masked_attention_output(None, q, k, v, am, None if sinks is None else sinks.to(cuda), D ** -0.5, 0.0, mask)
    torch.cuda.synchronize()
    assert "k_members_attn_mfma" in launched(N)

    G = Hq // Hkv
    qq, kk, vv = q.double().cpu(), k.double().cpu().repeat_interleave(G, 1), v.double().cpu().repeat_interleave(G, 1)
    z = qq @ kk.transpose(-1, -2) * D ** -0.5
    if am is not None:
        z = z + am.double().cpu()
    z = z.masked_fill(~member, -float("inf"))
    top = z.amax(-1, keepdim=True)
    e = torch.exp(z - top)
    den = e.sum(-1, keepdim=True)
    if sinks is not None:
        den = den + torch.exp(sinks.double().view(1, Hq, 1, 1) - top)
    p = e / den
    ref = (p @ vv).transpose(1, 2)
    mass = (p @ vv.abs()).transpose(1, 2)
    half = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)  # 8 / 11 significant bits: half a unit is 2^-8 / 2^-11 of the value at most
    logit = D * 2.0 ** -23 * float((qq.abs() @ kk.abs().transpose(-1, -2)).max()) * D ** -0.5
    tiny = 2.0 ** -25 if dtype == torch.float16 else 0.0  # half a unit below fp16's normal range
    bound = half * ref.abs() * 1.01 + (2.0 ** -19 + 2 * logit) * mass + tiny
    worst = float(((out.double().cpu() - ref).abs() / bound).max())
    assert worst <= 1.0, worst


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads", [False, True])  # a mask for all heads, or one for each
@pytest.mark.parametrize("pattern", ["lone", "runs"])  # every third 32-key tile with one element in one row; six tiles of eight
@pytest.mark.parametrize("shape,pad", [((2, 8, 2, 33, 1025, 128), 0), ((2, 8, 2, 40, 2047, 64), 1), ((4, 8, 2, 32, 1024, 128), 0)])
def test_attention_under_a_mask_of_few_tiles(cuda, dtype, heads, pattern, shape, pad):
    """Whether a tile's mask is all zeros is asked in whole lines, the elements come behind that answer: every row and place of
    a tile once, rows at odd elements, -0 in place of 0. Bound as above."""
    import sparse_attention_hub_amd.sparse_attention as sa
    from sparse_attention_hub_amd import _native as N
    from sparse_attention_hub_amd.sparse_attention.utils.mask_attention_utils import get_masked_attention_output

    B, Hq, Hkv, Lq, Lk, D = shape
    q, k, v = make_qkv(B, Hq, Hkv, Lq, Lk, D, dtype, seed=4, device=cuda)
    am = torch.zeros(B, Hq if heads else 1, Lq, Lk + pad, dtype=dtype)
    am[..., 1::2] = -0.0
    for t in range((Lk + 31) // 32):
        if pattern == "lone" and t % 3 == 1:
            am[:, :, (5 * t) % Lq, min(32 * t + (11 * t) % 32, Lk - 1)] = 2.0
        if pattern == "runs" and t % 8 < 6:
            am[:, :, :, 32 * t:32 * t + 32] += torch.linspace(-2.0, 2.0, Lq).view(1, 1, -1, 1).to(dtype)
    am = am.to(cuda)[..., :Lk]
    g = torch.Generator().manual_seed(2)
    member = torch.rand(B, Hq, Lq, Lk, generator=g) < 0.4
    member[..., 0] = True
    mask = sa.Mask.create_mask_from_dense_mask((B, Hq, Lq, Lk), member.to(dtype).to(cuda), dtype)
    N.timing_enable(True)
    out = get_masked_attention_output(None, q, k, v, am, None, D ** -0.5, 0.0, mask)
    torch.cuda.synchronize()
    assert "k_members_attn_mfma" in launched(N)

    G = Hq // Hkv
    qq, kk, vv = q.double().cpu(), k.double().cpu().repeat_interleave(G, 1), v.double().cpu().repeat_interleave(G, 1)
    z = (qq @ kk.transpose(-1, -2) * D ** -0.5 + am.double().cpu()).masked_fill(~member, -float("inf"))
    p = torch.softmax(z, -1)
    ref = (p @ vv).transpose(1, 2)
    mass = (p @ vv.abs()).transpose(1, 2)
    half = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    logit = D * 2.0 ** -23 * float((qq.abs() @ kk.abs().transpose(-1, -2)).max()) * D ** -0.5
    tiny = 2.0 ** -25 if dtype == torch.float16 else 0.0
    bound = half * ref.abs() * 1.01 + (2.0 ** -19 + 2 * logit) * mass + tiny
    worst = float(((out.double().cpu() - ref).abs() / bound).max())
    assert worst <= 1.0, worst


@pytest.mark.parametrize("chain", ["oracle", "hash"])
@pytest.mark.parametrize("shape,heavy,dense", [  # one round of rows, and a share of a round too many; rows and entries enough
    ((1, 8, 2, 32, 8192, 128), 250, False), ((1, 8, 2, 48, 2048, 128), 60, False), ((2, 32, 8, 40, 4096, 128), 400, True)])
def test_rows_go_dense_where_that_pays(cuda, chain, shape, heavy, dense):
    """Planned steps of several queries: which form the attention takes, and that the result is the masker-by-masker path's
    (another order of the sums: the last bit of bf16, and 2^-12 of the largest value where a sum cancels)."""
    import sparse_attention_hub_amd.sparse_attention as sa
    from sparse_attention_hub_amd import _native as N
    from sparse_attention_hub_amd.sparse_attention.utils.hashattention_utils import random_hat_weights

    B, Hq, Hkv, Lq, Lk, D = shape
    q, k, v = make_qkv(B, Hq, Hkv, Lq, Lk, D, torch.bfloat16, seed=9, device=cuda)
    top = sa.OracleTopKConfig(heavy_size=heavy) if chain == "oracle" else sa.HashAttentionTopKMaskerConfig(
        heavy_size=heavy, hat_bits=32, hat_mlp_layers=3, hat_mlp_hidden_size=128, hat_mlp_activation="silu",
        hat_weights=random_hat_weights(1, Hq, D, 32, 3, 128, dtype=torch.bfloat16, seed=1))
    outs = []
    for planned in (True, False):
        ra = sa.ResearchAttention.create_from_config(sa.ResearchAttentionConfig(masker_configs=[
            sa.SinkMaskerConfig(sink_size=16), sa.LocalMaskerConfig(window_size=64), top]))
        ra.return_attention_weights = False
        if not planned:
            ra._plan_kind = None
        meta = {}
        for _ in range(2):  # the first call fills the layer's cache
            N.timing_enable(True)
            out = ra.custom_attention(None, q, k, v, None, D ** -0.5, 0.0, sparse_meta_data=meta, layer_idx=0)[0]
            torch.cuda.synchronize()
            names = launched(N)
        assert ("k_members_attn_mfma" in names) == dense
        outs.append(out.double().cpu())
    assert bool(((outs[0] - outs[1]).abs() <= 2.0 ** -7 * outs[1].abs() + 2.0 ** -12 * float(outs[1].abs().max())).all())


def test_a_chain_reads_the_bitmaps_it_has_built_and_no_others(cuda):
    """Rows that the caller brings need no bitmap (their builder may have been asked to skip it); rows that a builder of the
    chain writes have one. A shape that goes dense where it may."""
    import ctypes as C

    import sparse_attention_hub_amd.sparse_attention as sa
    from sparse_attention_hub_amd import _native as N

    B, Hq, Hkv, Lq, Lk, D = 1, 8, 2, 48, 2048, 128
    q, k, v = make_qkv(B, Hq, Hkv, Lq, Lk, D, torch.bfloat16, seed=3, device=cuda)
    member = torch.rand(B, Hq, Lq, Lk, generator=torch.Generator().manual_seed(1)) < 0.6
    member[0, 0, 0] = True  # rows have room for every key
    rows = sa.Mask.create_mask_from_dense_mask(member.shape, member.to(q.dtype).to(cuda), q.dtype).to_rows(0)
    work = torch.empty(N.members_work_floats(B, Hq, Hkv, Lq, Lk, D), device=cuda)

    def attend(call, **fields):
        out = torch.empty(B, Lq, Hq, D, dtype=q.dtype, device=cuda)
        a = N.AttentionArgs()
        a.rows, a.q, a.k, a.v, a.out = rows.as_struct(), q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr()
        (a.qs_b, a.qs_h, a.qs_l), (a.ks_b, a.ks_h, a.ks_l), (a.vs_b, a.vs_h, a.vs_l) = q.stride()[:3], k.stride()[:3], v.stride()[:3]
        a.dtype, a.B, a.Hq, a.Hkv, a.Lq, a.Lk, a.D = N.dtype_code(q.dtype), B, Hq, Hkv, Lq, Lk, D
        a.scaling, a.unit_inv_w, a.max_cnt, a.work, a.work_floats = D ** -0.5, 1.0, rows.cap, work.data_ptr(), work.numel()
        a.stream = N.stream_ptr(cuda)
        chain = N.ChainArgs()
        chain.attention = C.addressof(a)
        for name, block in fields.items():
            setattr(chain, name, C.addressof(block))
        N.timing_enable(True)
        N.call(call, chain if call == "sah_run_chain" else a)
        torch.cuda.synchronize()
        return out, "k_members_attn_mfma" in launched(N)

    want, _ = attend("sah_sparse_attention")
    assert attend("sah_members_attention")[1]
    stale = rows.bitmap.clone()
    rows.bitmap.zero_()
    got, went_dense = attend("sah_run_chain")
    assert torch.equal(got, want) and not went_dense
    rows.bitmap.copy_(stale)
    sl = N.SinkLocalArgs(rows.as_struct(), Lq, 1024, 600, 1, 1, N.stream_ptr(cuda))
    assert attend("sah_run_chain", sink_local=sl)[1]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind", [None, "causal"])
@pytest.mark.parametrize("shape", [(1, 8, 2, 48, 2048, 128), (2, 8, 2, 66, 2100, 64), (4, 4, 4, 40, 1030, 128)])
def test_keys_that_are_not_finite_stay_with_the_rows_that_hold_them(cuda, dtype, kind, shape):
    """A few keys whose K or V row is not finite: rows without them have the result they have without such keys (two
    summation orders: the last bit of the type, and 2^-12 of its largest value where a sum cancels), rows with them are not finite."""
    import sparse_attention_hub_amd.sparse_attention as sa
    from sparse_attention_hub_amd import _native as N
    from sparse_attention_hub_amd.sparse_attention.utils.mask_attention_utils import get_masked_attention_output

    B, Hq, Hkv, Lq, Lk, D = shape
    q, k, v = make_qkv(B, Hq, Hkv, Lq, Lk, D, dtype, seed=13, device=cuda)
    am = question_mask(B, Lq, Lk, dtype, cuda, kind)
    member = torch.rand(B, Hq, Lq, Lk, generator=torch.Generator().manual_seed(4)) < 0.5
    member[..., 0] = True
    bad = {5: ("k", float("nan")), 70: ("k", float("inf")), 333: ("v", float("nan")), 900: ("v", float("-inf")), 1000: ("k", float("-inf"))}
    member[:, :, : Lq // 2][..., list(bad)] = False
    holds = member[..., list(bad)].any(-1).transpose(1, 2)
    mask = sa.Mask.create_mask_from_dense_mask(member.shape, member.to(dtype).to(cuda), dtype)
    clean = get_masked_attention_output(None, q, k, v, am, None, D ** -0.5, 0.0, mask).double().cpu()
    for at, (which, value) in bad.items():
        (k if which == "k" else v)[:, 0, at, 3] = value
    N.timing_enable(True)
    out = get_masked_attention_output(None, q, k, v, am, None, D ** -0.5, 0.0, mask).double().cpu()
    assert "k_members_attn_mfma" in launched(N)
    first = torch.arange(Hq) < Hq // Hkv  # the KV head with such keys
    held = holds & first
    unit = 2.0 ** (-7 if dtype == torch.bfloat16 else -10)
    near = (out - clean).abs() <= unit * clean.abs() + 2.0 ** -12 * float(clean.abs().max())
    assert bool(near[~held].all())
    bad_v = member[..., [333, 900]].any(-1).transpose(1, 2) & first
    assert bool(bad_v.any()) and not bool(torch.isfinite(out[..., 3][bad_v]).any())
    nan_k = member[..., 5].transpose(1, 2) & first
    assert bool(nan_k.any()) and not bool(torch.isfinite(out[nan_k]).any())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_weights_keep_their_fp32_precision(cuda, dtype):
    """Rows of two entries whose values nearly cancel: what is left shows the weights' error, 2^-20 of the values here
    (exp2 of a logit up to 4 in size and a few fp32 operations), beside the output's own rounding. One in eight rows holds
    the other keys: one of value 0 whose weight is 2^20 to 2^30 times the others', of value 1, whose sum is all that is left
    (logits up to 21: 2^-19)."""
    import sparse_attention_hub_amd.sparse_attention as sa
    from sparse_attention_hub_amd import _native as N
    from sparse_attention_hub_amd.sparse_attention.utils.mask_attention_utils import get_masked_attention_output

    B, H, Lq, Lk, D = 1, 8, 64, 4096, 128
    g = torch.Generator().manual_seed(8)
    q, k, v = torch.zeros(B, H, Lq, D), torch.zeros(B, H, Lk, D), torch.ones(B, H, Lk, D)
    q[..., 0] = torch.randint(-256, 257, (B, H, Lq), generator=g) / 64.0   # key 0: this logit; key 1: 0
    k[:, :, 0, 0] = 1.0
    v[:, :, :2] = 1 + torch.rand(B, H, 2, D, generator=g)
    v[:, :, 1] *= -1
    q[:, :, ::8] = 0.0
    q[:, :, ::8, 1] = torch.arange(H).view(1, H, 1) + 14.0 - 0.25
    k[:, :, 2, 1] = 1.0
    v[:, :, 2] = 0.0
    q, k, v = q.to(dtype), k.to(dtype), v.to(dtype)
    member = torch.zeros(B, H, Lq, Lk, dtype=torch.bool)
    member[..., :2] = True
    member[:, :, ::8, :2] = False
    member[:, :, ::8, 2:] = True
    mask = sa.Mask.create_mask_from_dense_mask(member.shape, member.to(dtype).to(cuda), dtype)
    N.timing_enable(True)
    out = get_masked_attention_output(None, q.to(cuda), k.to(cuda), v.to(cuda), None, None, 1.0, 0.0, mask).double().cpu()
    assert "k_members_attn_mfma" in launched(N)
    z = (q.double() @ k.double().transpose(-1, -2)).masked_fill(~member, -float("inf"))
    p = torch.softmax(z, -1)
    ref, mass = (p @ v.double()).transpose(1, 2), (p @ v.double().abs()).transpose(1, 2)
    half = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    exps = torch.where(torch.arange(Lq) % 8 == 0, 2.0 ** -19, 2.0 ** -20).view(1, Lq, 1, 1)
    worst = (out - ref).abs() / (1.01 * half * ref.abs() + exps * mass + (2.0 ** -25 if dtype == torch.float16 else 0.0))
    assert float(worst.max()) <= 1.0


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind", [None, "causal"])
@pytest.mark.parametrize("density", [None, 0.2])
def test_statistics_of_many_query_vectors(cuda, dtype, kind, density):
    """The row's largest logit and the denominator relative to it, at a shape whose plain call takes the matrix-core form,
    against fp64, and what is built on them. Bounds: a logit's fp32 error, D 2^-23 of sum |q k|, and for the numerator the
    output's rounding."""
    import sparse_attention_hub_amd.sparse_attention as sa
    from sparse_attention_hub_amd.sparse_attention.utils import mask_attention_utils as U

    B, Hq, Hkv, Lq, Lk, D = 1, 8, 2, 48, 2048, 128
    q, k, v = make_qkv(B, Hq, Hkv, Lq, Lk, D, dtype, seed=11, device=cuda)
    am = question_mask(B, Lq, Lk, dtype, cuda, kind)
    member = torch.ones(B, Hq, Lq, Lk, dtype=torch.bool)
    if density is not None:
        member = torch.rand(B, Hq, Lq, Lk, generator=torch.Generator().manual_seed(2)) < density
        member[..., 0] = True
    mask = (sa.Mask.create_full_mask(member.shape, dtype=dtype, device=cuda) if density is None
            else sa.Mask.create_mask_from_dense_mask(member.shape, member.to(dtype).to(cuda), dtype))
    z = q.double().cpu() @ k.double().cpu().repeat_interleave(Hq // Hkv, 1).transpose(-1, -2) * D ** -0.5
    if am is not None:
        z = z + am.double().cpu()
    vv = v.double().cpu().repeat_interleave(Hq // Hkv, 1)
    sel = z.masked_fill(~member, -float("inf"))
    top, top_all = sel.amax(-1, keepdim=True), z.amax(-1, keepdim=True)
    _, stats = U._run_attention(q, k, v, am, None, D ** -0.5, None if density is None else mask.to_rows(0), False, return_stats=True)
    assert float((stats[:, 0].double().cpu().view_as(top) - top).abs().max()) < 1e-4
    want = torch.exp(sel - top).sum(-1, keepdim=True)
    assert float(((stats[:, 1].double().cpu().view_as(top) - want) / want).abs().max()) < 1e-4
    e = torch.exp(sel - top_all)
    den = U.get_attention_denominator(None, q, k, am, D ** -0.5, 0.0, mask)
    num = U.get_attention_numerator(None, q, k, v, am, D ** -0.5, 0.0, mask)
    assert float(((den.double().cpu() - e.sum(-1, keepdim=True)) / e.sum(-1, keepdim=True)).abs().max()) < 2e-4
    half = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    assert bool(((num.double().cpu() - e @ vv).abs() <= 1.01 * half * (e @ vv).abs() + 3e-4 * (e @ vv.abs())).all())
    sinks = torch.linspace(-2.0, 6.0, Hq)
    _, den2, _ = U.apply_sink_bias(num, den, None, q, k, am, sinks.to(cuda), D ** -0.5)
    new = torch.maximum(top_all, sinks.double().view(1, Hq, 1, 1))
    want2 = e.sum(-1, keepdim=True) * torch.exp(top_all - new) + torch.exp(sinks.double().view(1, Hq, 1, 1) - new)
    assert float(((den2.double().cpu() - want2) / want2).abs().max()) < 2e-4


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind", [None, "causal", "general"])
@pytest.mark.parametrize("shape,pitch,form", [  # keys on either side of a lane's 8 and a workgroup's 2048; an odd code pitch
    # and few scores: the form of one thread per score
    ((1, 2, 3, 5), 16, "k_hamming_scores"), ((2, 3, 4, 2049), 2050, "k_hamming_scores"), ((1, 4, 33, 2055), 2064, "k_hamming_scores16"),
    ((1, 2, 1, 4096), 4096, "k_hamming_scores"), ((1, 2, 5, 40), 41, "k_hamming_scores"), ((64, 16, 33, 7), 16, "k_hamming_scores16"),
    ((9, 3, 4, 2049), 2050, "k_hamming_scores16"), ((25, 2, 1, 4096), 4096, "k_hamming_scores16"), ((9, 3, 4, 2049), 2051, "k_hamming_scores")])
def test_signature_scores_of_many_queries(cuda, dtype, kind, shape, pitch, form):
    """Whole numbers plus the mask, rounded once to the tensor type: exactly torch's values."""
    from sparse_attention_hub_amd import _native as N

    B, Hq, Lq, Lk = shape
    g = torch.Generator().manual_seed(Lk)

    def planes(*n):  # per component -1, 0 or 1, zeros rare
        v = torch.randint(0, 2, (*n, 32), generator=g) * 2 - 1
        return v * (torch.rand(*n, 32, generator=g) > 0.05)

    def pack(v):
        w = 2 ** torch.arange(32, dtype=torch.int64)
        p = torch.stack([((v > 0) * w).sum(-1), ((v != 0) * w).sum(-1)], -1)
        return torch.where(p >= 2 ** 31, p - 2 ** 32, p).to(torch.int32)

    kv, qv = planes(B, Hq, Lk), planes(B, Hq, Lq)
    codes = torch.zeros((B, Hq, pitch, 2), dtype=torch.int32)
    codes[:, :, :Lk] = pack(kv)
    codes, qcodes = codes.to(cuda), pack(qv).reshape(-1, 2).contiguous().to(cuda)
    am = question_mask(B, Lq, Lk, dtype, cuda, kind)
    ms = (0, 0, 0) if am is None else (am.stride(0), 0, am.stride(2))
    kp = (Lk + 63) // 64 * 64
    keys = torch.zeros((B * Hq * Lq, kp), dtype=torch.int16, device=cuda)
    N.timing_enable(True)
    N.call("sah_hamming_scores", N.HammingScoresArgs(codes.data_ptr(), pitch, qcodes.data_ptr(), B, Hq, Lq, Lk,
                                                     None if am is None else am.data_ptr(), *ms, N.dtype_code(dtype),
                                                     keys.data_ptr(), kp, N.stream_ptr(cuda)))
    torch.cuda.synchronize()
    assert launched(N) == {form}
    u = keys.cpu().to(torch.int32) & 0xFFFF
    assert bool((u[:, Lk:] == 0).all())  # nothing is written beyond the row's keys
    bits = torch.where((u & 0x8000) != 0, u & 0x7FFF, (~u) & 0xFFFF).to(torch.int16)
    ref = (qv.float() @ kv.float().transpose(-1, -2)).to(dtype)
    if am is not None:
        ref = ref + am.cpu()
    assert torch.equal(bits.view(dtype)[:, :Lk], ref.reshape(-1, Lk))


@pytest.mark.parametrize("table", [False, True])  # reseeds drawn where a centre is empty, and ahead of the run
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [  # (batch, KV heads, keys, head_dim, sub-spaces, centres): a few draws, and more than a block of
    (1, 1, 40, 16, 2, 8), (2, 3, 300, 64, 8, 256), (1, 2, 1500, 32, 4, 128)])  # 624 words of the generator; vector and matrix forms
def test_clustering_draws_its_start_and_its_reseeds_as_torch_does(cuda, monkeypatch, dtype, shape, table):
    """Keys of three distinct, well separated vectors: most centres are empty in every iteration and are reseeded, a mean of
    equal vectors is that vector, and equal distances go to the lowest centre. Codes and centres are then exact."""
    from oracle import reference_path as O
    from sparse_attention_hub_amd import _native as N
    from sparse_attention_hub_amd.sparse_attention.research_attention.maskers.fixed.implementations.utils import pq_utils
    from sparse_attention_hub_amd.sparse_attention.research_attention.maskers.fixed.implementations.utils.pq_utils import (
        gather_sub_vectors, kmeans_keys_batched, seeded_initial_centres,
    )

    if table:
        monkeypatch.setattr(pq_utils, "_RESEED_TABLE_FROM", 0)
    B, Hkv, n, D, n_sub, n_cent = shape
    off, iters, seed = 3, 3, 7919 * 2
    g = torch.Generator().manual_seed(n)
    vecs = torch.tensor([-4.0, 0.5, 8.0]).view(3, 1).expand(3, D) * torch.tensor([1.0, -1.0]).repeat(D // 2)
    k = vecs[torch.randint(0, 3, (B, Hkv, n + off), generator=g)].to(dtype)
    groups = B * Hkv * n_sub
    codes = torch.zeros((B, Hkv, n, n_sub), dtype=torch.uint8, device=cuda)
    N.timing_enable(True)
    centres, _ = kmeans_keys_batched(k.to(cuda), off, n_sub, n_cent, iters, codes, n, tol=-1.0, seed=seed)
    torch.cuda.synchronize()
    assert ("k_pq_reseed" in launched(N)) == table
    start = gather_sub_vectors(k, off, n_sub, seeded_initial_centres(groups, n, n_cent, seed, torch.device("cpu")))
    reseed = torch.randint(0, n, (iters, groups, n_cent), generator=torch.Generator().manual_seed(seed + 1), dtype=torch.int32)
    codes_o, cent_o = O.kmeans_lloyd(O.pq_split(k, off, n_sub), start, iters, reseed_idx=reseed, tol=-1.0)
    assert torch.equal(centres.cpu().reshape(-1), cent_o.float().reshape(-1))
    assert torch.equal(codes.cpu().permute(0, 1, 3, 2).reshape(groups, n).long(), codes_o.reshape(groups, n).long())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("chain", ["fixed", "hash", "oracle", "pq"])
@pytest.mark.parametrize("kind", ["padded", "hidden", "general"])
@pytest.mark.parametrize("shape", [(3, 8, 2, 1201, 128), (1, 14, 2, 700, 64), (24, 8, 8, 333, 64)])  # 24, 14 and 192 rows:
def test_masked_decode_plan_against_masker_by_masker(cuda, dtype, chain, kind, shape):  # several workgroups a row, and one
    """Decode steps under an additive mask, the cache growing by single keys and by a block: the planned steps against the
    masker-by-masker path. Same scores and selection; the softmax's sums are taken in another order, which moves a 16-bit
    result by its last bit here and there (2^-8 / 2^-11 of single elements) and an fp32 one by a few 2^-24 of its sums."""
    import sparse_attention_hub_amd.sparse_attention as sa
    from sparse_attention_hub_amd.sparse_attention.utils.hashattention_utils import random_hat_weights

    B, Hq, Hkv, Lk, D = shape
    cfgs = [sa.SinkMaskerConfig(sink_size=9), sa.LocalMaskerConfig(window_size=70)]
    if chain == "hash":
        cfgs.append(sa.HashAttentionTopKMaskerConfig(
            heavy_size=50, hat_bits=32, hat_mlp_layers=3, hat_mlp_hidden_size=128, hat_mlp_activation="silu",
            hat_weights=random_hat_weights(1, Hq, D, 32, 3, 128, dtype=dtype, seed=1)))
    elif chain == "oracle":
        cfgs.append(sa.OracleTopKConfig(heavy_size=50))
    elif chain == "pq":
        cfgs.append(sa.PQCacheConfig(heavy_size=50, pq_group_factor=8, pq_bits=4, kmeans_iter=3, init_offset=9, metric="euclidean"))
    steps = [Lk - 69, Lk - 68, Lk - 67, Lk - 1, Lk]
    _, k, v = make_qkv(B, Hq, Hkv, 1, Lk, D, dtype, seed=5, device=cuda)
    outs = []
    for planned in (True, False):
        ra = sa.ResearchAttention.create_from_config(sa.ResearchAttentionConfig(masker_configs=cfgs))
        ra.return_attention_weights = False
        assert ra._plan_kind == chain
        if not planned:
            ra._plan_kind = None
        meta, got = {}, []
        for i, n in enumerate([steps[0]] + steps):  # the first call fills the layer's cache
            q = make_qkv(B, Hq, Hkv, 1, 1, D, dtype, seed=100 + i, device=cuda)[0]
            m = torch.zeros((B, 1, 1, n + 3))  # wider than the keys
            hidden = -float("inf") if kind == "hidden" else float(torch.finfo(dtype).min)
            for b in range(B):
                m[b, ..., : (b + 1) * n // (2 * B + 2)] = hidden
            if kind == "general":
                m[..., ::3] -= 1.5
                m.clamp_(min=float(torch.finfo(dtype).min))
            out, _ = ra.custom_attention(None, q, k[:, :, :n], v[:, :, :n], m.to(dtype).to(cuda), D ** -0.5, 0.0,
                                         sparse_meta_data=meta, layer_idx=0)
            got.append(out.double().cpu())
        assert bool(ra._plans) == planned
        outs.append(torch.stack(got))
    a, b = outs
    assert bool(torch.isfinite(b).all())
    unit = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10, torch.float32: 2.0 ** -18}[dtype]
    assert bool(((a - b).abs() <= unit * b.abs() + (1e-6 if dtype == torch.float32 else 2.0 ** -18)).all())


@pytest.mark.parametrize("dtype,D,weights", [(torch.float32, 128, False), (torch.bfloat16, 32, False), (torch.bfloat16, 128, True)])
def test_calls_that_cannot_go_dense_ask_for_no_scratch_or_bitmaps_for_it(cuda, monkeypatch, dtype, D, weights):
    import sparse_attention_hub_amd.sparse_attention as sa
    from sparse_attention_hub_amd import _native as N

    asked = []
    monkeypatch.setattr(N, "members_work_floats", lambda *a: asked.append(a) or 0)
    q, k, v = make_qkv(1, 4, 2, 6, 700, D, dtype, seed=3, device=cuda)
    for planned in (True, False):
        ra = sa.ResearchAttention.create_from_config(sa.ResearchAttentionConfig(masker_configs=[
            sa.SinkMaskerConfig(sink_size=9), sa.LocalMaskerConfig(window_size=70), sa.OracleTopKConfig(heavy_size=50)]))
        ra.return_attention_weights = weights
        if not planned:
            ra._plan_kind = None
        ra.custom_attention(None, q, k, v, None, D ** -0.5, 0.0, sparse_meta_data={}, layer_idx=0)
        for plan in ra._plans.values():
            assert plan.select.skip_bitmap == 1
        assert bool(ra._plans) == (planned and not weights)
    torch.cuda.synchronize()
    assert not asked


def test_scratch_belongs_to_one_stream_and_one_thread(cuda):
    """Partial results of calls that nothing orders do not share memory; what a thread keeps is bounded."""
    import threading

    from sparse_attention_hub_amd import _native as N
    from sparse_attention_hub_amd.sparse_attention.utils.mask_attention_utils import _workspace

    def own():
        return _workspace(cuda, 1000, N.stream_ptr(cuda))

    mine = own()
    assert own() is mine and _workspace(cuda, mine.numel() + 1, N.stream_ptr(cuda)).numel() > mine.numel()
    mine = own()
    other, held = torch.cuda.Stream(), {mine.data_ptr()}
    with torch.cuda.stream(other):
        there = own()
        assert own() is there and there.data_ptr() not in held
    assert own() is mine
    got = []
    t = threading.Thread(target=lambda: got.append(own()))
    t.start()
    t.join()
    assert got[0].data_ptr() not in {mine.data_ptr(), there.data_ptr()}
    large = _workspace(cuda, (1 << 24) + 1, N.stream_ptr(cuda))
    assert large.numel() > 1 << 24 and own() is mine
    streams = [torch.cuda.Stream() for _ in range(12)]  # as many handles at once
    for st in streams:
        with torch.cuda.stream(st):
            own()
    with torch.cuda.stream(other):
        assert own() is not there  # given back


def test_a_captured_call_keeps_its_scratch(cuda):
    """Replays write to memory of their graph, also when the buffer of the capturing stream has gone to other tensors."""
    import sparse_attention_hub_amd.sparse_attention as sa
    from sparse_attention_hub_amd import _native as N
    from sparse_attention_hub_amd.sparse_attention.utils import mask_attention_utils as U

    B, Hq, Hkv, Lk, D = 1, 8, 2, 3000, 128
    q, k, v = make_qkv(B, Hq, Hkv, 1, Lk, D, torch.bfloat16, seed=5, device=cuda)
    floats = N.work_floats(B * Hq, Lk, D)
    assert floats > 0
    mask = sa.Mask.create_full_mask((B, Hq, 1, Lk), dtype=q.dtype, device=cuda)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        def step():
            return U.get_masked_attention_output(None, q, k, v, None, None, D ** -0.5, 0.0, mask)

        want = step()
        kept = dict(U._WORK.buffers)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            out = step()
        assert {key: t.data_ptr() for key, t in U._WORK.buffers.items()} == {key: t.data_ptr() for key, t in kept.items()}
        n = max(t.numel() for t in kept.values())
        U._WORK.buffers.clear()
        kept.clear()
        others = [torch.full((n,), 7.0, device=cuda) for _ in range(12)]
        for _ in range(3):
            out.zero_()
            graph.replay()
            side.synchronize()
            assert torch.equal(out, want) and all(bool((t == 7.0).all()) for t in others)


def test_a_masked_step_on_another_stream_has_buffers_of_its_own(cuda):
    """Planned steps under a mask on two streams, nothing between them: neither waits for the other, so they share no row
    buffers, keys or counters; results are those of steps one after the other."""
    import sparse_attention_hub_amd.sparse_attention as sa

    B, Hq, Hkv, Lk, D = 2, 8, 2, 900, 64
    _, k, v = make_qkv(B, Hq, Hkv, 1, Lk, D, torch.bfloat16, seed=5, device=cuda)
    qs = [make_qkv(B, Hq, Hkv, 1, 1, D, torch.bfloat16, seed=s, device=cuda)[0] for s in (1, 2)]
    m = torch.zeros((B, 1, 1, Lk), dtype=torch.bfloat16, device=cuda)
    m[0, ..., :100] = torch.finfo(torch.bfloat16).min
    ra = sa.ResearchAttention.create_from_config(sa.ResearchAttentionConfig(masker_configs=[
        sa.SinkMaskerConfig(sink_size=9), sa.LocalMaskerConfig(window_size=70), sa.OracleTopKConfig(heavy_size=50)]))
    ra.return_attention_weights = False

    def step(q):
        return ra.custom_attention(None, q, k, v, m, D ** -0.5, 0.0, sparse_meta_data={}, layer_idx=0)[0]

    want = [step(q) for q in qs]
    torch.cuda.synchronize()
    first = next(iter(ra._plans.values()))
    side = torch.cuda.Stream()
    a = step(qs[0])
    with torch.cuda.stream(side):
        b = step(qs[1])
    second = next(iter(ra._plans.values()))
    assert len(ra._plans) == 1 and second is not first
    assert second.keybuf is not None and second.residbuf is None  # no remainders of masked scores
    assert {t.data_ptr() for t in (first.cols, first.keybuf, first.tickets)}.isdisjoint(
        {t.data_ptr() for t in (second.cols, second.keybuf, second.tickets)})
    torch.cuda.synchronize()
    assert torch.equal(a, want[0]) and torch.equal(b, want[1])


@pytest.mark.parametrize("chain", ["fixed", "hash", "oracle", "pq"])
def test_captured_masked_steps_share_nothing(cuda, chain):
    """Two graphs of a step under a mask, captured one after the other on one stream: each runs by itself, in any order,
    with other work in between, and leaves no plan behind whose counters only a replay would clear."""
    import sparse_attention_hub_amd.sparse_attention as sa
    from sparse_attention_hub_amd.sparse_attention.utils.hashattention_utils import random_hat_weights

    B, Hq, Hkv, Lk, D = 2, 8, 2, 900, 64
    _, k, v = make_qkv(B, Hq, Hkv, 1, Lk, D, torch.bfloat16, seed=5, device=cuda)
    q = make_qkv(B, Hq, Hkv, 1, 1, D, torch.bfloat16, seed=1, device=cuda)[0]
    m = torch.zeros((B, 1, 1, Lk), dtype=torch.bfloat16, device=cuda)
    m[0, ..., :100] = torch.finfo(torch.bfloat16).min
    top = {"oracle": sa.OracleTopKConfig(heavy_size=50),
           "pq": sa.PQCacheConfig(heavy_size=50, pq_group_factor=8, pq_bits=4, kmeans_iter=3, init_offset=9, metric="euclidean"),
           "hash": sa.HashAttentionTopKMaskerConfig(
               heavy_size=50, hat_bits=32, hat_mlp_layers=3, hat_mlp_hidden_size=128, hat_mlp_activation="silu",
               hat_weights=random_hat_weights(1, Hq, D, 32, 3, 128, dtype=torch.bfloat16, seed=1))}
    ra = sa.ResearchAttention.create_from_config(sa.ResearchAttentionConfig(
        masker_configs=[sa.SinkMaskerConfig(sink_size=9), sa.LocalMaskerConfig(window_size=70)] + ([top[chain]] if chain in top else [])))
    ra.return_attention_weights = False
    meta = {}

    def step():
        return ra.custom_attention(None, q, k, v, m, D ** -0.5, 0.0, sparse_meta_data=meta, layer_idx=0)[0]

    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        step()  # fills the layer's cache
        want = step()
        plans = dict(ra._plans)
        pairs = []
        for _ in range(2):
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=side):
                out = step()
            pairs.append((graph, out))
        assert ra._plans == plans and plans
        for graph, out in pairs[::-1] * 3:
            out.zero_()
            graph.replay()
            side.synchronize()
            assert torch.equal(out, want)
            assert torch.equal(step(), want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (1, 1, 1, 7), (3, 1, 1, 8193), (2, 1, 48, 4099), (1, 4, 700, 1025)])  # one workgroup,
def test_what_a_mask_holds_is_read_back(cuda, dtype, shape):  # and several; rows that start at odd elements
    from sparse_attention_hub_amd import _native as N
    from sparse_attention_hub_amd.sparse_attention.utils.mask_attention_utils import AdditiveMaskFacts

    lowest = float(torch.finfo(dtype).min)
    B, H, L, n = shape
    zero = torch.zeros(B, H, L, n + 3, dtype=dtype, device=cuda)[..., 1: n + 1]
    other = torch.cuda.Stream()
    other.wait_stream(torch.cuda.current_stream())
    for at in ((0, 0, 0, 0), (B - 1, H - 1, L - 1, n - 1), (B // 2, H // 2, L // 2, n // 2)):
        for value, want in ((0.0, 0), (-0.0, 0), (lowest, N.AMASK_NONZERO), (-float("inf"), N.AMASK_NONZERO),
                            (-1.0, N.AMASK_NONZERO | N.AMASK_GENERAL), (float("nan"), N.AMASK_NONZERO | N.AMASK_GENERAL)):
            m = zero.clone(memory_format=torch.preserve_format)
            m[at] = value
            other.wait_stream(torch.cuda.current_stream())
            assert AdditiveMaskFacts().flags(m) == want, (at, value)
            with torch.cuda.stream(other):
                assert AdditiveMaskFacts().flags(m) == want, (at, value)
        assert AdditiveMaskFacts().flags(zero) == 0


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("shape", [(1, 1, 1, 7), (2, 1, 48, 4099), (1, 4, 3, 2049)])
def test_what_a_mask_holds_into_device_memory(cuda, dtype, shape):
    """`sah_amask_classify`: the answer of `sah_amask_read` in a word of device memory, which it adds to."""
    from sparse_attention_hub_amd import _native as N
    from sparse_attention_hub_amd.sparse_attention.utils.mask_attention_utils import AdditiveMaskFacts

    B, H, L, n = shape
    m = torch.zeros(B, H, L, n + 3, dtype=dtype, device=cuda)[..., 1: n + 1]
    for value in (0.0, -0.0, float(torch.finfo(dtype).min), -float("inf"), -1.0, float("nan")):
        m[B - 1, H - 1, L - 1, n - 1] = value
        flags = torch.zeros(1, dtype=torch.int32, device=cuda)
        N.call("sah_amask_classify", N.AmaskClassifyArgs(m.data_ptr(), *m.stride()[:3], N.dtype_code(dtype), B, H, L, n, flags.data_ptr(), N.stream_ptr(cuda)))
        assert int(flags) == AdditiveMaskFacts().flags(m), value


def test_the_next_mask_may_be_read_by_another_stream(cuda):
    """The device words an answer went through are zero when the call returns, not only when its kernel has ended: the
    thread's next question uses them from whatever stream it comes."""
    from sparse_attention_hub_amd import _native as N
    from sparse_attention_hub_amd.sparse_attention.utils import mask_attention_utils as U

    masks = [torch.zeros(1, 1, 64, 8192, device=cuda) for _ in range(2)]  # many workgroups
    masks[1][0, 0, 63, 8191] = -1.0
    streams = [torch.cuda.Stream() for _ in range(3)]
    for s in streams:
        s.wait_stream(torch.cuda.current_stream())
    for i in range(60):
        with torch.cuda.stream(streams[i % 3]):
            assert U.AdditiveMaskFacts().flags(masks[i % 2]) == (i % 2) * (N.AMASK_NONZERO | N.AMASK_GENERAL)
        if i % 5 == 0:
            with torch.cuda.stream(streams[(i + 1) % 3]):
                assert U._ANSWERS.words[cuda.index or 0][0].tolist() == [0, 0]


def test_a_mask_is_not_read_back_under_capture(cuda):
    from sparse_attention_hub_amd.sparse_attention.utils.mask_attention_utils import AdditiveMaskFacts

    m = torch.zeros(1, 1, 1, 64, device=cuda)
    assert AdditiveMaskFacts().flags(m) == 0
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream), torch.cuda.graph(graph, stream=stream):
        m.add_(0.0)
        with pytest.raises(RuntimeError, match="captured"):
            AdditiveMaskFacts().flags(m)
    assert AdditiveMaskFacts().flags(m) == 0


def test_a_first_question_under_capture_leaves_nothing_behind(cuda):
    """A thread whose first question comes under capture is refused before it has words to be answered through: the ones it
    makes afterwards belong to no graph, are clear, and a replay does not touch them."""
    from concurrent.futures import ThreadPoolExecutor

    from sparse_attention_hub_amd import _native as N
    from sparse_attention_hub_amd.sparse_attention.utils import mask_attention_utils as U

    zeros = torch.zeros(1, 1, 64, 8192, device=cuda)  # many workgroups
    other = zeros.clone()
    other[0, 0, 63, 8191] = -1.0
    kept = torch.zeros(1, dtype=torch.int64, pin_memory=True)  # another pinned block of that size is there to be handed out
    del kept
    torch.cuda.synchronize()

    def first():
        assert not U._ANSWERS.words
        graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        with torch.cuda.stream(stream), torch.cuda.graph(graph, stream=stream):
            zeros.add_(0.0)
            with pytest.raises(RuntimeError, match="captured"):
                U.AdditiveMaskFacts().flags(zeros)
        assert not U._ANSWERS.words
        for _ in range(3):
            assert U.AdditiveMaskFacts().flags(zeros) == 0
            assert U.AdditiveMaskFacts().flags(other) == N.AMASK_NONZERO | N.AMASK_GENERAL
            graph.replay()
            torch.cuda.synchronize()

    with ThreadPoolExecutor(1) as pool:
        pool.submit(first).result()


def test_words_are_clear_before_another_stream_asks(cuda):
    """The device words a thread's first question makes are cleared on its stream; if that question is refused, nothing else
    orders the next one, of another stream, behind the clearing."""
    from concurrent.futures import ThreadPoolExecutor

    from sparse_attention_hub_amd.sparse_attention.utils import mask_attention_utils as U

    zeros = torch.zeros(1, 1, 64, 8192, device=cuda)  # many workgroups
    torch.cuda.synchronize()

    def first():
        a, b = torch.cuda.Stream(), torch.cuda.Stream()
        with torch.cuda.stream(a):
            block = torch.full((2,), 7, dtype=torch.int32, device=cuda)
            a.synchronize()
            del block  # the next small allocation of this stream
            torch.cuda._sleep(20_000_000)
            with pytest.raises(ValueError, match="65535"):
                U.AdditiveMaskFacts().flags(zeros.expand(1, 1100, 64, 8192))
        with torch.cuda.stream(b):
            assert U.AdditiveMaskFacts().flags(zeros) == 0

    with ThreadPoolExecutor(1) as pool:
        pool.submit(first).result()


def _hide(m, kind, n, window, lowest):
    """What the rows of a padded batch hide: left padding; all but a few columns, fewer than the selection takes; all of them;
    columns here and there, at the lowest value and at -inf."""
    for b in range(m.shape[0]):
        if kind == "padded":
            m[b, ..., : (b + 1) * n // (m.shape[0] + 2)] = lowest
        elif kind == "few":
            m[b, ..., : n - window - 20 - b] = lowest
        elif kind == "none visible":
            m[b] = lowest if b % 2 == 0 else 0.0
        else:
            m[b, ..., b::3] = lowest
            m[b, ..., 1::7] = -float("inf")
    return m


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("kind", ["padded", "few", "none visible", "mixed"])
@pytest.mark.parametrize("shape", [(3, 8, 2, 1201, 128), (1, 14, 2, 333, 64), (17, 16, 8, 515, 64), (2, 4, 4, 34001, 64)])
def test_hash_steps_under_a_mask_that_hides_columns(cuda, dtype, kind, shape):
    """The one-kernel step against the masker-by-masker path; signatures with components that are zero among the keys'."""
    import sparse_attention_hub_amd.sparse_attention as sa
    from sparse_attention_hub_amd import _native as N
    from sparse_attention_hub_amd.sparse_attention.utils.hashattention_utils import random_hat_weights

    B, Hq, Hkv, Lk, D = shape
    window = 70
    wts = random_hat_weights(1, Hq, D, 32, 3, 128, dtype=dtype, seed=1)
    cfgs = [sa.SinkMaskerConfig(sink_size=9), sa.LocalMaskerConfig(window_size=window), sa.HashAttentionTopKMaskerConfig(
        heavy_size=50, hat_bits=32, hat_mlp_layers=3, hat_mlp_hidden_size=128,
        hat_mlp_activation="silu" if D == 128 else "relu", hat_weights=wts)]
    _, k, v = make_qkv(B, Hq, Hkv, 1, Lk, D, dtype, seed=5, device=cuda)
    k[:, :, ::5] = 0.0  # (zero keys: relu leaves signature components that are zero)
    lowest = float(torch.finfo(dtype).min)
    outs = []
    for planned in (True, False):
        ra = sa.ResearchAttention.create_from_config(sa.ResearchAttentionConfig(masker_configs=cfgs))
        ra.return_attention_weights = False
        if not planned:
            ra._plan_kind = None
        meta, got = {}, []
        for i, n in enumerate((Lk - 64, Lk - 64, Lk - 63, Lk)):  # the first call fills the layer's cache
            q = make_qkv(B, Hq, Hkv, 1, 1, D, dtype, seed=100 + i, device=cuda)[0]
            m = _hide(torch.zeros((B, 1, 1, n + 3)), kind, n, window, lowest)
            N.timing_enable(True)
            out, _ = ra.custom_attention(None, q, k[:, :, :n], v[:, :, :n], m.to(dtype).to(cuda), D ** -0.5, 0.0,
                                         sparse_meta_data=meta, layer_idx=0)
            torch.cuda.synchronize()
            assert ("k_hash_decode_attn" in launched(N)) == (planned and i > 0 and dtype != torch.float16)
            got.append(out.double().cpu())
        outs.append(torch.stack(got))
    a, b = outs
    # as above; fp16 and rows of which every entry is hidden leave nothing to select by but sums beyond the type's range
    ok = torch.isfinite(b)
    assert torch.equal(ok, torch.isfinite(a)) and (bool(ok.all()) or kind == "none visible")
    unit = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10, torch.float32: 2.0 ** -18}[dtype]
    assert bool(((a - b).abs() <= unit * b.abs() + (1e-6 if dtype == torch.float32 else 2.0 ** -18))[ok].all())


def test_a_masked_step_does_not_read_what_another_stream_writes(cuda):
    """The compact codes are written by the first planned step; a step on another stream, nothing between the two, takes the way
    that does not read them."""
    import sparse_attention_hub_amd.sparse_attention as sa
    from sparse_attention_hub_amd import _native as N
    from sparse_attention_hub_amd.sparse_attention.utils.hashattention_utils import random_hat_weights

    B, Hq, Hkv, Lk, D = 2, 8, 2, 900, 128
    _, k, v = make_qkv(B, Hq, Hkv, 1, Lk, D, torch.bfloat16, seed=5, device=cuda)
    q = make_qkv(B, Hq, Hkv, 1, 1, D, torch.bfloat16, seed=1, device=cuda)[0]
    m = _hide(torch.zeros((B, 1, 1, Lk)), "padded", Lk, 70, float(torch.finfo(torch.bfloat16).min)).to(torch.bfloat16).to(cuda)
    ra = sa.ResearchAttention.create_from_config(sa.ResearchAttentionConfig(masker_configs=[
        sa.SinkMaskerConfig(sink_size=9), sa.LocalMaskerConfig(window_size=70), sa.HashAttentionTopKMaskerConfig(
            heavy_size=50, hat_bits=32, hat_mlp_layers=3, hat_mlp_hidden_size=128, hat_mlp_activation="silu",
            hat_weights=random_hat_weights(1, Hq, D, 32, 3, 128, dtype=torch.bfloat16, seed=1))]))
    ra.return_attention_weights = False
    meta = {}

    def step():
        return ra.custom_attention(None, q, k, v, m, D ** -0.5, 0.0, sparse_meta_data=meta, layer_idx=0)[0]

    step()
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    N.timing_enable(True)
    a = step()
    with torch.cuda.stream(side):
        b = step()
    torch.cuda.synchronize()
    seen = N.timing_collect()
    N.timing_enable(False)
    assert seen["k_hash_decode_attn"][0] == 1 and seen["k_hamming_scores"][0] == 1
    assert bool(((a.double() - b.double()).abs() <= 2.0 ** -7 * b.double().abs() + 2.0 ** -18).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("chain", ["fixed", "hash", "oracle", "pq"])
def test_steps_launched_on_a_guess_about_their_mask(cuda, dtype, chain):
    """A step's first layer is launched as if its mask were like the last step's: every order of zero, hiding and general masks,
    new keys in between, against an instance that has no last step; then masks of several queries, and of one row for several."""
    import sparse_attention_hub_amd.sparse_attention as sa
    from sparse_attention_hub_amd.sparse_attention.utils.hashattention_utils import random_hat_weights

    B, Hq, Hkv, Lk, D = 2, 8, 2, 900, 64
    cfgs = [sa.SinkMaskerConfig(sink_size=9), sa.LocalMaskerConfig(window_size=70)]
    if chain == "hash":
        cfgs.append(sa.HashAttentionTopKMaskerConfig(
            heavy_size=50, hat_bits=32, hat_mlp_layers=3, hat_mlp_hidden_size=128, hat_mlp_activation="silu",
            hat_weights=random_hat_weights(1, Hq, D, 32, 3, 128, dtype=dtype, seed=1)))
    elif chain == "oracle":
        cfgs.append(sa.OracleTopKConfig(heavy_size=50))
    elif chain == "pq":
        cfgs.append(sa.PQCacheConfig(heavy_size=50, pq_group_factor=8, pq_bits=4, kmeans_iter=3, init_offset=9, metric="euclidean"))

    def make():
        ra = sa.ResearchAttention.create_from_config(sa.ResearchAttentionConfig(masker_configs=cfgs))
        ra.return_attention_weights = False
        return ra

    lowest = float(torch.finfo(dtype).min)
    _, k, v = make_qkv(B, Hq, Hkv, 1, Lk, D, dtype, seed=5, device=cuda)
    guessing, meta, meta_ref = make(), {}, {}
    unit = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}[dtype]
    order = "z" + "zhzghhggzgz"  # the first call fills the cache
    for i, kind in enumerate(order):
        n = Lk - 100 + 9 * i
        q = make_qkv(B, Hq, Hkv, 1, 1, D, dtype, seed=100 + i, device=cuda)[0]
        m = torch.zeros((B, 1, 1, n))
        if kind != "z":
            m[0, ..., :200] = lowest
        if kind == "g":
            m[..., 1::3] -= 1.5
            m.clamp_(min=lowest)
        m = m.to(dtype).to(cuda)
        args = (None, q, k[:, :, :n], v[:, :, :n], m, D ** -0.5, 0.0)
        got = guessing.custom_attention(*args, sparse_meta_data=meta, layer_idx=0)[0].double()
        want = make().custom_attention(*args, sparse_meta_data=meta_ref, layer_idx=0)[0].double()
        assert guessing._mask_facts.known(m) == {"z": 0, "h": 1, "g": 3}[kind]
        assert bool(((got - want).abs() <= unit * want.abs() + 2.0 ** -18).all()), (i, kind)
    for shape, kind in (((B, 1, 5, Lk), "h"), ((1, 1, 5, Lk), "z"), ((B, Hq, 5, Lk), "g"), ((1, 1, 1, Lk), "z")):
        q = make_qkv(B, Hq, Hkv, 5, 1, D, dtype, seed=7, device=cuda)[0]
        m = torch.zeros(shape)
        if kind != "z":
            m[..., :100] = lowest if kind == "h" else -1.0
        m = m.to(dtype).to(cuda)
        args = (None, q, k, v, m, D ** -0.5, 0.0)
        got = guessing.custom_attention(*args, sparse_meta_data=dict(meta), layer_idx=0)[0].double()
        want = make().custom_attention(*args, sparse_meta_data=dict(meta), layer_idx=0)[0].double()
        assert guessing._mask_facts.known(m) == {"z": 0, "h": 1, "g": 3}[kind]
        assert bool(((got - want).abs() <= unit * want.abs() + 2.0 ** -18).all()), (shape, kind)
    # a mask that covers nothing of the call is refused if it holds something, whatever was guessed
    bad = torch.full((1, 1, 3, Lk), -1.0, dtype=dtype, device=cuda)
    with pytest.raises(ValueError, match="does not cover"):
        guessing.custom_attention(None, q, k, v, bad, D ** -0.5, 0.0, sparse_meta_data=meta, layer_idx=0)


@pytest.mark.parametrize("chain", ["fixed", "hash", "oracle", "pq"])
def test_padded_and_unpadded_sessions_on_two_streams(cuda, chain):
    """Two sessions of one instance and geometry, unpadded on one stream and padded on the other, nothing between the two: every
    step gives what it gives alone."""
    import sparse_attention_hub_amd.sparse_attention as sa
    from sparse_attention_hub_amd.sparse_attention.utils.hashattention_utils import random_hat_weights

    B, Hq, Hkv, Lk, D = 2, 8, 2, 1500, 128
    cfgs = [sa.SinkMaskerConfig(sink_size=9), sa.LocalMaskerConfig(window_size=70)]
    if chain == "hash":
        cfgs.append(sa.HashAttentionTopKMaskerConfig(
            heavy_size=50, hat_bits=32, hat_mlp_layers=3, hat_mlp_hidden_size=128, hat_mlp_activation="silu",
            hat_weights=random_hat_weights(1, Hq, D, 32, 3, 128, dtype=torch.bfloat16, seed=1)))
    elif chain == "oracle":
        cfgs.append(sa.OracleTopKConfig(heavy_size=50))
    elif chain == "pq":
        cfgs.append(sa.PQCacheConfig(heavy_size=50, pq_group_factor=8, pq_bits=4, kmeans_iter=3, init_offset=9, metric="euclidean"))
    _, k, v = make_qkv(B, Hq, Hkv, 1, Lk, D, torch.bfloat16, seed=5, device=cuda)
    qs = [make_qkv(B, Hq, Hkv, 1, 1, D, torch.bfloat16, seed=s, device=cuda)[0] for s in range(12)]
    zero = torch.zeros((B, 1, 1, Lk))
    padded = _hide(zero.clone(), "padded", Lk, 70, float(torch.finfo(torch.bfloat16).min))
    masks = [(padded if i % 2 else zero).to(torch.bfloat16).to(cuda) for i in range(12)]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    results = []
    for together in (False, True):
        ra = sa.ResearchAttention.create_from_config(sa.ResearchAttentionConfig(masker_configs=cfgs))
        ra.return_attention_weights = False
        metas, outs = ({}, {}), []
        torch.cuda.synchronize()
        for i in range(12):  # (the first two fill the layers' caches)
            with torch.cuda.stream(streams[i % 2]):
                outs.append(ra.custom_attention(None, qs[i], k, v, masks[i], D ** -0.5, 0.0, sparse_meta_data=metas[i % 2], layer_idx=0)[0])
            if not together or i < 2:
                torch.cuda.synchronize()
        torch.cuda.synchronize()
        results.append(torch.stack(outs))
    assert torch.equal(results[0], results[1])


def test_a_replay_takes_the_mask_as_it_is_then(cuda):
    """A HashAttention step captured under a mask that only hides columns, replayed after a bias has been written into it."""
    import sparse_attention_hub_amd.sparse_attention as sa
    from sparse_attention_hub_amd.sparse_attention.utils.hashattention_utils import random_hat_weights

    B, Hq, Hkv, Lk, D = 2, 8, 2, 900, 64
    lowest = float(torch.finfo(torch.bfloat16).min)
    _, k, v = make_qkv(B, Hq, Hkv, 1, Lk, D, torch.bfloat16, seed=5, device=cuda)
    q = make_qkv(B, Hq, Hkv, 1, 1, D, torch.bfloat16, seed=1, device=cuda)[0]
    kinds = {"h": _hide(torch.zeros((B, 1, 1, Lk)), "padded", Lk, 70, lowest)}
    kinds["g"] = (kinds["h"] - 3.0 * (torch.arange(Lk) % 5 == 0)).clamp_(min=lowest)
    kinds = {name: m.to(torch.bfloat16).to(cuda) for name, m in kinds.items()}
    m = kinds["h"].clone()
    ra = sa.ResearchAttention.create_from_config(sa.ResearchAttentionConfig(masker_configs=[
        sa.SinkMaskerConfig(sink_size=9), sa.LocalMaskerConfig(window_size=70), sa.HashAttentionTopKMaskerConfig(
            heavy_size=50, hat_bits=32, hat_mlp_layers=3, hat_mlp_hidden_size=128, hat_mlp_activation="silu",
            hat_weights=random_hat_weights(1, Hq, D, 32, 3, 128, dtype=torch.bfloat16, seed=1))]))
    ra.return_attention_weights = False
    meta = {}

    def step(mask):
        return ra.custom_attention(None, q, k, v, mask, D ** -0.5, 0.0, sparse_meta_data=meta, layer_idx=0)[0]

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        want = {name: [step(mask.clone()) for _ in range(2)][1].double() for name, mask in kinds.items()}
        step(m)
        step(m)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            out = step(m)
        for kind in "hghgg":
            m.copy_(kinds[kind])
            out.zero_()
            graph.replay()
            assert bool(((out.double() - want[kind]).abs() <= 2.0 ** -7 * want[kind].abs() + 2.0 ** -18).all()), kind
        side.synchronize()
    assert not bool(((want["h"] - want["g"]).abs() <= 2.0 ** -4 * want["h"].abs()).all())  # the bias does change what is chosen


def _signature_planes(codes):
    """The +-1 / 0 components of packed codes (..., 2)."""
    c = codes.to(torch.int64) & 0xFFFFFFFF
    shifts = torch.arange(32, device=codes.device)
    return ((((c[..., :1] >> shifts) & 1) * 2 - 1) * ((c[..., 1:] >> shifts) & 1)).float()


@pytest.mark.parametrize("form", ["two planes", "compact"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kind", ["padded", "few", "mixed", "never"])
@pytest.mark.parametrize("shape", [  # rows in several workgroups and in one; keys on either side of 256, 8192 and 16384
    (2, 8, 2, 253, 128), (3, 8, 2, 1281, 64), (20, 16, 8, 700, 128), (1, 8, 2, 8191, 128), (1, 8, 2, 16320, 128), (1, 4, 4, 16451, 64)])
def test_one_kernel_masked_step_against_the_oracle(cuda, monkeypatch, form, dtype, kind, shape):
    """Both forms of the codes, given the kernel's signatures; `never`: -inf wherever the padded batch is hidden, and in all of
    a row."""
    import sparse_attention_hub_amd.sparse_attention as sa
    from oracle import reference_path as O
    from sparse_attention_hub_amd import _native as N
    from sparse_attention_hub_amd.sparse_attention.research_attention import decode_plan
    from sparse_attention_hub_amd.sparse_attention.utils.hashattention_utils import random_hat_weights

    if form == "compact":
        monkeypatch.setattr(decode_plan, "_TWO_PLANE_KEYS", 0)
        monkeypatch.setattr(decode_plan, "_TWO_PLANE_STEPS", 0)
    else:
        monkeypatch.setattr(decode_plan, "_TWO_PLANE_KEYS", 1 << 30)
    B, Hq, Hkv, n, D = shape
    sink, window, heavy = 9, 70, 50
    lowest = float(torch.finfo(dtype).min)
    ra = sa.ResearchAttention.create_from_config(sa.ResearchAttentionConfig(masker_configs=[
        sa.SinkMaskerConfig(sink_size=sink), sa.LocalMaskerConfig(window_size=window), sa.HashAttentionTopKMaskerConfig(
            heavy_size=heavy, hat_bits=32, hat_mlp_layers=3, hat_mlp_hidden_size=128, hat_mlp_activation="relu" if D == 64 else "silu",
            hat_weights=random_hat_weights(1, Hq, D, 32, 3, 128, dtype=dtype, seed=1))]))
    ra.return_attention_weights = False
    q, k, v = make_qkv(B, Hq, Hkv, 1, n, D, dtype, seed=5)
    k[:, :, ::5] = 0.0  # (zero keys: relu leaves signature components that are zero)
    m = _hide(torch.zeros((B, 1, 1, n)), "padded" if kind == "never" else kind, n, window, -float("inf") if kind == "never" else lowest)
    if kind == "never" and B > 1:
        m[B - 1] = -float("inf")
    m = m.to(dtype)
    args = [t.to(cuda) for t in (q, k, v, m)]
    meta = {}
    for i in range(2):
        N.timing_enable(True)
        out = ra.custom_attention(None, *args, D ** -0.5, 0.0, sparse_meta_data=meta, layer_idx=0)[0]
        torch.cuda.synchronize()
        names = launched(N)
        assert i == 0 or "k_hash_decode_attn" in names
    assert (meta["key"][0].pos is not None) == (form == "compact")
    qcodes = torch.empty((B, Hq, 1, 2), dtype=torch.int32, device=cuda)
    ra.maskers[2]._hash(args[0], Hq, Hq, 0, 1, 0, "query", qcodes, 1, 0)
    state = {"key_sig": _signature_planes(meta["key"][0].codes[:, :, :n]).cpu(), "query_sig": _signature_planes(qcodes).cpu()}
    want = O.research_attention([("sink", sink), ("local", window), ("hash_topk", heavy, None, None)],
                                q.float(), k.float(), v.float(), m.float().masked_fill(m == lowest, float(torch.finfo(torch.float32).min)),
                                D ** -0.5, None, state)[0].double()
    got = out.cpu().double()
    ok = torch.isfinite(want)
    assert bool(ok.all()) or kind == "never"
    assert torch.equal(ok, torch.isfinite(got))
    # rounding of the output, and the order of the fp32 sums (values of about 1, at most 129 of them)
    unit = {torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -23}[dtype]
    assert bool(((got - want).abs() <= unit * want.abs() + 129 * 2.0 ** -23)[ok].all()), float(((got - want).abs())[ok].max())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_masked_steps_go_over_to_the_compact_codes(cuda, monkeypatch, dtype):
    """A session whose rows grow past the length, and whose steps past the number, from which the compact form is built, with new
    keys hashed in between: against the masker-by-masker path."""
    import sparse_attention_hub_amd.sparse_attention as sa
    from sparse_attention_hub_amd.sparse_attention.research_attention import decode_plan
    from sparse_attention_hub_amd.sparse_attention.utils.hashattention_utils import random_hat_weights

    monkeypatch.setattr(decode_plan, "_TWO_PLANE_KEYS", 600)
    monkeypatch.setattr(decode_plan, "_TWO_PLANE_STEPS", 6)
    B, Hq, Hkv, D, window = 2, 8, 2, 128, 70
    cfgs = [sa.SinkMaskerConfig(sink_size=9), sa.LocalMaskerConfig(window_size=window), sa.HashAttentionTopKMaskerConfig(
        heavy_size=50, hat_bits=32, hat_mlp_layers=3, hat_mlp_hidden_size=128, hat_mlp_activation="silu",
        hat_weights=random_hat_weights(1, Hq, D, 32, 3, 128, dtype=dtype, seed=1))]
    _, k, v = make_qkv(B, Hq, Hkv, 1, 800, D, dtype, seed=5, device=cuda)
    outs = []
    for planned in (True, False):
        ra = sa.ResearchAttention.create_from_config(sa.ResearchAttentionConfig(masker_configs=cfgs))
        ra.return_attention_weights = False
        if not planned:
            ra._plan_kind = None
        meta, got, built = {}, [], []
        for i in range(14):
            n = 560 + 16 * i  # (every fourth step hashes 64 new keys)
            q = make_qkv(B, Hq, Hkv, 1, 1, D, dtype, seed=100 + i, device=cuda)[0]
            m = _hide(torch.zeros((B, 1, 1, n)), "padded", n, window, float(torch.finfo(dtype).min)).to(dtype).to(cuda)
            got.append(ra.custom_attention(None, q, k[:, :, :n], v[:, :, :n], m, D ** -0.5, 0.0, sparse_meta_data=meta, layer_idx=0)[0].double())
            built.append(meta["key"][0].pos is not None)
        if planned:  # (the first call fills the cache)
            assert built == [False] * 7 + [True] * 7
            assert meta["key"][0].n_compact == meta["key"][0].n
        outs.append(torch.stack(got))
    a, b = outs
    unit = {torch.bfloat16: 2.0 ** -7, torch.float32: 2.0 ** -18}[dtype]  # as of the steps under a mask that hides columns
    assert bool(((a - b).abs() <= unit * b.abs() + (1e-6 if dtype == torch.float32 else 2.0 ** -18)).all())
