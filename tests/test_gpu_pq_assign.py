"""Lloyd assignment on the matrix cores (`sah_pq_kmeans_assign`): the split form (bf16 keys in sub-vectors of 8 and more) and
the fp32 form at the edges of their tiles, against fp64; sums and counts against the codes, bit for bit."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sums", [True, False])
@pytest.mark.parametrize("shape", [  # (B, Hkv, keys, sub-vectors, dims, centres, row stride beyond the sub-vectors)
    (1, 2, 1024, 16, 8, 256, 0), (1, 1, 1057, 3, 8, 33, 0), (2, 1, 2081, 2, 16, 31, 8), (1, 1, 1, 2, 32, 5, 0),
    (1, 1, 95, 2, 64, 64, 0), (1, 1, 700, 1, 128, 65, 0), (1, 1, 700, 1, 128, 256, 0),  # the last: three terms outgrow LDS
    (1, 2, 1030, 4, 8, 40, 4), (1, 2, 1030, 4, 4, 100, 0)])  # rows of 72 bytes, sub-vectors of 4: the fp32 form
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_assignment(cuda, dtype, shape, sums):
    """The chosen centre's ||c||^2 - 2 x.c in fp64 is within the evaluation's error of the smallest: two values, each with at
    most 3 d + 4 roundings (the fp32 norm's d, the product's, a few for the alignment inside an instruction) of
    2^-23 (||c||^2 + 2 sum |x c|)."""
    from sparse_attention_hub_amd import _native as N

    B, H, n, n_sub, d, n_cent, pad = shape
    g = torch.Generator().manual_seed(n + d)
    k = torch.randn(B, H, n, n_sub * d + pad, generator=g).to(dtype)
    k[..., 1] *= 8.0
    c = torch.randn(B * H * n_sub, n_cent, d, generator=g) * torch.linspace(0.01, 3.0, n_cent).view(1, -1, 1)
    kd, cd = k.to(cuda), c.to(cuda)
    codes = torch.full((B * H, n + 3, n_sub), 255, dtype=torch.uint8, device=cuda)
    S = torch.zeros(B * H * n_sub, n_cent, d, dtype=torch.int64, device=cuda)
    C = torch.zeros(B * H * n_sub, n_cent, dtype=torch.int32, device=cuda)
    top = kd.float().abs().max().view(1)
    flag = torch.zeros(1, dtype=torch.int32, device=cuda)  # given as in the Lloyd loop: few keys go the same way as many
    a = N.PqAssignArgs()
    a.k = kd.data_ptr(); a.ks_b, a.ks_h, a.ks_l = kd.stride()[:3]; a.dtype = N.dtype_code(dtype)
    a.B, a.Hkv, a.n_sub, a.d_sub, a.n_cent, a.key_offset, a.n_keys = B, H, n_sub, d, n_cent, 0, n
    a.centres = cd.data_ptr(); a.codes = codes.data_ptr(); a.code_pitch = n + 3; a.code_offset = 3
    a.skip_flag = flag.data_ptr(); a.stream = N.stream_ptr(cuda)
    if sums:
        a.sums = S.data_ptr(); a.counts = C.data_ptr(); a.absmax_bits = top.data_ptr()
    N.timing_enable(True)
    N.call("sah_pq_kmeans_assign", a)
    torch.cuda.synchronize()
    names = set(N.timing_collect())
    N.timing_enable(False)
    if d > 17 or n >= 1024:
        assert "k_pq_assign_mfma" in names
    assert bool((codes[:, :3] == 255).all())
    got = codes[:, 3:].cpu().permute(0, 2, 1).reshape(-1, n).long()
    x = k[..., : n_sub * d].reshape(B * H, n, n_sub, d).permute(0, 2, 1, 3).reshape(-1, n, d).double()
    y = c.double()
    norm = (y * y).sum(-1).unsqueeze(1)
    dist = norm - 2 * x @ y.transpose(-1, -2)
    mass = (norm + 2 * x.abs() @ y.abs().transpose(-1, -2)).amax(-1)
    chosen = dist.gather(2, got.unsqueeze(-1)).squeeze(-1)
    assert bool((chosen - dist.amin(-1) <= 2 * (3 * d + 4) * 2.0 ** -23 * mass).all())
    if sums:
        scale = 2.0 ** (40 - math.frexp(float(top))[1])
        fixed = torch.round(x * scale).to(torch.int64)  # exact: a power of two and 24 bits
        assert torch.equal(S.cpu(), torch.zeros_like(S.cpu()).scatter_add_(1, got.unsqueeze(-1).expand(-1, -1, d), fixed))
        assert torch.equal(C.cpu(), torch.zeros_like(C.cpu()).scatter_add_(1, got, torch.ones_like(got, dtype=torch.int32)))


def _assign(N, dev, k, n_sub, d, c, top=None):
    """Codes (heads, keys, sub-vectors) of keys (1, H, n, .) against centres (H n_sub, n_cent, d); with the largest |element|
    `top` also the centres' sums and counts."""
    H, n = k.shape[1], k.shape[2]
    codes = torch.full((H, n, n_sub), 255, dtype=torch.uint8, device=dev)
    flag = torch.zeros(1, dtype=torch.int32, device=dev)
    a = N.PqAssignArgs()
    a.k = k.data_ptr(); a.ks_b, a.ks_h, a.ks_l = k.stride()[:3]; a.dtype = N.dtype_code(k.dtype)
    a.B, a.Hkv, a.n_sub, a.d_sub, a.n_cent, a.key_offset, a.n_keys = 1, H, n_sub, d, c.shape[1], 0, n
    a.centres = c.data_ptr(); a.codes = codes.data_ptr(); a.code_pitch = n; a.code_offset = 0
    a.skip_flag = flag.data_ptr(); a.stream = N.stream_ptr(dev)
    if top is not None:
        S = torch.zeros(c.shape, dtype=torch.int64, device=dev)
        C = torch.zeros(c.shape[:2], dtype=torch.int32, device=dev)
        a.sums = S.data_ptr(); a.counts = C.data_ptr(); a.absmax_bits = top.data_ptr()
    N.call("sah_pq_kmeans_assign", a)
    torch.cuda.synchronize()
    return codes.cpu() if top is None else (codes.cpu(), S.cpu(), C.cpu())


@pytest.mark.parametrize("d,n_sub,n_cent", [(8, 16, 256), (8, 2, 33), (16, 4, 128), (32, 2, 64), (64, 2, 64), (128, 1, 65)])
def test_the_split_form_gives_the_codes_of_the_fp32_form(cuda, d, n_sub, n_cent):
    """bf16 keys in rows of whole 16 bytes (split form) and the same keys in rows that are not (fp32 form): equal codes, also
    where centres come in pairs a few units of the last place apart, in equal pairs, and for keys that are not finite."""
    from sparse_attention_hub_amd import _native as N

    n, H = 1500, 2
    g = torch.Generator().manual_seed(d)
    k = torch.randn(1, H, n, n_sub * d, generator=g)
    k[..., 1] *= 8.0
    k[:, :, :200] += 20.0
    k[0, 0, 300, 3], k[0, 1, 301, 0], k[0, 0, 302, 5] = float("inf"), float("-inf"), float("nan")
    k = k.bfloat16().to(cuda)
    c = torch.randn(H * n_sub, n_cent, d, generator=g)
    half = n_cent // 2
    c[:, half:2 * half] = c[:, :half] * (1 + torch.randint(-3, 4, (H * n_sub, half, 1), generator=g) * 2.0 ** -23)
    c = c.to(cuda)
    wide = torch.zeros(1, H, n, n_sub * d + 4, dtype=torch.bfloat16, device=cuda)
    wide[..., : n_sub * d] = k
    assert torch.equal(_assign(N, cuda, k, n_sub, d, c), _assign(N, cuda, wide[..., : n_sub * d], n_sub, d, c))


@pytest.mark.parametrize("d,n_sub,n_cent", [(8, 2, 256), (16, 2, 130), (64, 2, 64), (128, 1, 64)])
@pytest.mark.parametrize("copies", [2, 3, 4, 5, 9, 33, 64])
def test_equal_centres(cuda, d, n_sub, n_cent, copies):
    """Every centre `copies` times, in as many slots of the search: few are evaluated one by one, many by the matrix
    instructions again. The first of them is taken, in both forms, with the same sums; some keys are equal to a centre."""
    from sparse_attention_hub_amd import _native as N

    n, H = 1500, 2
    g = torch.Generator().manual_seed(copies)
    base = torch.randn(H * n_sub, max(1, n_cent // copies), d, generator=g).bfloat16().float()
    c = base.repeat(1, n_cent // base.shape[1] + 1, 1)[:, :n_cent].contiguous().to(cuda)
    k = torch.randn(1, H, n, n_sub * d, generator=g)
    for h in range(H):
        for s in range(n_sub):
            k[0, h, 700:900, s * d: (s + 1) * d] = base[h * n_sub + s, torch.randint(0, base.shape[1], (200,), generator=g)]
    k = k.bfloat16()
    wide = torch.zeros(1, H, n, n_sub * d + 4, dtype=torch.bfloat16, device=cuda)
    forms = (k.to(cuda), wide[..., : n_sub * d].copy_(k))
    top = k.float().abs().max().view(1).to(cuda)
    (codes, S, C), other = (_assign(N, cuda, f, n_sub, d, c, top) for f in forms)
    assert int(codes.max()) < base.shape[1]
    assert torch.equal(codes, other[0]) and torch.equal(S, other[1]) and torch.equal(C, other[2])


@pytest.mark.parametrize("d,n_sub,n_cent", [(8, 2, 64), (16, 2, 33), (64, 2, 64), (128, 1, 256)])  # the last: sums apart
def test_an_element_that_is_not_a_number_adds_nothing(cuda, d, n_sub, n_cent):
    """NaN as the only values that are not finite, which the largest |element| passes over: it counts as 0 in its centre's
    sums in the split form, the fp32 form and the launch of its own, and a whole run's centres are the same in both forms."""
    from sparse_attention_hub_amd import _native as N
    from sparse_attention_hub_amd.sparse_attention.research_attention.maskers.fixed.implementations.utils.pq_utils import kmeans_keys_batched

    n, H = 1500, 2
    g = torch.Generator().manual_seed(d)
    k = torch.randn(1, H, n, n_sub * d, generator=g)
    k[0, 0, 300, 3], k[0, 1, 301, 0], k[0, 1, 1499, d - 1] = float("nan"), float("nan"), float("nan")
    k[0, 0, 700:732, :d] = float("nan")
    k = k.bfloat16()
    wide = torch.zeros(1, H, n, n_sub * d + 4, dtype=torch.bfloat16, device=cuda)
    forms = (k.to(cuda), wide[..., : n_sub * d].copy_(k))
    c = torch.randn(H * n_sub, n_cent, d, generator=g).to(cuda)
    x = torch.nan_to_num(k.view(H, n, n_sub, d).permute(0, 2, 1, 3).reshape(-1, n, d).double())
    top = x.abs().max().float().view(1)
    fixed = torch.round(x * 2.0 ** (40 - math.frexp(float(top))[1])).to(torch.int64)  # exact: a power of two and 8 bits
    for form in forms:
        codes, S, C = _assign(N, cuda, form, n_sub, d, c, top.to(cuda))
        at = codes.permute(0, 2, 1).reshape(-1, n).long()
        assert torch.equal(S, torch.zeros_like(S).scatter_add_(1, at.unsqueeze(-1).expand(-1, -1, d), fixed))
        assert torch.equal(C, torch.zeros_like(C).scatter_add_(1, at, torch.ones_like(at, dtype=torch.int32)))
    runs = []
    for form in forms:
        codes = torch.zeros((1, H, n, n_sub), dtype=torch.uint8, device=cuda)
        centres, _ = kmeans_keys_batched(form, 0, n_sub, n_cent, 4, codes, n, seed=41)
        torch.cuda.synchronize()
        runs.append((centres.cpu(), codes.cpu()))
    assert torch.equal(torch.nan_to_num(runs[0][0], nan=1e30), torch.nan_to_num(runs[1][0], nan=1e30)) and torch.equal(runs[0][1], runs[1][1])


@pytest.mark.parametrize("d", [4, 8, 16, 64])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_a_centre_that_is_not_a_number_loses_alone(cuda, dtype, d):
    """Such a centre takes no key, and the others of its tile take theirs: as if it were far away."""
    from sparse_attention_hub_amd import _native as N

    g = torch.Generator().manual_seed(d)
    k = torch.randn(1, 2, 1200, 2 * d, generator=g).to(dtype).to(cuda)
    c = torch.randn(4, 70, d, generator=g).to(cuda)
    far = c.clone()
    for at in (0, 37, 68):  # slot 0 of a tile, and others
        c[:, at, d - 1] = float("nan")
        far[:, at] = 1e6
    assert torch.equal(_assign(N, cuda, k, 2, d, c), _assign(N, cuda, k, 2, d, far))


# numbers drawn: the generator hands out 312 at first, then 227 at a time, to 256 threads
@pytest.mark.parametrize("groups,n_cent", [(1, 1), (1, 256), (4, 78), (1, 227), (7, 77), (49, 11), (3, 255), (256, 3), (16, 256)])
def test_start_vectors_are_the_seeded_stratified_draw(cuda, groups, n_cent):
    from sparse_attention_hub_amd.sparse_attention.research_attention.maskers.fixed.implementations.utils.pq_utils import (
        gather_sub_vectors, kmeans_keys_batched, seeded_initial_centres,
    )

    n, d = 613, 8
    k = torch.randn(1, groups, n, d, generator=torch.Generator().manual_seed(groups)).to(torch.bfloat16)
    codes = torch.zeros((1, groups, n, 1), dtype=torch.uint8, device=cuda)
    centres, _ = kmeans_keys_batched(k.to(cuda), 0, 1, n_cent, 0, codes, n, seed=41)  # no iteration: the start itself
    torch.cuda.synchronize()
    want = gather_sub_vectors(k, 0, 1, seeded_initial_centres(groups, n, n_cent, 41, torch.device("cpu")))
    assert torch.equal(centres.cpu().reshape(-1), want.float().reshape(-1))
