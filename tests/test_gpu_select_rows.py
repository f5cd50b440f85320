"""`sah_select_topk` on 16-bit keys through the C ABI: more mask rows than compute units, where several share one, and few, which
have one to themselves. Every register form (candidates around each limit), the bracket taken from a sample and what happens
when it misses the threshold, lanes with more bracket keys than slots, ties, active columns that rank, repeated keys. Checked
against a stable sort."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _keys(kind, n_rows, pitch, g):
    j = torch.arange(pitch, device=g.device)
    if kind == "float":  # bf16 scores: sign and exponent in the high byte
        u = (torch.randn(n_rows, pitch, generator=g, device=g.device) * 20).to(torch.bfloat16).view(torch.int16).int() & 0xFFFF
        return torch.where(u >= 0x8000, 0xFFFF - u, u | 0x8000)
    if kind == "spread":
        return torch.randint(0, 65536, (n_rows, pitch), generator=g, device=g.device)
    if kind == "few":
        return torch.randint(1, 8, (n_rows, pitch), generator=g, device=g.device) * 16 + 0x8000
    if kind == "equal":
        return torch.full((n_rows, pitch), 0x8123, device=g.device)
    if kind[:6] in ("hidden", "hiding"):  # that share of the columns, the first or any, at the excluded key of hidden ones
        share, seen = int(kind[6:]) / 100, _keys("float", n_rows, pitch, g)
        return torch.where((j < share * pitch) if kind[:6] == "hidden" else (torch.rand(n_rows, pitch, generator=g, device=g.device) < share), 0x0080, seen)
    if kind == "zero":  # the smallest key, which missing candidates carry too
        return torch.where(torch.rand(n_rows, pitch, generator=g, device=g.device) < 0.02, 7, 0)
    # "striped": what is large depends on the place inside a group of eight, from which the sample takes one
    base = torch.randint(0, 4096, (n_rows, pitch), generator=g, device=g.device)
    return base + torch.where(j % 8 == 0, 0xC000, 0x4000)


@pytest.mark.parametrize("n_cand,k,kind,n_active,ek", [
    (5, 2, "spread", 1, 0),
    (511, 40, "float", 30, 0x0080),
    (513, 513, "spread", 20, 0),
    (4096, 205, "striped", 64, 0x0080),       # one chunk a wave: the sample sees the large keys alone
    (4097, 1, "float", 64, 0x0080),
    (8192, 900, "few", 100, 0x8040),          # active columns tie with the threshold
    (8193, 900, "few", 100, 0xFFFF),          # ... and rank above it
    (16384, 8192, "float", 300, 0x0080),      # a threshold near zero: a bracket of more key values than counters
    (16385, 820, "float", 300, 0x0080),
    (20480, 1024, "equal", 300, 0x0080),
    (20481, 300, "zero", 300, 0),
    (32768, 1638, "float", 640, 0x0080),
    (32769, 1638, "striped", 640, 0x0080),
    (36864, 2048, "few", 640, 0x0080),        # more bracket keys in a lane than slots
    (36865, 2048, "float", 640, 0x0080),
    (65536, 3000, "float", 640, 0x0080),
    (65537, 3000, "spread", 640, 0x0080),
    (131072, 2621, "float", 1152, 0x0080),
    (131073, 2621, "float", 1152, 0x0080),    # keys read from memory in every pass
])
@pytest.mark.parametrize("offset", [0, 13])
def test_rows_share_a_compute_unit(cuda, n_cand, k, kind, n_active, ek, offset):
    _select(cuda, 258, n_cand, k, kind, n_active, ek, offset)


@pytest.mark.parametrize("n_rows", [3, 258])  # sixteen waves a row, and eight
@pytest.mark.parametrize("n_cand,k,kind", [
    (16384, 900, "float"), (16385, 900, "float"), (32768, 1638, "few"), (32769, 1638, "float"), (65536, 3000, "striped"),
    (65537, 3000, "float"),
    (20481, 1200, "hidden90"), (20481, 1200, "hiding97"),
    (33000, 300, "equal"), (33280, 1500, "equal"),  # the last wave's two chunks fit its slots, the others' do not
    (36800, 1900, "hidden90"), (41000, 1500, "hidden97"), (41000, 3000, "hiding97"), (65500, 2000, "few"), (66000, 3500, "hiding90"),
    (66100, 1, "equal"), (98000, 4800, "hidden97"), (131072, 9000, "hidden90"), (131072, 6000, "equal"), (131072, 60000, "few"),
])
def test_rows_of_repeated_keys(cuda, n_rows, n_cand, k, kind):
    """Lanes that add to one counter do it together, waves full of the bracket's keys count them where they are."""
    _select(cuda, n_rows, n_cand, k, kind, 200, 0x0080, 5)


def _select(cuda, n_rows, n_cand, k, kind, n_active, ek, offset):
    from sparse_attention_hub_amd import _native as N

    n_keys = n_cand + offset
    pitch = (n_cand + 7) // 8 * 8
    g = torch.Generator(device=cuda).manual_seed(n_cand + k)
    keys = _keys(kind, n_rows, pitch, g)
    active = torch.rand(n_rows, n_keys, generator=g, device=cuda).argsort(dim=1)[:, :n_active]
    flags = torch.zeros(n_rows, n_keys, dtype=torch.bool, device=cuda).scatter_(1, active, True)
    n_words, cap = (n_keys + 31) // 32, min(n_keys, n_active + k)

    def words(f):
        padded = torch.zeros(n_rows, n_words * 32, dtype=torch.int64, device=cuda)
        padded[:, :n_keys] = f
        w = (padded.view(n_rows, n_words, 32) << torch.arange(32, device=cuda)).sum(-1)
        return torch.where(w >= 1 << 31, w - (1 << 32), w).to(torch.int32)

    cols = torch.full((n_rows, cap), -1, dtype=torch.int32, device=cuda)
    cols[:, :n_active] = active
    cnt = torch.full((n_rows,), n_active, dtype=torch.int32, device=cuda)
    bitmap = words(flags)
    stored = torch.where(keys >= 1 << 15, keys - (1 << 16), keys).to(torch.int16).contiguous()
    rows = N.Rows(cols.data_ptr(), cnt.data_ptr(), None, bitmap.data_ptr(), n_rows, cap, n_keys, n_words)
    N.call("sah_select_topk", N.SelectTopkArgs(rows, stored.data_ptr(), pitch, 16, n_cand, offset, k, ek, 0, 0, 0, N.stream_ptr(cuda)))
    torch.cuda.synchronize()

    mine = flags[:, offset:]
    eff = torch.where(mine, ek, keys[:, :n_cand])
    best = torch.sort(eff, dim=1, descending=True, stable=True).indices[:, :k]
    chosen = torch.zeros_like(mine).scatter_(1, best, True) & ~mine
    want = flags.clone()
    want[:, offset:] |= chosen
    assert torch.equal(cnt.long(), want.sum(1)), "counts"
    assert torch.equal(bitmap, words(want)), "bitmaps"
    at = torch.arange(cap, device=cuda)
    listed = torch.zeros(n_rows, n_keys + 1, dtype=torch.int32, device=cuda)
    listed.scatter_add_(1, torch.where(at < cnt[:, None], cols, n_keys).long(), torch.ones_like(cols))
    assert torch.equal(listed[:, :n_keys], want.to(torch.int32)), "every column once in its row's list"
    assert torch.equal(cols[:, :n_active].long(), active), "entries from before stay where they were"
