"""What is known, guessed and asked about an additive mask, and whose buffers a step uses meanwhile: host logic, with the
native calls recorded instead of made."""
import threading

import pytest
import torch

from sparse_attention_hub_amd import _native as N
from sparse_attention_hub_amd import sparse_attention as sa
from sparse_attention_hub_amd.sparse_attention.research_attention import decode_plan
from sparse_attention_hub_amd.sparse_attention.research_attention.maskers.fixed.implementations.hashattention_top_k import (
    PackedSignatureCache,
)
from sparse_attention_hub_amd.sparse_attention.utils import mask_attention_utils as U
from sparse_attention_hub_amd.sparse_attention.utils.hashattention_utils import random_hat_weights

B, HQ, HKV, LK, D = 2, 4, 2, 400, 64
LOWEST = float(torch.finfo(torch.bfloat16).min)


class Recorder:
    """Native calls by name, the stream they were made on and the buffers that a chain's blocks name."""

    def __init__(self):
        self.stream, self.capturing, self.fails, self.fits = 0, False, None, 1
        self.calls, self.masks = [], {}

    def call(self, name, args):
        if self.fails is not None and name == "sah_run_chain":
            self.fails(N.AttentionArgs.from_address(args.attention).amask)
        if name == "sah_hash_decode_masked":
            if args.ask:
                args.fits = self.fits
                return
            hd = N.HashDecodeArgs.from_address(args.decode)
            self.calls.append((name, self.stream, {hd.rows.cols, hd.rows.cnt, args.tickets, N.HashSigArgs.from_address(hd.query_sig).codes},
                               N.HashDecodeArgs.from_buffer_copy(hd)))
        elif name == "sah_run_chain":
            used = {args.tickets}
            if args.select:
                se = N.SelectTopkArgs.from_address(args.select)
                used |= {se.keys, se.rows.cols, se.rows.cnt}
            if args.hash_decode:
                hd = N.HashDecodeArgs.from_address(args.hash_decode)
                used |= {hd.rows.cols, hd.rows.cnt, N.HashSigArgs.from_address(hd.query_sig).codes}
            if args.attention:
                at = N.AttentionArgs.from_address(args.attention)
                used |= {at.rows.cols, at.rows.cnt}
            self.calls.append((name, self.stream, used, bool(args.compact)))
        else:
            if name == "sah_amask_answer":
                m = self.masks[args.read.mask.amask]
                args.read.flags = (1 if bool((m != 0).any()) else 0) | (2 if bool(((m != 0) & (m != LOWEST)).any()) else 0)
            self.calls.append((name, self.stream, set(), None))

    def launches(self):
        return [c for c in self.calls if c[0] == "sah_hash_decode_masked" or c[0] == "sah_run_chain"]


@pytest.fixture
def device(monkeypatch):
    r = Recorder()
    words = threading.local()

    def answer_words(dev):
        if not hasattr(words, "pair"):
            words.pair = (torch.zeros(2, dtype=torch.int32), torch.zeros(1, dtype=torch.int64))
        return words.pair

    monkeypatch.setattr(torch.Tensor, "is_cuda", True, raising=False)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: r.capturing)
    monkeypatch.setattr(N, "call", r.call)
    monkeypatch.setattr(N, "stream_ptr", lambda device: r.stream)
    monkeypatch.setattr(N, "work_floats", lambda *a: 64)
    monkeypatch.setattr(N, "members_work_floats", lambda *a: 64)
    monkeypatch.setattr(U, "_answer_words", answer_words)
    monkeypatch.setattr(U, "_ANSWERS", U._AnswerWords())
    return r


def attention(chain):
    cfgs = [sa.SinkMaskerConfig(sink_size=4), sa.LocalMaskerConfig(window_size=32)]
    if chain == "oracle":
        cfgs.append(sa.OracleTopKConfig(heavy_size=20))
    elif chain == "hash":
        cfgs.append(sa.HashAttentionTopKMaskerConfig(
            heavy_size=20, hat_bits=32, hat_mlp_layers=3, hat_mlp_hidden_size=128, hat_mlp_activation="silu",
            hat_weights=random_hat_weights(1, HQ, D, 32, 3, 128, dtype=torch.bfloat16, seed=1)))
    ra = sa.ResearchAttention.create_from_config(sa.ResearchAttentionConfig(masker_configs=cfgs))
    ra.return_attention_weights = False
    return ra


class Session:
    """One sequence's steps: its caches, and a new mask tensor for every step."""

    def __init__(self, r, ra, chain, n=LK):
        self.r, self.ra, self.kept = r, ra, []
        self.meta = {}
        if chain == "hash":
            cache = PackedSignatureCache(B, HQ, 32, n + 4096, torch.device("cpu"))
            cache.n = n
            self.meta["key"] = {0: cache}
            self.cache = cache
        self.q = torch.zeros(B, HQ, 1, D, dtype=torch.bfloat16)
        self.k = torch.zeros(B, HKV, n + 64, D, dtype=torch.bfloat16)

    def mask(self, kind, n=LK, n_q=1):
        m = torch.zeros(B, 1, n_q, n, dtype=torch.bfloat16)
        if kind != "z":
            m[0, ..., :50] = LOWEST if kind == "h" else -1.0
        self.r.masks[m.data_ptr()] = m
        self.kept.append(m)
        return m

    def step(self, kind, stream=0, n=LK, mask=None):
        """The launches of one step under a new mask (or the given one): zero, hiding, general or none."""
        before = len(self.r.launches())
        m = mask if mask is not None else None if kind == "-" else self.mask(kind, n)
        self.r.stream = stream
        out = self.ra.custom_attention(None, self.q, self.k[:, :, :n], self.k[:, :, :n], m, D ** -0.5, 0.0,
                                       sparse_meta_data=self.meta, layer_idx=0)[0]
        self.kept.append((out, list(self.ra._plans.values())))  # (no address is given out twice)
        return self.r.launches()[before:]


@pytest.mark.parametrize("other", ["stream", "thread"])
@pytest.mark.parametrize("chain", ["fixed", "hash", "oracle"])
@pytest.mark.parametrize("order", ["zh", "zzh", "hz", "zhzh", "zzhhz", "zhhzz"])  # z: the unpadded session's turn, h: the padded one's
def test_sessions_that_are_not_ordered_share_no_buffers(device, chain, order, other):
    """An unpadded session on one stream or thread and a padded one of the same geometry on another: whatever is launched for
    the padded one, on a guess or not, uses nothing that the unpadded one uses."""
    ra = attention(chain)
    plain, padded = Session(device, ra, chain), Session(device, ra, chain)
    used = {"z": set(), "h": set()}
    for kind in order:
        if kind == "z":
            launches = plain.step("z", 1)
        elif other == "stream":
            launches = padded.step("h", 2)
        else:
            out = []
            t = threading.Thread(target=lambda: out.extend(padded.step("h", 1)))
            t.start()
            t.join()
            launches = out
        assert launches
        for _, _, buffers, _ in launches:
            used[kind] |= buffers - {None}
    assert used["z"] and used["h"] and used["z"].isdisjoint(used["h"])


@pytest.mark.parametrize("chain", ["fixed", "oracle"])
def test_sessions_in_turn_are_launched_once_a_step(device, chain):
    """The guess is the session's: padded and unpadded ones that one instance serves in turn are each guessed right. A session's
    own change of mask costs it one launch."""
    ra = attention(chain)
    plain, padded = Session(device, ra, chain), Session(device, ra, chain)
    for _ in range(3):
        assert len(plain.step("z")) == 1 and len(padded.step("h")) == 1
    assert [len(plain.step(kind)) for kind in "zhhz"] == [1, 2, 1, 1]  # (a zero mask is right under a plan that takes a mask)
    answers = [i for i, c in enumerate(device.calls) if c[0] == "sah_amask_answer"]
    launches = [i for i, c in enumerate(device.calls) if c[0] == "sah_run_chain"]
    assert launches[-1] < answers[-1]  # the step's answer is read with the step under way


def test_an_instance_guesses_nothing_from_another_one(device):
    first = attention("oracle")
    session = Session(device, first, "oracle")
    session.step("z")
    session.ra = attention("oracle")
    assert len(session.step("h")) == 1
    session.meta = None  # a chain that keeps nothing takes this, too
    assert [len(session.step(kind)) for kind in "hzh"] == [1, 1, 1]


def one_kernel(launches):
    return any(c[0] == "sah_hash_decode_masked" for c in launches)


@pytest.fixture
def compact_at_once(monkeypatch):
    monkeypatch.setattr(decode_plan, "_TWO_PLANE_KEYS", 0)
    monkeypatch.setattr(decode_plan, "_TWO_PLANE_STEPS", 0)


def test_compact_codes_of_two_streams_are_no_masked_steps(device, compact_at_once):
    """One stream has written most of the compact codes, another has added to them: a masked step on either would read what the
    other has written, and goes without them."""
    s = Session(device, attention("hash"), "hash")
    assert one_kernel(s.step("h", 1)) and one_kernel(s.step("h", 1))
    assert not one_kernel(s.step("h", 2))
    s.step("-", 2, LK + 40)
    assert s.cache.n_compact == LK + 40
    assert not one_kernel(s.step("h", 2, LK + 40)) and not one_kernel(s.step("h", 1, LK + 40))
    s.cache.reserve(s.cache.capacity + 1)  # other buffers, written anew
    assert one_kernel(s.step("h", 2, LK + 40)) and not one_kernel(s.step("h", 1, LK + 40))


def test_compact_buffers_belong_to_the_stream_that_clears_them(device, compact_at_once):
    s = Session(device, attention("hash"), "hash")
    device.fits = 0
    assert not one_kernel(s.step("h", 1))  # makes the buffers, and then has no use for them
    device.fits = 1
    assert not one_kernel(s.step("h", 2)) and one_kernel(s.step("h", 1))


@pytest.mark.parametrize("kind", ["z", "h"])
def test_a_guess_reads_no_compact_codes_of_another_stream(device, kind):
    s = Session(device, attention("hash"), "hash")
    s.step("z", 1)
    s.step("z", 1)
    before = len(device.calls)
    s.step(kind, 2)
    names = [c[0] for c in device.calls[before:]]
    assert "sah_run_chain" not in names[:names.index("sah_amask_answer")]
    assert s.cache.n_compact == LK


def test_a_captured_step_does_not_rely_on_what_its_mask_holds(device):
    s = Session(device, attention("hash"), "hash")
    m = s.mask("h")
    assert one_kernel(s.step("h", 1, mask=m)) and one_kernel(s.step("h", 1, mask=m))
    device.capturing = True
    assert not one_kernel(s.step("h", 1, mask=m))
    device.capturing = False
    assert one_kernel(s.step("h", 1, mask=m))


def test_what_a_launch_on_a_guess_raises(device):
    """The step's own error if the guess was right, nothing if it was wrong; memory for buffers of the guess's own is no one's."""
    tries = []

    def fail(amask):
        tries.append(amask)
        raise N.NativeLibraryError("device")

    s = Session(device, attention("oracle"), "oracle")
    s.step("z")
    device.fails = fail
    with pytest.raises(N.NativeLibraryError, match="device"):
        s.step("z")
    assert tries == [None] and not U._ANSWERS.open
    device.fails = lambda amask: fail(amask) if amask is None else None
    assert len(s.step("h")) == 1 and len(tries) == 2
    device.fails = None
    s.step("z")
    s.step("z")

    def out_of_memory(amask):
        device.fails = None
        raise torch.OutOfMemoryError("buffers")

    device.fails = out_of_memory
    assert len(s.step("z")) == 1


def test_a_mask_that_covers_nothing_of_the_call_is_launched_on_no_guess(device):
    s = Session(device, attention("oracle"), "oracle")
    s.step("z")
    s.step("z")
    before = len(device.launches())
    wide = torch.zeros(B + 1, 1, 1, LK, dtype=torch.bfloat16)
    device.masks[wide.data_ptr()] = wide
    names = len(device.calls)
    assert len(s.step("z", mask=wide)) == 1  # adds nothing anywhere
    assert [c[0] for c in device.calls[names:]][:2] == ["sah_amask_ask", "sah_amask_answer"]
    other = wide.clone().fill_(LOWEST)
    device.masks[other.data_ptr()] = other
    with pytest.raises(ValueError, match="does not cover"):
        s.step("h", mask=other)
    assert len(device.launches()) == before + 1


def test_a_call_that_fails_leaves_no_question_open(device, monkeypatch):
    """A mask of several queries is asked about while the maskers run: the answer is taken whatever becomes of them."""
    from sparse_attention_hub_amd.sparse_attention.research_attention import base

    s = Session(device, attention("fixed"), "fixed")
    m = s.mask("h", n_q=3)
    monkeypatch.setattr(base.Mask, "create_empty_mask", lambda *a, **k: (_ for _ in ()).throw(ValueError("masker")))
    with pytest.raises(ValueError, match="masker"):
        s.ra.custom_attention(None, torch.zeros(B, HQ, 3, D, dtype=torch.bfloat16), s.k[:, :, :LK], s.k[:, :, :LK], m, D ** -0.5, 0.0,
                              sparse_meta_data=s.meta, layer_idx=0)
    assert not U._ANSWERS.open and s.ra._mask_facts.known(m) == N.AMASK_NONZERO


def test_a_session_of_few_masked_steps_builds_no_compact_codes(device, monkeypatch):
    s = Session(device, attention("hash"), "hash")
    for _ in range(20):
        assert one_kernel(s.step("h"))
    assert s.cache.pos is None  # rows of this length never need them
    monkeypatch.setattr(decode_plan, "_TWO_PLANE_KEYS", LK - 1)
    s = Session(device, attention("hash"), "hash")
    for i in range(decode_plan._TWO_PLANE_STEPS + 2):
        launches = s.step("h")
        assert one_kernel(launches) and len(launches) == (2 if i == decode_plan._TWO_PLANE_STEPS else 1)
        assert bool(launches[-1][3].pos_codes) == (s.cache.pos is not None) == (i >= decode_plan._TWO_PLANE_STEPS)


def test_guesses_of_several_threads_make_one_plan_each(device):
    """Unpadded sessions of two streams in turn keep their plans; only so many are kept."""
    from sparse_attention_hub_amd.sparse_attention.research_attention import base

    ra = attention("oracle")
    sessions = [Session(device, ra, "oracle") for _ in range(2)]
    for _ in range(2):
        for stream, s in enumerate(sessions):
            s.step("z", stream)
    plans = dict(ra._plans)
    assert len(plans) == 3  # with the one of steps that are known to have no mask
    for _ in range(3):
        for stream, s in enumerate(sessions):
            s.step("z", stream)
    assert ra._plans == plans
    for stream in range(2 * base._GUESSED_PLANS):
        sessions[0].step("z", stream)
    assert len(ra._plans) == base._GUESSED_PLANS + 1


def test_a_saved_session_may_be_of_an_earlier_version(device):
    """A pickled signature cache holds the attributes its class had then."""
    s = Session(device, attention("hash"), "hash")
    for name in ("compact_stream", "masked_steps"):
        s.cache.__dict__.pop(name, None)
    assert one_kernel(s.step("h")) and len(s.step("-")) == 1
