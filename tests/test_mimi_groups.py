"""Calls of several frames run them through the codec together (mimi_engine.hip, MimiGroup): every output bit and the streaming state must be
those of the same frames one by one - across the attention ring's wrap, between groups of different sizes, around single frames, after a
reset, under an exec mask (frame by frame if it leaves a stream out), after and from a snapshot - and that they were run together."""
import ctypes
import gc
from dataclasses import replace

import pytest
import torch

from moshi_amd import MimiModel, tiny_mimi_config
from moshi_amd.config import MimiConfig
from moshi_amd.weights import random_mimi_state_dict


def check_calls_equal_frames(make, device, cfg, B, sizes, K=4):
    sd = random_mimi_state_dict(cfg, seed=5, device=device)
    gen = torch.Generator().manual_seed(B)
    n, fs = sum(sizes), cfg.frame_size
    x = (0.3 * torch.randn(B, 1, n * fs, generator=gen)).to(device)
    q = torch.randint(0, cfg.q_bins, (B, K, n), generator=gen).to(device)
    a, b = make(sd, cfg, K, B), make(sd, cfg, K, B)

    def same(at, size, what, a=a, rows=slice(None)):
        part = x[..., at * fs:(at + size) * fs].contiguous()
        codes = torch.cat([b.encode(x[..., f * fs:(f + 1) * fs].contiguous()) for f in range(at, at + size)], -1)
        assert torch.equal(a.encode(part)[rows], codes[rows]), f"{what}: codes of frames {at}..{at + size}"
        pcm = torch.cat([b.decode(q[..., f:f + 1].contiguous()) for f in range(at, at + size)], -1)
        assert torch.equal(a.decode(q[..., at:at + size].contiguous())[rows], pcm[rows]), f"{what}: samples of frames {at}..{at + size}"

    def together(m):                                           # has this stream run a group in each direction (True), or none at all (False)?
        kernels = [{k for _, k in m.launch_list(which)} for which in ("encode_group", "decode_group")]
        assert bool(kernels[0]) == bool(kernels[1]) and all("k_mimi_group_rope" in k for k in kernels if k)
        return bool(kernels[0])
    with a.streaming(B), b.streaming(B):
        at = 0
        for size in sizes:
            same(at, size, "stream")
            at += size
            assert together(a) == any(n > 1 for n in sizes[:sizes.index(size) + 1])
        assert not together(b)
        for m in (a, b):
            m.reset_streaming()
        same(0, sizes[0], "after a reset")
        state = a.get_streaming_state()
        b.set_streaming_state(state)
        same(0, sizes[-1], "after a snapshot")
        b.set_streaming_state(state)
        c = make(sd, cfg, K, B)
        with c.streaming(B):
            c.set_streaming_state(state)
            same(0, sizes[-1], "from a snapshot", c)
            assert together(c) == (sizes[-1] > 1)
    if B > 1:
        mask = (torch.arange(B) % 2 == 0)
        with a.streaming(B), b.streaming(B):
            for m in (a, b):
                m.set_exec_mask(mask.to(device))
            same(0, 2, "under a mask", rows=mask)
            assert not together(a)
            for m in (a, b):
                m.reset_streaming(~mask.to(device))            # the others again: they start here
            same(2, 2, "after a reset of those that stood still")
            assert together(a)
            for m in (a, b):
                m.set_exec_mask(torch.ones(B, dtype=torch.bool, device=device))
            same(1, 3, "under a mask of all streams")
        with a.streaming(B):
            a.set_exec_mask(torch.ones(B, dtype=torch.bool, device=device))
            a.encode(x[..., :2 * fs].contiguous()), a.decode(q[..., :2].contiguous())
            assert together(a)
    whole = a.encode(x)                                        # a fresh, temporary stream
    with b.streaming(B):
        assert torch.equal(whole, torch.cat([b.encode(x[..., f * fs:(f + 1) * fs].contiguous()) for f in range(n)], -1)), "temporary stream"


@pytest.mark.parametrize("B,sizes", [(1, (2, 1, 7, 3)), (3, (5, 1, 4))])
def test_tiny_calls_equal_frames(sim_lib, B, sizes):
    check_calls_equal_frames(lambda sd, cfg, K, mb: MimiModel(sd, cfg, device="cpu", max_batch=mb, num_codebooks=K, lib=sim_lib), "cpu", tiny_mimi_config(), B, sizes)


@pytest.mark.parametrize("ff", [60, 63, 65])
def test_calls_equal_frames_where_operands_are_padded(sim_lib, monkeypatch, ff):
    """A feed-forward width that is no multiple of 8: the packed operand between its two products has rows that nobody stores, which must
    not hold what the memory held before (the simulator allocates NaN; a used slab is made to with MMI_DEBUG_POISON)."""
    monkeypatch.setenv("MMI_DEBUG_POISON", "1")
    cfg = replace(tiny_mimi_config(), tr_dim_feedforward=ff)
    check_calls_equal_frames(lambda sd, cfg, K, mb: MimiModel(sd, cfg, device="cpu", max_batch=mb, num_codebooks=K, lib=sim_lib), "cpu", cfg, 2, (3, 1, 4))


def sim_bytes(lib):
    lib.cdll.hipsim_live_bytes.restype = lib.cdll.hipsim_peak_bytes.restype = ctypes.c_ulonglong
    return int(lib.cdll.hipsim_live_bytes())


def test_memory_of_groups_is_the_largest_one_s(sim_lib):
    """What groups hold is what the largest of them needs, whatever sizes came before it, and never two of them at a time; it is given
    back by a stream that runs single frames, and with the handle.  (256 channels: buffers of more than 32 MB)"""
    cfg = replace(tiny_mimi_config(), channels=256, n_filters=2, ratios=[8, 8, 4, 3], sample_rate=768 * 25, tr_num_layers=1)
    sd = random_mimi_state_dict(cfg, seed=1, device="cpu")

    def held(sizes, decode):
        gc.collect()
        empty = sim_bytes(sim_lib)
        m = MimiModel(sd, cfg, device="cpu", max_batch=1, num_codebooks=2, lib=sim_lib)
        before = sim_bytes(sim_lib)
        sim_lib.cdll.hipsim_peak_bytes()

        def call(n):
            if decode:
                m.decode(torch.zeros(1, 2, n, dtype=torch.int64))
            else:
                m.encode(torch.zeros(1, cfg.channels, n * cfg.frame_size))
        with m.streaming(1):
            for n in sizes:
                call(n)
            most = sim_lib.cdll.hipsim_peak_bytes() - before
            streaming = sim_bytes(sim_lib) - before
        kept = sim_bytes(sim_lib) - before
        with m.streaming(1):
            call(1)
        given_back = sim_bytes(sim_lib) == before
        del m
        gc.collect()
        assert sim_bytes(sim_lib) == empty
        return streaming, kept, most, given_back

    for decode in (False, True):
        alone, alone_kept, alone_most, back = held([28], decode)
        assert back and alone_kept <= alone == alone_most
        assert held([24, 26, 28, 3, 25, 2], decode) == (alone, alone_kept, alone_most, True)


def test_calls_go_frame_by_frame_where_memory_is_short(sim_lib):
    """No memory for a group's buffers, from the start or when a call is longer than the ones before: the call gives what its frames give
    one by one, the next ones too, and nothing of the attempt stays allocated."""
    cfg = tiny_mimi_config()
    sd = random_mimi_state_dict(cfg, seed=5, device="cpu")
    gen = torch.Generator().manual_seed(3)
    n, fs, set_memory = 20, cfg.frame_size, sim_lib.cdll.hipsim_set_memory
    set_memory.argtypes = [ctypes.c_ulonglong]
    x = 0.3 * torch.randn(2, 1, n * fs, generator=gen)
    q = torch.randint(0, cfg.q_bins, (2, 4, n), generator=gen)
    a, b = (MimiModel(sd, cfg, device="cpu", max_batch=2, num_codebooks=4, lib=sim_lib) for _ in range(2))
    for first in (0, 2):                                       # frames of a call that finds memory
        with a.streaming(2), b.streaming(2):
            codes = [b.encode(x[..., f * fs:(f + 1) * fs].contiguous()) for f in range(n)]
            pcm = [b.decode(q[..., f:f + 1].contiguous()) for f in range(n)]
            empty = sim_bytes(sim_lib)
            try:
                at = 0
                for size in (first, 5, 1, 3, n - 9 - first):
                    part = slice(at, at + size)
                    for call, want, arg in ((a.encode, codes, x[..., at * fs:(at + size) * fs]), (a.decode, pcm, q[..., part])):
                        if at or not first:
                            set_memory(sim_bytes(sim_lib))
                        if size:
                            assert torch.equal(call(arg.contiguous()), torch.cat(want[part], -1)), (first, at)
                    assert (sim_bytes(sim_lib) > empty) == (first > at)
                    at += size
            finally:
                set_memory(0)


@pytest.mark.parametrize("blocking", [False, True])
def test_calls_while_another_thread_captures(sim_lib, blocking):
    """While another thread captures, the runtime neither allocates nor frees, and a capture that blocks the null stream does not let it be
    asked: single frames go on beside an earlier stream's group memory, calls of several go frame by frame, and the memory is given back
    by the first single frame after it."""
    cfg = tiny_mimi_config()
    sd = random_mimi_state_dict(cfg, seed=5, device="cpu")
    fs, n, capture_elsewhere = cfg.frame_size, 6, sim_lib.cdll.hipsim_set_capture_elsewhere
    x = 0.3 * torch.randn(1, 1, n * fs, generator=torch.Generator().manual_seed(4))
    q = torch.randint(0, cfg.q_bins, (1, 4, n), generator=torch.Generator().manual_seed(7))
    m, other = (MimiModel(sd, cfg, device="cpu", max_batch=1, num_codebooks=4, lib=sim_lib) for _ in range(2))
    codes, pcm = other.encode(x), other.decode(q)
    before = sim_bytes(sim_lib)
    with m.streaming(1):
        stream = sim_bytes(sim_lib) - before
    m.encode(x[..., :2 * fs].contiguous()), m.decode(q[..., :2].contiguous())
    assert sim_bytes(sim_lib) > before
    with m.streaming(1):
        try:
            capture_elsewhere(1 + blocking)
            for f, k in ((0, 1), (1, 1), (2, 3)):
                assert torch.equal(m.encode(x[..., f * fs:(f + k) * fs].contiguous()), codes[..., f:f + k])
                assert torch.equal(m.decode(q[..., f:f + k].contiguous()), pcm[..., f * fs:(f + k) * fs])
        finally:
            capture_elsewhere(0)
        assert torch.equal(m.encode(x[..., 5 * fs:].contiguous()), codes[..., 5:]) and torch.equal(m.decode(q[..., 5:].contiguous()), pcm[..., 5 * fs:])
        assert sim_bytes(sim_lib) == before + stream


def test_a_stream_starts_where_groups_hold_the_memory(sim_lib):
    """What groups of an earlier stream have left is given back where the next stream would not start beside it."""
    cfg = tiny_mimi_config()
    sd = random_mimi_state_dict(cfg, seed=5, device="cpu")
    set_memory = sim_lib.cdll.hipsim_set_memory
    set_memory.argtypes = [ctypes.c_ulonglong]
    m = MimiModel(sd, cfg, device="cpu", max_batch=2, num_codebooks=4, lib=sim_lib)
    before = sim_bytes(sim_lib)
    x = torch.zeros(2, 1, 8 * cfg.frame_size)
    with m.streaming(2):
        stream = sim_bytes(sim_lib) - before
    want = m.encode(x)
    assert sim_bytes(sim_lib) > before
    try:
        set_memory(before + stream)
        with m.streaming(2):
            assert sim_bytes(sim_lib) == before + stream
            assert torch.equal(m.encode(x), want)
        set_memory(before + stream - 1)
        with pytest.raises(RuntimeError):
            m.streaming_forever(2)
        assert sim_bytes(sim_lib) == before
    finally:
        set_memory(0)
    assert torch.equal(m.encode(x), want)


def check_files_in_a_row(make, device, cfg, lengths, K=4):
    """A handle keeps what one file's stream has built for the next one: every file gives the bits that a fresh handle gives - after files of
    other lengths, of NaNs and infinities, of more rows, after a stream of the caller's own, with other codebooks, in either direction."""
    sd = random_mimi_state_dict(cfg, seed=11, device=device)
    gen = torch.Generator().manual_seed(13)
    m, fs = make(sd, cfg, K, 3), cfg.frame_size

    def file(B, n, k=K, bad=None):
        x = (0.3 * torch.randn(B, 1, n * fs - 5, generator=gen)).to(device)
        q = torch.randint(0, cfg.q_bins, (B, k, n), generator=gen).to(device)
        if bad is not None:
            x[:, :, ::7] = bad
        return x, q

    def same(x, q):
        fresh = make(sd, cfg, m.num_codebooks, 3)
        for got, want in ((m.encode(x), fresh.encode(x)), (m.decode(q), fresh.decode(q)), (m.encode_to_latent(x, quantize=False), fresh.encode_to_latent(x, quantize=False))):
            assert torch.equal(got, want) or (torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(), want.nan_to_num()))
    for n in lengths:
        same(*file(1, n))
    for bad in (float("nan"), float("inf")):                   # (the longest goes round the ring; behind it a file that is as long, shorter ones, one frame)
        for n in (max(lengths), lengths[0] - 1, 1, max(lengths)):
            same(*file(1, max(lengths), bad=bad)), same(*file(1, n))
    same(*file(2, 3)), same(*file(2, 3)), same(*file(1, lengths[0]))
    x, q = file(1, 3)
    with m.streaming(1):
        m.encode(x[..., :fs].contiguous()), m.decode(q)
    same(x, q)
    m.set_num_codebooks(2)
    same(x, q[:, :2]), same(x, q[:, :1])
    with pytest.raises(AssertionError, match="codebooks"):
        m.decode(torch.zeros(1, cfg.q_n_q + 1, 2, dtype=torch.int64, device=device))
    same(x, q[:, :2])


# (poison: what a file may not see of the one before it is NaNs in front of its reset, in the decoder too, whose inputs are always finite)
@pytest.mark.parametrize("poison", [False, True])
def test_files_in_a_row(sim_lib, monkeypatch, poison):
    if poison:
        monkeypatch.setenv("MMI_DEBUG_POISON", "1")
    cfg = tiny_mimi_config()
    m = MimiModel(random_mimi_state_dict(cfg, seed=5, device="cpu"), cfg, device="cpu", max_batch=1, num_codebooks=4, lib=sim_lib)
    before = sim_bytes(sim_lib)
    m.encode(torch.zeros(1, 1, cfg.frame_size))
    assert sim_bytes(sim_lib) > before                         # (something is kept)
    assert 2 * 14 > cfg.tr_context
    check_files_in_a_row(lambda sd, cfg, K, mb: MimiModel(sd, cfg, device="cpu", max_batch=mb, num_codebooks=K, lib=sim_lib), "cpu", cfg, (4, 1, 4, 14))


@pytest.mark.gpu
@pytest.mark.parametrize("poison", [False, True])
def test_full_size_files_in_a_row(monkeypatch, poison):
    if poison:
        monkeypatch.setenv("MMI_DEBUG_POISON", "1")
    check_files_in_a_row(lambda sd, cfg, K, mb: MimiModel(sd, cfg, device="cuda", max_batch=mb, num_codebooks=K), "cuda", MimiConfig(), (40, 1, 40, 170, 9), K=8)


def test_what_a_file_leaves_goes_with_the_next_stream(sim_lib):
    cfg = tiny_mimi_config()
    sd = random_mimi_state_dict(cfg, seed=5, device="cpu")
    gc.collect()
    empty = sim_bytes(sim_lib)
    m = MimiModel(sd, cfg, device="cpu", max_batch=2, num_codebooks=4, lib=sim_lib)
    before = sim_bytes(sim_lib)
    with m.streaming(2):
        stream = sim_bytes(sim_lib) - before
    m.encode(torch.zeros(1, 1, cfg.frame_size))
    assert 0 < sim_bytes(sim_lib) - before <= 128 << 20
    assert not m.is_streaming
    with m.streaming(2):
        assert sim_bytes(sim_lib) == before + stream
    assert sim_bytes(sim_lib) == before
    m.encode(torch.zeros(1, 1, cfg.frame_size))
    del m
    gc.collect()
    assert sim_bytes(sim_lib) == empty


@pytest.mark.parametrize("blocking", [False, True])
def test_files_while_another_thread_captures(sim_lib, blocking):
    """The runtime does not free while another thread captures: what a file's stream has left is not lost then, whether the next file is of
    other rows (it fails, as without an earlier one), of the same rows (it fails where the null stream cannot be asked, and the one behind the
    capture finds everything still there) or the handle goes."""
    cfg = tiny_mimi_config()
    sd = random_mimi_state_dict(cfg, seed=5, device="cpu")
    fs, capture_elsewhere = cfg.frame_size, sim_lib.cdll.hipsim_set_capture_elsewhere
    x = 0.3 * torch.randn(2, 1, fs, generator=torch.Generator().manual_seed(4))
    gc.collect()
    empty = sim_bytes(sim_lib)
    m = MimiModel(sd, cfg, device="cpu", max_batch=2, num_codebooks=4, lib=sim_lib)
    before = sim_bytes(sim_lib)
    want = m.encode(x[:1])
    kept = sim_bytes(sim_lib)
    assert kept > before
    try:
        for _ in range(2):
            capture_elsewhere(1 + blocking)
            if blocking:
                with pytest.raises(RuntimeError):
                    m.encode(x[:1])
            else:
                assert torch.equal(m.encode(x[:1]), want)
            assert sim_bytes(sim_lib) == kept and not m.is_streaming
            with pytest.raises(RuntimeError):
                m.encode(x)
            capture_elsewhere(0)
            assert torch.equal(m.encode(x[:1]), want) and sim_bytes(sim_lib) == kept
        other = MimiModel(sd, cfg, device="cpu", max_batch=2, num_codebooks=4, lib=sim_lib)
        other.encode(torch.cat([x[:1]] * 9, -1))               # (with a group's memory)
        capture_elsewhere(1 + blocking)
        del m, other
        gc.collect()
        assert sim_bytes(sim_lib) > empty
    finally:
        capture_elsewhere(0)
    MimiModel(sd, cfg, device="cpu", max_batch=2, num_codebooks=4, lib=sim_lib)
    gc.collect()
    assert sim_bytes(sim_lib) == empty


def test_a_file_whose_wait_fails(sim_lib):
    """A call on a file that cannot wait for the device raises.  Its stream has ended then, for the model and the engine; what it has left stays
    until a wait succeeds (work on the device may use it), and the next file is a fresh one."""
    cfg = tiny_mimi_config()
    sd = random_mimi_state_dict(cfg, seed=5, device="cpu")
    fs, sync_fails = cfg.frame_size, sim_lib.cdll.hipsim_set_sync_fails
    x = 0.3 * torch.randn(1, 1, 2 * fs, generator=torch.Generator().manual_seed(4))
    gc.collect()
    empty = sim_bytes(sim_lib)
    m = MimiModel(sd, cfg, device="cpu", max_batch=1, num_codebooks=4, lib=sim_lib)
    want = m.encode(x)
    kept = sim_bytes(sim_lib)
    for begin in (lambda: m.encode(x), lambda: m.decode(want), lambda: m.streaming_forever(1)):
        try:
            sync_fails(1)
            for call in (lambda: m.encode(x), begin):
                with pytest.raises(RuntimeError, match="hipDeviceSynchronize"):
                    call()
                assert not m.is_streaming and sim_bytes(sim_lib) == kept
        finally:
            sync_fails(0)
        assert torch.equal(m.encode(x), want) and sim_bytes(sim_lib) == kept
    with m.streaming(1):
        assert torch.equal(m.encode(x), want)
    del m
    gc.collect()
    assert sim_bytes(sim_lib) == empty


def test_what_a_file_leaves_goes_where_memory_is_short(sim_lib):
    """The state and the groups' buffers that a file has left go when an allocation finds no memory - another handle's stream, its groups, a new
    handle - and when they are asked to (a stop while not streaming).  The handle's next file is what it was, and nothing goes from one that streams."""
    cfg = replace(tiny_mimi_config(), n_filters=4, ratios=[4, 4, 3, 2], sample_rate=96 * 25)
    sd = random_mimi_state_dict(cfg, seed=5, device="cpu")
    set_memory, fs = sim_lib.cdll.hipsim_set_memory, cfg.frame_size
    set_memory.argtypes = [ctypes.c_ulonglong]
    x = 0.3 * torch.randn(1, 1, 9 * fs, generator=torch.Generator().manual_seed(4))
    gc.collect()
    empty = sim_bytes(sim_lib)
    a, b = (MimiModel(sd, cfg, device="cpu", max_batch=1, num_codebooks=4, lib=sim_lib) for _ in range(2))
    handle = (sim_bytes(sim_lib) - empty) // 2
    before = sim_bytes(sim_lib)
    codes = b.encode(x)
    pcm = b.decode(codes)
    all_of_it = sim_bytes(sim_lib) - before
    with b.streaming(1):
        b.encode(x[..., :fs].contiguous()), b.decode(codes[..., :1].contiguous())      # single frames: the groups' buffers go
        stream = sim_bytes(sim_lib) - before
    assert sim_bytes(sim_lib) == before and stream < all_of_it

    def leave():
        assert torch.equal(a.encode(x), codes) and torch.equal(a.decode(codes), pcm)
        assert sim_bytes(sim_lib) - before == all_of_it
    try:
        leave()
        set_memory(before + all_of_it)
        with b.streaming(1):                                   # its state: what a has left goes
            assert sim_bytes(sim_lib) - before == stream
        set_memory(0)
        leave()
        with b.streaming(1):
            set_memory(before + all_of_it + stream)
            assert torch.equal(b.encode(x), codes)             # its group: the same
            assert "k_mimi_group_rope" in {k for _, k in b.launch_list("encode_group")}
            assert sim_bytes(sim_lib) - before < all_of_it + stream
            set_memory(sim_bytes(sim_lib))
            with pytest.raises(RuntimeError):                  # a stream keeps what it has
                a.encode(x)
            assert torch.equal(b.decode(codes), pcm)
        set_memory(0)
        assert torch.equal(b.encode(x[..., :fs].contiguous()), codes[..., :1])
        leave_b = sim_bytes(sim_lib) - before
        set_memory(before + leave_b + handle - 1)
        c = MimiModel(sd, cfg, device="cpu", max_batch=1, num_codebooks=4, lib=sim_lib)
        assert sim_bytes(sim_lib) == before + handle
        set_memory(0)
        assert torch.equal(c.encode(x), codes) and torch.equal(b.encode(x), codes)
        for m in (b, c):
            sim_lib.check(sim_lib.mmi_mimi_streaming_stop(m._handle))
        assert sim_bytes(sim_lib) == before + handle
    finally:
        set_memory(0)
    assert torch.equal(a.encode(x), codes) and torch.equal(c.decode(codes), pcm)
    del a, b, c, m
    gc.collect()
    assert sim_bytes(sim_lib) == empty


@pytest.mark.parametrize("what", ["duplex", "batcher"])
def test_what_a_file_leaves_goes_for_a_pipeline(sim_lib, what):
    """A duplex pipeline and a session batcher ask for memory of their own, beside the models': what other handles' files have left goes for those too."""
    from moshi_amd.batcher import SessionBatcher
    from moshi_amd.duplex import DuplexStream
    from moshi_amd.lm import LMGen
    from tests.batcher_cases import tiny_pair
    cfg, set_memory = tiny_mimi_config(), sim_lib.cdll.hipsim_set_memory
    set_memory.argtypes = [ctypes.c_ulonglong]
    sd = random_mimi_state_dict(cfg, seed=5, device="cpu")
    others = [MimiModel(sd, cfg, device="cpu", max_batch=1, num_codebooks=4, lib=sim_lib) for _ in range(4)]
    mimi, lm, _, _ = tiny_pair("cpu", sim_lib, 2)
    gen = LMGen(lm, use_sampling=False)
    gc.collect()
    before = sim_bytes(sim_lib)

    def leave(spare=0):
        for m in others:
            m.encode(torch.zeros(1, 1, cfg.frame_size))
        set_memory(sim_bytes(sim_lib) + spare)
    try:
        if what == "batcher":                                  # its own buffers come before the models' streams
            with mimi.streaming(2), gen.streaming(2):
                streams = sim_bytes(sim_lib)
            with SessionBatcher(mimi, lm, 2, use_sampling=False):
                own = sim_bytes(sim_lib) - streams             # (half of it pinned host memory, which the simulator counts too, and comes first)
            leave(own // 2)
            with SessionBatcher(mimi, lm, 2, use_sampling=False) as b:
                assert b.step() == 0
        else:
            with mimi.streaming(2), gen.streaming(2):
                leave()
                d = DuplexStream(mimi, gen)
                d.join()
                del d
    finally:
        set_memory(0)
    gc.collect()
    assert sim_bytes(sim_lib) == before


def test_a_snapshot_of_another_stream_is_reset_where_it_was_loaded(sim_lib):
    """The tables of where a stream's histories lie are not part of what a snapshot brings: a reset behind a load clears the histories of the
    stream it is called on, and leaves the one that the snapshot came from alone."""
    cfg = tiny_mimi_config()
    sd = random_mimi_state_dict(cfg, seed=5, device="cpu")
    fs = cfg.frame_size
    x = 0.3 * torch.randn(1, 1, 9 * fs, generator=torch.Generator().manual_seed(6))
    q = torch.randint(0, cfg.q_bins, (1, 4, 9), generator=torch.Generator().manual_seed(7))
    a, b = (MimiModel(sd, cfg, device="cpu", max_batch=1, num_codebooks=4, lib=sim_lib) for _ in range(2))
    codes, pcm = b.encode(x), b.decode(q)
    with a.streaming(1), b.streaming(1):
        a.encode(x[..., :3 * fs].contiguous()), a.decode(q[..., :3].contiguous())
        b.set_streaming_state(a.get_streaming_state())
        b.reset_streaming()
        assert torch.equal(a.encode(x[..., 3 * fs:].contiguous()), codes[..., 3:])
        assert torch.equal(a.decode(q[..., 3:].contiguous()), pcm[..., 3 * fs:])
        assert torch.equal(b.encode(x), codes) and torch.equal(b.decode(q), pcm)


def test_a_failed_call_is_reported_once(sim_lib):
    """A failure of the runtime stays its last error until it is taken: it must not fail the next call, of this handle or another's."""
    cfg = tiny_mimi_config()
    sd = random_mimi_state_dict(cfg, seed=5, device="cpu")
    set_memory = sim_lib.cdll.hipsim_set_memory
    set_memory.argtypes = [ctypes.c_ulonglong]
    a = MimiModel(sd, cfg, device="cpu", max_batch=1, num_codebooks=4, lib=sim_lib)
    x = torch.zeros(1, 1, cfg.frame_size)
    with a.streaming(1):
        want = a.encode(x)
        a.reset_streaming()
        try:
            set_memory(sim_bytes(sim_lib) + 4096)
            with pytest.raises(RuntimeError):
                MimiModel(sd, cfg, device="cpu", max_batch=1, num_codebooks=4, lib=sim_lib)
        finally:
            set_memory(0)
        assert torch.equal(a.encode(x), want)


def test_a_group_does_not_need_the_frame_program_s_capture(sim_lib, monkeypatch):
    """The capture behind a group's launches is for a later call: the simulator cannot capture, which a call of several frames does not
    notice (its state has moved on by then), and a single frame does."""
    cfg = tiny_mimi_config()
    sd = random_mimi_state_dict(cfg, seed=5, device="cpu")
    x = 0.3 * torch.randn(1, 1, 7 * cfg.frame_size, generator=torch.Generator().manual_seed(4))
    want = MimiModel(sd, cfg, device="cpu", max_batch=1, num_codebooks=4, lib=sim_lib).encode(x)
    monkeypatch.delenv("MMI_NO_GRAPH")
    m = MimiModel(sd, cfg, device="cpu", max_batch=1, num_codebooks=4, lib=sim_lib)
    with m.streaming(1):
        got = [m.encode(x[..., f * cfg.frame_size:(f + n) * cfg.frame_size].contiguous()) for f, n in ((0, 3), (3, 4))]
        assert torch.equal(torch.cat(got, -1), want)
        with pytest.raises(RuntimeError, match="hipStreamBeginCapture"):
            m.encode(x[..., :cfg.frame_size].contiguous())


def test_frames_of_2048_samples_are_refused(sim_lib):
    """The frame program divides column numbers by the samples of a frame with 11 bits; a stream of longer frames is refused when it
    starts, however few they are.  One hop less is taken."""
    cfg = replace(tiny_mimi_config(), n_filters=1, dimension=16, tr_d_model=16, tr_num_heads=1, compress=1)
    for ratios, ok in (([8, 8, 4, 4], False), ([8, 4, 31, 1], True)):
        c = replace(cfg, ratios=ratios)
        c = replace(c, sample_rate=c.hop_length * 25)
        assert c.frame_size == (1984 if ok else 2048)
        m = MimiModel(random_mimi_state_dict(c, seed=1, device="cpu"), c, device="cpu", max_batch=1, num_codebooks=2, lib=sim_lib)
        if ok:
            with m.streaming(1):
                assert m.is_streaming
            continue
        with pytest.raises(NotImplementedError, match="index arithmetic"):
            m.streaming_forever(1)


@pytest.mark.gpu
@pytest.mark.parametrize("B,sizes", [(1, (1, 2, 65, 160, 161, 3)), (3, (21, 1, 53, 54)), (32, (2, 1, 5, 6)), (64, (3, 1))])
def test_full_size_calls_equal_frames(B, sizes):
    check_calls_equal_frames(lambda sd, cfg, K, mb: MimiModel(sd, cfg, device="cuda", max_batch=mb, num_codebooks=K), "cuda", MimiConfig(), B, sizes, K=8)


@pytest.mark.gpu
def test_a_mask_set_by_a_graph_is_seen():
    """A captured set_exec_mask leaves no trace on the host when it is replayed: calls of several frames look at the mask itself."""
    cfg, B = tiny_mimi_config(), 3
    sd = random_mimi_state_dict(cfg, seed=5, device="cuda")
    a, b = (MimiModel(sd, cfg, device="cuda", max_batch=B, num_codebooks=4) for _ in range(2))
    fs = cfg.frame_size
    x = (0.3 * torch.randn(B, 1, 12 * fs, generator=torch.Generator().manual_seed(9))).cuda()
    mask = torch.tensor([True, False, True], device="cuda")

    def same(at, rows):
        want = torch.cat([b.encode(x[..., f * fs:(f + 1) * fs].contiguous()) for f in range(at, at + 3)], -1)
        assert torch.equal(a.encode(x[..., at * fs:(at + 3) * fs].contiguous())[rows], want[rows]), at
    with a.streaming(B), b.streaming(B):
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            a.set_exec_mask(mask)                              # (recorded, not run)
        everyone = torch.ones(B, dtype=torch.bool, device="cuda")
        same(0, everyone)
        a.reset_streaming(), b.reset_streaming()
        same(3, everyone)
        for at in (6, 9):
            graph.replay(), b.set_exec_mask(mask)
            same(at, mask)
            for m in (a, b):
                m.set_exec_mask(everyone)
            same(0, everyone)                                  # the stream that stood still goes on where it stood


@pytest.mark.parametrize("heads,ff", [(9, 2056), (33, 2048)])
def test_norms_and_linears_of_many_columns(sim_lib, heads, ff):
    """k_mimi_lin_rows (a feed-forward of some 2048 rows on 114 columns, enough workgroups for it) against k_mimi_lin's frame-by-frame bits: rows
    that fill no whole workgroup, a norm over 9 and over 33 fragments (pieces that are empty, and longer than four)."""
    cfg = replace(tiny_mimi_config(), dimension=16 * heads, tr_d_model=16 * heads, tr_num_heads=heads, tr_dim_feedforward=ff, tr_num_layers=1)
    m = MimiModel(random_mimi_state_dict(cfg, seed=8), cfg, device="cpu", max_batch=1, num_codebooks=2, lib=sim_lib)
    codes = torch.randint(0, cfg.q_bins, (1, 2, 57), generator=torch.Generator().manual_seed(3))
    with m.streaming(1):
        whole = m.decode(codes)
    with m.streaming(1):
        assert torch.equal(whole, torch.cat([m.decode(codes[..., f:f + 1]) for f in range(57)], -1))


@pytest.mark.parametrize("enough,ks,filters,B,frames", [(1, 1, 10, 1, 23), (1, 8, 10, 1, 29), (1, 1, 14, 1, 23), (1, 3, 22, 1, 23), (60, 3, 12, 2, 13)])
def test_convs_of_many_columns(sim_lib, monkeypatch, enough, ks, filters, B, frames):
    """k_conv_cols (one, two and four m-tiles per wave, groups of two and of four quads) against the frame program's bits: column tiles that are cut
    (552 columns, 696, 1104), workgroups with waves past the last one, channels that are no multiple of 32 and m-tiles that are none of a
    wave's, reductions in pieces that are empty, shorter than a group and of an odd length, sums split over 3 and 8 workgroups, two streams."""
    monkeypatch.setenv("MMI_CONV_COLS", str(enough))
    monkeypatch.setenv("MMI_CONV_KSPLIT", str(ks))
    monkeypatch.setenv("MMI_DEBUG_POISON", "1")
    cfg = replace(tiny_mimi_config(), n_filters=filters)
    sd, fs = random_mimi_state_dict(cfg, seed=6, device="cpu"), cfg.frame_size
    m = MimiModel(sd, cfg, device="cpu", max_batch=B, num_codebooks=3, lib=sim_lib)
    x = 0.3 * torch.randn(B, 1, fs * frames, generator=torch.Generator().manual_seed(filters))
    with m.streaming(B):
        codes = m.encode(x)
        pcm = m.decode(codes)
        assert all("k_conv_cols" in {k for _, k in m.launch_list(which)} for which in ("encode_group", "decode_group"))
    with m.streaming(B):
        assert torch.equal(codes, torch.cat([m.encode(x[..., f * fs:(f + 1) * fs].contiguous()) for f in range(frames)], -1))
        assert torch.equal(pcm, torch.cat([m.decode(codes[..., f:f + 1].contiguous()) for f in range(frames)], -1))


@pytest.mark.parametrize("heads,frames,rows", [(60, 57, True), (61, 57, False), (61, 10, False), (64, 65, False)])
def test_widths_whose_columns_fit_the_group_memory(sim_lib, heads, frames, rows):
    """k_mimi_lin_rows keeps the normalised columns in 64 KB of LDS, 1 KB for every 16 channels beside 1 KB of its own: widths of up to 960 take it,
    wider ones k_mimi_lin - two row tiles to a norm (20 columns), two column tiles (114, 130), 32 x 32 tiles (130 columns) - with the frames' bits."""
    cfg = replace(tiny_mimi_config(), dimension=16 * heads, tr_d_model=16 * heads, tr_num_heads=heads, tr_dim_feedforward=2048, tr_num_layers=1, n_filters=1, compress=1)
    m = MimiModel(random_mimi_state_dict(cfg, seed=9), cfg, device="cpu", max_batch=1, num_codebooks=2, lib=sim_lib)
    codes = torch.randint(0, cfg.q_bins, (1, 2, frames), generator=torch.Generator().manual_seed(3))
    with m.streaming(1):
        whole = m.decode(codes)
        kernels = {k for _, k in m.launch_list("decode_group")}
    assert "k_mimi_lin" in kernels and ("k_mimi_lin_rows" in kernels) == rows
    with m.streaming(1):
        assert torch.equal(whole[..., :4 * cfg.frame_size], torch.cat([m.decode(codes[..., f:f + 1]) for f in range(4)], -1))
