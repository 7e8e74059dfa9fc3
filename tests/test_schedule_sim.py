"""Race check on the kernel simulator: a kernel's result may not depend on the order in which the waves of a workgroup (and, between
two wave-level synchronisation points, the lanes of a wave) happen to run.

The simulator's default schedule - wave 0 first, lane 0 first - is only ONE of the orders the hardware may take between two barriers;
a kernel with a missing `__syncthreads()` (wave 1 reading what wave 0 has just written to LDS) passes under it by luck and fails on
the GPU now and then.  `hipsim_set_schedule` (tests/hipsim/hipsim.cpp) walks waves and lanes BACKWARDS, or in a fresh random
permutation at every scheduling pass; the engine's outputs - tokens, codes, logits, hidden states, PCM - must come out bit for bit
as under the default schedule.  (A nondeterministic launch was once found by comparing runs with each other, not with the
checker.  That one was an instruction-level hazard no simulator sees; this test covers the class a simulator CAN see.)

The whole simulator suite was also run once under `HIPSIM_SCHED=reverse` and `HIPSIM_SCHED=random:7`
(profiles/r05_logs/sim_suite_schedule_{reverse,random7}.log)."""
from contextlib import contextmanager
from pathlib import Path

import numpy as np
import pytest
import torch

from moshi_amd import MimiModel, tiny_mimi_config
from moshi_amd.config import tiny_lm_config
from tests import duplex_cases, lm_cases, mimi_cases

HIPSIM = Path(__file__).resolve().parent / "hipsim"
FORWARD, REVERSE, RANDOM = 0, 1, 2
SCHEDULES = [(REVERSE, 1), (RANDOM, 7), (RANDOM, 2024)]


@contextmanager
def schedule(lib, mode, seed=1):
    lib.cdll.hipsim_set_schedule(int(mode), int(seed))
    try:
        yield
    finally:
        lib.cdll.hipsim_set_schedule(FORWARD, 1)


def test_schedule_switch_is_live(sim_lib):
    with schedule(sim_lib, RANDOM, 5):
        assert sim_lib.cdll.hipsim_get_schedule() == RANDOM
    assert sim_lib.cdll.hipsim_get_schedule() == FORWARD


def test_perturbed_schedules_expose_a_missing_barrier(sim_lib, tmp_path):
    """Negative control: tests/hipsim/race_selftest.cpp is one kernel with and without the barrier between an LDS write and the read
    of another wave's slot.  The racy form must give different bits under the perturbed schedules, the correct form the same."""
    import ctypes
    import subprocess
    import sys
    sys.path.insert(0, str(HIPSIM))
    import build_sim
    so = tmp_path / "race_selftest.so"
    subprocess.check_call([build_sim._cxx(), "-O1", "-w", "-std=c++17", "-fPIC", "-shared", "-pthread", f"-I{HIPSIM}",
                           str(HIPSIM / "race_selftest.cpp"), str(HIPSIM / "hipsim.cpp"), "-o", str(so)])
    lib = ctypes.CDLL(str(so))

    def run(racy, mode, seed=1):
        lib.hipsim_set_schedule(mode, seed)
        out = np.zeros(128, np.float32)
        lib.race_selftest_run(out.ctypes.data_as(ctypes.c_void_p), racy)
        return out
    good = run(0, FORWARD)
    assert np.array_equal(good, np.roll(np.arange(1, 129, dtype=np.float32), 64))
    assert all(np.array_equal(run(0, m, sd), good) for m, sd in SCHEDULES + [(RANDOM, k) for k in range(8)])
    racy = run(1, FORWARD)
    assert not np.array_equal(run(1, REVERSE), racy), "the reversed schedule does not expose the missing barrier"
    assert any(not np.array_equal(run(1, RANDOM, k), racy) for k in range(8)), "no random schedule exposes the missing barrier"


@pytest.mark.parametrize("B,quantize,env", [
    (3, False, {}),                                                    # 16-row tiles, the one-session style kernels
    (18, False, {"MMI_GEMM_LDS": "2", "MMI_GEMM_KSPLIT": "2"}),        # 32-row tile, LDS-resident GEMM with split-K
    (34, True, {}),                                                    # two batch tiles, int8 x int8: k_gemm_xp<32, 2> + k_gemm_q8 per tile
    (5, "fp8", {"MMI_ATTN_NS": "3"}),                                  # fp8 MFMA; the ring split over workgroups + merge
    (18, False, {"MMI_GEMM_ONCE": "a", "MMI_GEMM_LDS": "0"}),          # k_gemm_xp_once on every GEMM whose slices fit
    (18, False, {"MMI_GEMM_REG": "5"}),                                # k_gemm_xreg: register-resident activations, sums of the waves per tile
    (34, True, {"MMI_GEMM_REG": "8"}),                                 # ... of two batch tiles at int8
    (1, False, {"MMI_GEMM_REG": "3"}),                                 # k_gemm_xreg16 with the norm inside: two scratches in turn, one meeting per tile
    (16, False, {"MMI_GEMM_REG": "3"}),                                # ... of a full tile of sessions
    (5, False, {"MMI_GEMM_RING": "2", "MMI_GEMM_OSPLIT": "0", "MMI_GEMM_KSPLIT": "1"}),                                 # k_gemm_xring16
    (1, False, {"MMI_GEMM_RING": "2", "MMI_GEMM_OSPLIT": "0", "MMI_ATTN_NS": "3", "MMI_ATTN_SOLO": "0"}),               # ... that merges the attention's partials
    (9, "guided-cross", {}),                                           # guidance twins + cross-attention block + k_cfg_mix
])
def test_lm_step_is_independent_of_the_wave_schedule(sim_lib, monkeypatch, B, quantize, env):
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    if quantize == "guided-cross":
        from dataclasses import replace

        def perturb_gc(r):
            mode, seed = SCHEDULES[r]
            sim_lib.cdll.hipsim_set_schedule(mode, seed)
        try:
            lm_cases.reproducible_between_streams("cpu", sim_lib, replace(tiny_lm_config(), cross_attention=True), B=B, steps=2,
                                                  repeats=len(SCHEDULES), seed=31 + B, before_repeat=perturb_gc, guided_cross=(5, 2.0))
        finally:
            sim_lib.cdll.hipsim_set_schedule(FORWARD, 1)
        return

    def perturb(r):
        mode, seed = SCHEDULES[r]
        sim_lib.cdll.hipsim_set_schedule(mode, seed)
    try:
        lm_cases.reproducible_between_streams("cpu", sim_lib, tiny_lm_config(), B=B, quantize=quantize, steps=2,
                                              repeats=len(SCHEDULES), seed=31 + B, before_repeat=perturb)
    finally:
        sim_lib.cdll.hipsim_set_schedule(FORWARD, 1)


def test_mimi_codec_is_independent_of_the_wave_schedule(sim_lib):
    """The reference's golden schedule (exec masks, a partial reset) through encode and decode: codes and PCM bit-identical."""
    def make(sd, cfg, K, max_batch=8):
        return MimiModel(sd, cfg, device="cpu", max_batch=max_batch, num_codebooks=K, lib=sim_lib)
    _, codes0, pcm0 = mimi_cases.run_tiny_schedule(make, "cpu")
    for mode, seed in SCHEDULES:
        with schedule(sim_lib, mode, seed):
            _, codes, pcm = mimi_cases.run_tiny_schedule(make, "cpu")
        assert np.array_equal(codes, codes0), f"schedule {(mode, seed)}: codes differ"
        assert np.array_equal(pcm.view(np.uint32), pcm0.view(np.uint32)), f"schedule {(mode, seed)}: PCM differs"


def test_mimi_wide_batch_kernels_are_independent_of_the_wave_schedule(sim_lib, monkeypatch):
    """B = 6 puts the audio-rate layers on k_conv_wide and the rest on k_pack_b_f32 + k_gemm_f32 (split-K over waves and workgroups),
    the first residual block on k_resblock."""
    from moshi_amd.weights import random_mimi_state_dict
    monkeypatch.setenv("MMI_CONV_MTB", "2")
    monkeypatch.setenv("MMI_CONV_W", "4")
    monkeypatch.setenv("MMI_CONV_KSPLIT", "3")
    monkeypatch.setenv("MMI_MIMI_RES_FUSION_MIN", "1")
    cfg = tiny_mimi_config()
    sd = random_mimi_state_dict(cfg, seed=12)
    rng = np.random.default_rng(12)
    x = torch.from_numpy((0.2 * rng.standard_normal((6, 1, 3 * cfg.frame_size))).astype(np.float32))

    def run():
        m = MimiModel(sd, cfg, device="cpu", max_batch=6, num_codebooks=5, lib=sim_lib)
        with m.streaming(6):
            codes = m.encode(x)
            pcm = m.decode(codes)
        return codes.numpy().copy(), pcm.numpy().copy()
    codes0, pcm0 = run()
    for mode, seed in SCHEDULES[:2]:
        with schedule(sim_lib, mode, seed):
            codes, pcm = run()
        assert np.array_equal(codes, codes0), f"schedule {(mode, seed)}: codes differ"
        assert np.array_equal(pcm.view(np.uint32), pcm0.view(np.uint32)), f"schedule {(mode, seed)}: PCM differs"


def test_duplex_pipeline_is_independent_of_the_wave_schedule(sim_lib):
    with schedule(sim_lib, RANDOM, 11):
        assert duplex_cases.check_pipeline_is_bit_identical("cpu", sim_lib, B=3, steps=6, use_sampling=True, join_every=3) >= 4


def test_full_size_codec_at_the_c2_batch_is_independent_of_the_wave_schedule(sim_lib):
    """The released codec's shapes, 8 streams: every kernel at its production tiling (the wide-batch convs, the
    split-K GEMMs of the 12.5 / 25 Hz layers, both transformers, the RVQ).  ~1 minute.  (The LM's benchmark kernels at the 7B widths
    take minutes per run: tests/tools/sim_full_width_schedules.py, profiles/r05_logs/sim_full_width_schedules.log.)"""
    from moshi_amd import MimiConfig
    from moshi_amd.weights import random_mimi_state_dict
    cfg = MimiConfig()
    sd = random_mimi_state_dict(cfg, seed=3)
    rng = np.random.default_rng(3)
    B, F = 8, 2
    x = torch.from_numpy((0.1 * rng.standard_normal((B, 1, F * cfg.frame_size))).astype(np.float32))

    def run():
        m = MimiModel(sd, cfg, device="cpu", max_batch=B, num_codebooks=8, lib=sim_lib)
        with m.streaming(B):
            codes = m.encode(x)
            pcm = m.decode(codes)
        return codes.numpy().copy(), pcm.numpy().copy()
    codes0, pcm0 = run()
    for mode, seed in SCHEDULES[:2]:
        with schedule(sim_lib, mode, seed):
            codes, pcm = run()
        assert np.array_equal(codes, codes0), f"schedule {(mode, seed)}: codes differ"
        assert np.array_equal(pcm.view(np.uint32), pcm0.view(np.uint32)), f"schedule {(mode, seed)}: PCM differs"
