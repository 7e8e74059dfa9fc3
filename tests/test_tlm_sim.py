"""Token language models on the kernel simulator: the cases of tests/tlm_cases.py, and bit-identical results under perturbed schedules."""
import os
import sys

import numpy as np
import pytest

from tests import tlm_cases as tc
from tests.conftest import ROOT

DEV = "cpu"


@pytest.fixture(scope="session")
def tlm_lib():
    os.environ["MMI_NO_GRAPH"] = "1"
    sys.path.insert(0, str(ROOT / "tests" / "hipsim"))
    import build_sim
    from moshi_amd import _capi
    return _capi.load_tlm(os.environ.get("MMI_TLM_SIM_LIB") or build_sim.build_tlm())


@pytest.mark.parametrize("name", sorted(tc.MECHANISMS))
def test_mechanism_fp32(tlm_lib, name):
    tc.check_mechanism(name, DEV, tlm_lib)


@pytest.mark.parametrize("name", ["mingru_experts", "attention_experts", "wide_latent", "repeated", "mixed", "grouped_attention", "delta", "lightning", "glu",
                                  "projected_passes", "bibapel"])
def test_mechanism_bf16(tlm_lib, name):
    tc.check_mechanism(name, DEV, tlm_lib, tc.BF16)


@pytest.mark.parametrize("dim,vdim,n", tc.CHUNK_EDGES)
def test_chunk_edges(tlm_lib, dim, vdim, n):
    tc.check_chunk_edges(DEV, tlm_lib, dim, vdim, n)


@pytest.mark.parametrize("lightning", [False, True], ids=["delta", "lightning"])
@pytest.mark.parametrize("dim,vdim", tc.BESIDE_CHUNKS)
def test_tokens_beside_chunks(tlm_lib, dim, vdim, lightning):
    tc.check_tokens_beside_chunks(DEV, tlm_lib, dim, vdim, lightning=lightning)


@pytest.mark.parametrize("far", [False, True])
def test_activation_branches(tlm_lib, far):
    tc.check_activation_branches(DEV, tlm_lib, far)


def test_sigmoid(tmp_path):
    """Every exponent on both sides, the clamps' and the underflow's surroundings, subnormal results, infinities and NaN.  Bound, in units of 2^-24 of
    the result: 0.7 from the argument of 2^f, |f| <= 1/2, rounded twice; 2 from 2^f, good to one in its last place; 1 from the sum; 2 from the
    reciprocal behind its step and its rounding; and half of the smallest subnormal number."""
    import ctypes
    import subprocess
    import sys
    from pathlib import Path
    import torch
    here = Path(__file__).resolve().parent / "hipsim"
    sys.path.insert(0, str(here))
    import build_sim
    so = tmp_path / "sigmoid_selftest.so"
    subprocess.check_call([build_sim._cxx(), "-O1", "-w", "-std=c++17", "-fPIC", "-shared", "-pthread", "-ffp-contract=off", f"-I{here}", f"-I{build_sim.CSRC}",
                           str(here / "sigmoid_selftest.cpp"), str(here / "hipsim.cpp"), "-o", str(so)])
    g = torch.Generator().manual_seed(1)
    size = torch.exp2(torch.linspace(-149, 127.99, 40000)) * (1 + torch.rand(40000, generator=g) / 4)
    edges = torch.tensor([0.0, 0.34657359, 87.33655, 88.0, 88.37626, 88.72284, 103.2789, 103.97208, 104.0, 104.00001, 105.0, 3.4e38, float("inf")])
    x = torch.cat([size, edges, torch.rand(40000, generator=g) * 110])
    x = torch.cat([x, -x])
    y, nan = torch.empty_like(x), torch.tensor([float("nan")])
    lib = ctypes.CDLL(str(so))
    lib.sigmoid_selftest_run(ctypes.c_void_p(x.data_ptr()), x.numel(), ctypes.c_void_p(y.data_ptr()))
    lib.sigmoid_selftest_run(ctypes.c_void_p(nan.data_ptr()), 1, ctypes.c_void_p(nan.data_ptr()))
    want = torch.sigmoid(x.double())
    assert ((y.double() - want).abs() <= 6 * 2.0 ** -24 * want + 2.0 ** -150).all()
    assert y[x == float("inf")].eq(1).all() and y[x == -float("inf")].eq(0).all() and nan.isnan().all()


def test_portions_of_a_prompt(tlm_lib):
    tc.check_portions(DEV, tlm_lib)


def test_portions_of_a_prompt_bf16(tlm_lib):
    tc.check_portions(DEV, tlm_lib, tc.BF16, n=100, cut_sets=((2,), (65, 1)))


def test_prompt_then_decode(tlm_lib):
    tc.check_prompt_then_decode(DEV, tlm_lib)


def test_unequal_requests_in_one_batch(tlm_lib):
    tc.check_unequal_batch(DEV, tlm_lib)


def test_batched_decode(tlm_lib):
    tc.check_batched_decode(DEV, tlm_lib, steps=4)


def test_pages_and_slots_are_used_again(tlm_lib):
    tc.check_reuse(DEV, tlm_lib)


def test_decoding_longer_than_the_pool(tlm_lib):
    tc.check_long_decode(DEV, tlm_lib)


def test_long_prompt(tlm_lib):
    tc.check_long_prompt(DEV, tlm_lib)


@pytest.mark.parametrize("window", [70, 64, 0])
def test_single_keys(tlm_lib, window):
    tc.check_single_keys(DEV, tlm_lib, window)


def test_state_reaches_far_back(tlm_lib):
    tc.check_far_state(DEV, tlm_lib)


def test_first_tokens(tlm_lib):
    tc.check_first_tokens(DEV, tlm_lib)


def test_greedy_generation_through_the_scheduler(tlm_lib):
    tc.check_generation(DEV, tlm_lib)


def test_sampling(tlm_lib):
    tc.check_sampling(DEV, tlm_lib)


def test_limits_and_errors(tlm_lib):
    tc.check_limits(DEV, tlm_lib)


def test_trace_replay(tlm_lib, tmp_path):
    tc.check_replay(DEV, tlm_lib, tmp_path)


# ---- the mixers with matrix states, grouped attention, and the network that has them all -------------------------------------------
def test_portions_of_a_prompt_bibapel(tlm_lib):
    tc.check_portions(DEV, tlm_lib, n=100, cut_sets=((2,), (3, 2, 61, 7), (65, 1), (5,)), name="bibapel")


def test_prompt_then_decode_bibapel(tlm_lib):
    tc.check_prompt_then_decode(DEV, tlm_lib, n=90, tail=20, name="bibapel")


def test_unequal_requests_in_one_batch_bibapel(tlm_lib):
    tc.check_unequal_batch(DEV, tlm_lib, name="bibapel")


def test_long_prompt_beside_decoding(tlm_lib):
    tc.check_long_prompt_beside_decoding(DEV, tlm_lib, name="all")


def test_batched_decode_bibapel(tlm_lib):
    tc.check_batched_decode(DEV, tlm_lib, steps=4, name="bibapel")


def test_pages_and_slots_are_used_again_bibapel(tlm_lib):
    tc.check_reuse(DEV, tlm_lib, name="bibapel")


def test_decoding_longer_than_the_pool_with_kept_pages(tlm_lib):
    tc.check_long_decode(DEV, tlm_lib, name="two_kept_windows", n=400, held=4)


@pytest.mark.parametrize("window,keep", [(70, 7), (64, 1), (33, 64), (0, 0)])
def test_single_kept_keys(tlm_lib, window, keep):
    tc.check_single_kept_keys(DEV, tlm_lib, window, keep, queries=(128, 103) if window else (128,))


@pytest.mark.parametrize("case", ["sink", "matrix_state_far", "decay_extremes", "glu_limits", "previous_token", "last_position"])
def test_single_mechanisms(tlm_lib, case):
    getattr(tc, f"check_{case}")(DEV, tlm_lib)


def test_first_tokens_bibapel(tlm_lib):
    tc.check_first_tokens(DEV, tlm_lib, name="bibapel")


def test_greedy_generation_through_the_scheduler_bibapel(tlm_lib):
    tc.check_generation(DEV, tlm_lib, name="bibapel")


@pytest.mark.parametrize("name", ["mixed", "bibapel"])
def test_perturbed_schedules_give_the_same_bits(tlm_lib, name):
    """Waves and lanes of a workgroup in other orders (a missing barrier would show); the order of a routed expert's pairs comes from
    atomics and must not matter either."""
    cfg = tc.MECHANISMS[name]
    toks = tc.tokens_of(cfg, 80)

    def run(mode, seed):
        tlm_lib.cdll.hipsim_set_schedule(mode, seed)
        try:
            return [tc.run_cut(tc.make(cfg, DEV, tlm_lib, dt)[0], toks, [70, 1, 9]) for dt in (tc.F32, tc.BF16)]
        finally:
            tlm_lib.cdll.hipsim_set_schedule(0, 1)
    want = run(0, 1)
    for mode, seed in ((1, 1), (2, 7)):
        for a, b in zip(run(mode, seed), want):
            assert np.array_equal(a, b), (mode, seed)
