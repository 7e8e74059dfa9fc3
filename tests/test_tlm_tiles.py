"""Every block form of the tiled product kernel (k_tlm_gemm_tile) - 64 x 32 in three and four stages, 64 x 64 in stages of one and of two k-steps,
128 x 64, 128 x 128 in three and four stages, 256 x 128, whole and split reductions, gathered and listed expert rows - at row counts just past a
tile and sizes that are no multiples of one: a prompt fed at once must give the logits that the same prompt gives in portions of at most 64
tokens, which take the weight-streaming kernel.  Each case says which forms its launches must have."""
from dataclasses import replace

import pytest
import torch

from tests import tlm_cases as tc
from moshi_amd.config import (DenseGLUConfig, GroupedAttentionConfig, LatentAttentionConfig, MinGRUConfig, MoEConfig, TokenLayerConfig, TokenLMConfig)
from moshi_amd.tlm import TokenLM
from moshi_amd.weights import random_token_lm_state_dict
from oracle.token_lm_oracle import TokenLMOracle


def experts_model(width, ff):
    att = LatentAttentionConfig(heads=4, dim=64, vdim=64, rot_dim=32, q_rank=200, kv_rank=120, scale=0.1)
    moe = MoEConfig(experts=5, top=2, ff=ff)
    return TokenLMConfig("Kesirax", vocab=331, width=width, layers=[TokenLayerConfig(MinGRUConfig(width + 16), moe), TokenLayerConfig(att, moe)])


def dense_model(width, ff):
    att = GroupedAttentionConfig(heads=8, kv_heads=2, dim=64, vdim=64, scale=0.125)
    return TokenLMConfig("Bibapel", vocab=331, width=width, layers=[TokenLayerConfig(att, DenseGLUConfig(ff=ff, limit=7.0))], norms=2, layer_scales=False, tied_head=True)


def from_oracle(got, sd, model, prompt, want):
    """Relative error (2-norm) against the oracle's float64.  At bf16 a layer rounds its normed input, queries, keys, values, the attention's output, the
    feed-forward's input and its hidden row, each by 2^-9 / sqrt(3) (RMS): 3e-3 together, if nothing shrank on the way; below 8e-3 asked."""
    ref = torch.from_numpy(TokenLMOracle({k: v.cpu() for k, v in sd.items()}, model).logits(prompt)[want])
    return float((got.cpu().double() - ref).norm() / ref.norm())


def check_prompt_at_once(device, lib, model, T, dtype, want_forms, monkeypatch, capfd):
    monkeypatch.setenv("MMI_TLM_FORMS", "1")
    sd = random_token_lm_state_dict(model, seed=T, device=device)
    lm = TokenLM(sd, model, dtype=dtype, max_slots=2, max_tokens=4096, max_step_tokens=T, **({} if lib is None else {"device": device, "lib": lib}))
    prompt = torch.randint(0, model.vocab, (T,), generator=torch.Generator().manual_seed(T)).tolist()
    want = sorted({0, 15, 16, 63, 64, T // 2, T - 2, T - 1})
    a = lm.open()
    capfd.readouterr()
    whole = lm.step([(a, prompt, want)])
    assert "k_tlm_gemm_tile" in {k for _, k, _ in lm.launch_list()}
    assert {line[5:line.index(",")] for line in capfd.readouterr().err.splitlines() if line.startswith("tile ")} == want_forms
    b = lm.open()
    parts = torch.cat([lm.step([(b, prompt[i:i + 64], [w - i for w in want if i <= w < i + 64])]) for i in range(0, T, 64)])
    rel = float((whole - parts).double().norm() / parts.double().norm())
    # fp32: sums of up to 6000 products in another order, over a handful of layers (eps sqrt(6000) ~ 5e-6); bf16: an activation on the other
    # side of a rounding boundary here and there (2^-9 each)
    assert rel < (1e-5 if dtype == torch.float32 else 8e-3), rel


# form: features x rows of a block, stages in its ring, k-steps per stage
SMALL32, SMALL16 = {"64x32 stages 4 of 2"}, {"64x64 stages 4 of 2"}


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("model,T,fp32,bf16", [
    (experts_model(208, 144), 65, SMALL32, SMALL16), (experts_model(528, 400), 130, SMALL32, SMALL16),        # (a reduction's last stage half empty)
    (dense_model(2080, 3800), 200, SMALL32, {"64x64 stages 4 of 1", "64x64 stages 4 of 2"}),                  # 524 equal blocks; 264 long beside 132 short
    (experts_model(2080, 3800), 100, {"64x32 stages 3 of 2", "64x32 stages 4 of 2"}, {"64x64 stages 4 of 1", "64x64 stages 4 of 2"}),
    (dense_model(2080, 3800), 460, {"64x32 stages 3 of 2", "64x32 stages 4 of 2"}, {"128x64 stages 4 of 1", "64x64 stages 4 of 2"}),   # 264 long beside 264 short
    (dense_model(1040, 4000), 577, {"64x32 stages 3 of 2", "64x32 stages 4 of 2"}, {"128x64 stages 4 of 1", "64x64 stages 4 of 2"}),
    (dense_model(1040, 1200), 641, {"128x128 stages 4 of 1"}, {"128x128 stages 4 of 1"}),
    (experts_model(1040, 2064), 1025, {"128x128 stages 3 of 1", "128x128 stages 4 of 1"}, {"128x128 stages 3 of 1", "128x128 stages 4 of 1"}),
    (dense_model(1040, 6000), 1157, {"128x128 stages 3 of 1"}, {"256x128 stages 3 of 1", "128x128 stages 4 of 1"}),
], ids=["65", "130", "200", "100", "460", "577", "641", "1025", "1157"])
def test_prompt_at_once_equals_portions(model, T, fp32, bf16, dtype, monkeypatch, capfd):
    check_prompt_at_once("cuda", None, model, T, dtype, fp32 if dtype == torch.float32 else bf16, monkeypatch, capfd)


@pytest.mark.parametrize("model,T,forms", [
    (dense_model(64, 8200), 70, {"64x64 stages 4 of 1", "64x64 stages 4 of 2"}),               # 538 equal blocks of two k-steps; then a few
    (dense_model(2080, 8000), 66, {"64x64 stages 4 of 1", "64x64 stages 4 of 2"}),             # 524 equal blocks of 65 k-steps; then 66 long ones beside 66 short
    (experts_model(80, 4200), 96, {"64x64 stages 4 of 1", "64x64 stages 4 of 2"}),             # listed blocks: more than 512, and fewer
], ids=["dense", "long", "experts"])
def test_prompt_at_once_on_the_simulator(model, T, forms, monkeypatch, capfd):
    """64 x 64 blocks in stages of one and of two k-steps, the forms that no tiny model's launches are large enough for."""
    import os
    import sys
    from pathlib import Path
    from moshi_amd import _capi
    monkeypatch.setenv("MMI_NO_GRAPH", "1")
    sys.path.insert(0, str(Path(__file__).resolve().parent / "hipsim"))
    import build_sim
    lib = _capi.load_tlm(os.environ.get("MMI_TLM_SIM_LIB") or build_sim.build_tlm())
    check_prompt_at_once("cpu", lib, model, T, torch.bfloat16, forms, monkeypatch, capfd)


def check_wide_heights(device, lib, model, T, heights, monkeypatch, capfd):
    """k_tlm_gemm_wide forms every sum as k_tlm_gemm_tile does: with the same splits a prompt's logits have the same bits, however high its blocks are.
    They are the oracle's."""
    monkeypatch.setenv("MMI_TLM_FORMS", "1")
    sd = random_token_lm_state_dict(model, seed=T, device=device)
    prompt = torch.randint(0, model.vocab, (T,), generator=torch.Generator().manual_seed(T)).tolist()
    want = sorted({0, 15, 16, 31, 32, 63, 64, T // 2, T - 2, T - 1})
    base = None
    for height in [None, *heights]:
        monkeypatch.setenv("MMI_TLM_WIDE", str(height)) if height else monkeypatch.delenv("MMI_TLM_WIDE", raising=False)
        lm = TokenLM(sd, model, dtype=torch.bfloat16, max_slots=1, max_tokens=4096, max_step_tokens=T, **({} if lib is None else {"device": device, "lib": lib}))
        capfd.readouterr()
        got = lm.step([(lm.open(), prompt, want)])
        forms = {line.split(",")[0] for line in capfd.readouterr().err.splitlines() if line.startswith("wide ")}
        assert forms == ({f"wide 256x{height}"} if height else set())
        base = got if base is None else base
        assert torch.equal(got, base), height
    assert from_oracle(base, sd, model, prompt, want) < 8e-3


@pytest.mark.gpu
@pytest.mark.parametrize("model,T,heights", [
    (dense_model(1040, 1200), 641, [32, 64, 96, 128, 160, 192, 224, 256]),      # 33 k-steps (one more than whole pairs), 65 and 163 n-tiles, a last block of one row
    (dense_model(1024, 2048), 97, [32, 96, 256]),                               # 32 and 64 k-steps, three rows in the last fragment, blocks higher than the rows
    (dense_model(48, 80), 300, [96, 160, 256]),                                 # two k-steps: fewer than the ring has places
], ids=["odd", "even", "short"])
def test_wide_blocks_have_the_bits_of_the_narrow_ones(model, T, heights, monkeypatch, capfd):
    check_wide_heights("cuda", None, model, T, heights, monkeypatch, capfd)


@pytest.mark.parametrize("model,T,heights", [(dense_model(144, 200), 270, [32, 64, 96, 128, 160, 192, 224, 256]), (dense_model(48, 80), 97, [64, 128, 256])], ids=["odd", "short"])
def test_wide_blocks_on_the_simulator(model, T, heights, monkeypatch, capfd):
    import os
    import sys
    from pathlib import Path
    from moshi_amd import _capi
    monkeypatch.setenv("MMI_NO_GRAPH", "1")
    sys.path.insert(0, str(Path(__file__).resolve().parent / "hipsim"))
    import build_sim
    lib = _capi.load_tlm(os.environ.get("MMI_TLM_SIM_LIB") or build_sim.build_tlm())
    check_wide_heights("cpu", lib, model, T, heights, monkeypatch, capfd)


@pytest.mark.gpu
@pytest.mark.parametrize("model,T,form", [(dense_model(4160, 12000), 300, "wide 256x160"), (dense_model(5200, 14000), 97, "wide 256x"), (dense_model(3088, 9000), 641, "wide 256x")],
                         ids=["4160", "5200", "3088"])
def test_large_prompts_take_wide_blocks(model, T, form, monkeypatch, capfd):
    """Chosen by the sizes alone, with splits of its own: the logits of a prompt fed at once are the oracle's, and those of the same prompt in
    portions of 64."""
    monkeypatch.setenv("MMI_TLM_FORMS", "1")
    sd = random_token_lm_state_dict(model, seed=T, device="cuda")
    lm = TokenLM(sd, model, dtype=torch.bfloat16, max_slots=2, max_tokens=4096, max_step_tokens=T)
    prompt = torch.randint(0, model.vocab, (T,), generator=torch.Generator().manual_seed(T)).tolist()
    want = sorted({w for w in (0, 63, 64, T // 2, 159, 160, T - 1) if w < T})
    capfd.readouterr()
    whole = lm.step([(lm.open(), prompt, want)])
    assert any(line.startswith(form) for line in capfd.readouterr().err.splitlines())
    b = lm.open()
    parts = torch.cat([lm.step([(b, prompt[i:i + 64], [w - i for w in want if i <= w < i + 64])]) for i in range(0, T, 64)])
    assert float((whole - parts).double().norm() / parts.double().norm()) < 8e-3      # (as in check_prompt_at_once)
    assert from_oracle(whole, sd, model, prompt, want) < 8e-3


@pytest.mark.parametrize("rise", [0.0, 0.3, 3.7, 7.9, 8.1, 40.0])
def test_the_largest_weight_is_exactly_one(tmp_path, rise):
    """bf16 attention rounds a weight relative to itself, so it must be formed against the maximum so far: the largest one is then exact,
    however little the maximum has moved from one block of keys to the next (column c moves by c / 16 of `rise`)."""
    import ctypes
    import subprocess
    import sys
    from pathlib import Path
    here = Path(__file__).resolve().parent / "hipsim"
    sys.path.insert(0, str(here))
    import build_sim
    so = tmp_path / "softmax_selftest.so"
    subprocess.check_call([build_sim._cxx(), "-O1", "-w", "-std=c++17", "-fPIC", "-shared", "-pthread", "-ffp-contract=off", f"-I{here}", f"-I{build_sim.CSRC}",
                           str(here / "softmax_selftest.cpp"), str(here / "hipsim.cpp"), "-o", str(so)])
    lib, blocks = ctypes.CDLL(str(so)), 3
    scores = torch.rand(blocks, 32, 16, generator=torch.Generator().manual_seed(3)) - 1.0
    for b in range(1, blocks):
        scores[b, 5 * b] = b * rise * torch.arange(16) / 16
    p, m, l = torch.empty_like(scores), torch.empty(blocks, 16), torch.empty(16)
    lib.softmax_selftest_run(*(ctypes.c_void_p(t.data_ptr()) if torch.is_tensor(t) else t for t in (scores, blocks, p, m, l)))
    top = scores.amax(1).cummax(0).values
    assert torch.equal(m, top)
    want = torch.exp2(scores.double() - top[:, None].double())
    assert torch.equal(p[scores == top[:, None]], torch.ones(int((scores == top[:, None]).sum())))
    assert ((p - want).abs() <= want * 2.0 ** -8 + 2.0 ** -126).all()        # one rounding to bf16, 2^-9, and a few of fp32; no subnormal numbers
    assert torch.allclose(l.double(), (want * torch.exp2(top - top[-1])[:, None].double()).sum((0, 1)), rtol=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("times", [8, -1, 0])
@pytest.mark.parametrize("name", ["latent_36", "latent_128", "latent_200", "gqa_24", "gqa_128"])
def test_attention_of_steep_turned_and_flat_scores(name, times):
    """Prompts' attention where maxima move far from block to block (steep), where it is the other end of the scores that counts (a
    negative scale) and where nothing moves (scale 0); the window's and the sequence's ends fall inside blocks of 32 keys."""
    cfg = {**tc.WIDE_PROMPTS, **tc.WIDE_PROMPTS_2}[name]
    mixer = cfg.layers[0].mixer
    cfg = replace(cfg, layers=[replace(cfg.layers[0], mixer=replace(mixer, scale=mixer.scale * times))])
    lm, orc = tc.make(cfg, "cuda", None, max_tokens=1024)
    toks = tc.tokens_of(cfg, 731, seed=7)
    slot = lm.open()
    pick = [0, 1, 31, 32, 33, 63, 64, 89, 90, 91, 300, 301, 702, 703, 704, 719]
    got = lm.step([(slot, toks[:720], pick)])
    want = orc.logits(toks)
    # a score is off by some eps |score| and its weight by as much relatively: the steep ones by 8 times what the plain ones are
    assert tc.rel(got.cpu().numpy(), want[pick]) < tc.TOL[torch.float32] * max(1, times)
    assert tc.rel(tc.run_cut(lm, toks[720:], [1], slot), want[720:]) < tc.TOL[torch.float32] * max(1, times)
