"""Steps of one sequence as one launch (token.hip) against the same steps in launches; either way is compared with the oracle's decode chain
elsewhere (test_gpu_inference.py).  The largest and smallest widths that the one launch takes, shares of rows that do not come out even, columns
behind whole steps of 512, contexts up to and over its last key, and what it leaves to the launches."""
import sys

import numpy as np
import pytest

from llm_metal_amd.configs import GEMMA3, QWEN3, SFTConfig
from llm_metal_amd.sft import InferenceState, SFTState
from llm_metal_amd.synth import make_model

pytestmark = pytest.mark.gpu

SHAPES = {
    # few workgroups (a share of D / 4), columns behind the last whole step
    "gemma_320": SFTConfig("t", GEMMA3, NL=3, D=320, Hq=4, Hkv=1, hd=256, IS=448, V=516, tied=True),
    # the widest that threads hold five and seven entries of
    "gemma_1280_7168": SFTConfig("t", GEMMA3, NL=2, D=1280, Hq=4, Hkv=2, hd=256, IS=7168, V=1000, tied=True),
    # a step of 64 columns behind two whole ones, heads of 128
    "gemma_1088_hd128": SFTConfig("t", GEMMA3, NL=2, D=1088, Hq=6, Hkv=3, hd=128, IS=2880, V=2052, tied=True),
    "qwen_1152": SFTConfig("t", QWEN3, NL=2, D=1152, Hq=4, Hkv=1, hd=256, IS=6912, V=4100),
    # the widest of all, vocabulary in several parts per workgroup
    "qwen_2560_10240": SFTConfig("t", QWEN3, NL=2, D=2560, Hq=32, Hkv=8, hd=128, IS=10240, V=45004),
    "qwen_1344": SFTConfig("t", QWEN3, NL=4, D=1344, Hq=10, Hkv=2, hd=128, IS=4160, V=772),
}


def say(*a):
    print(*a, flush=True, file=sys.stderr)


def one_launch(inf):
    return inf.L.hip_inference_steps_in_one_launch(inf.h)


@pytest.mark.parametrize("fmt", ["f16", "q8_0"])
@pytest.mark.parametrize("shape", list(SHAPES))
def test_a_step_as_one_launch_is_the_step_in_launches(shape, fmt):
    say("one launch", shape, fmt)
    c = SHAPES[shape].with_(weight_format=fmt)
    model = make_model(c, seed=41, gamma_jitter=0.1)
    toks = [int(t) for t in np.random.default_rng(42).integers(0, c.V, 262)]
    with InferenceState(c, model, max_seq=262, use_fp16=fmt == "f16") as inf:
        inf.L.hip_gemm_profile_enable(1)                   # a profile counts launches
        want = np.stack([inf.forward_token(t) for t in toks])
        inf.L.hip_gemm_profile_enable(0)
        assert one_launch(inf) == 0
        inf.reset()
        got = np.stack([inf.forward_token(t) for t in toks])
        assert one_launch(inf) == 256                      # the last contexts are longer than it takes
        # both sum the same fp32 products in another order: 2^-24 per operation, some 200 roundings in a row between embedding and logits
        err = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
        assert err.max() < 200 * 2.0 ** -24, err.max()
        inf.reset()
        best = [inf.forward_token_argmax(t) for t in toks]
        assert one_launch(inf) == 512
        srt = np.sort(want, axis=1)
        clear = srt[:, -1] - srt[:, -2] > 1e-4 * np.abs(srt[:, -1])
        assert clear.mean() > 0.9 and (np.asarray(best)[clear] == want.argmax(1)[clear]).all()
        # the argmax is that of what the call beside it hands out
        inf.reset()
        assert best[0] == int(got[0].argmax()) == inf.forward_token_argmax(toks[0])


def test_a_wait_that_runs_out_takes_the_step_again_in_launches():
    c = SHAPES["gemma_320"].with_(weight_format="f16")
    model = make_model(c, seed=43, gamma_jitter=0.1)
    toks = [int(t) for t in np.random.default_rng(44).integers(0, c.V, 12)]
    with InferenceState(c, model, max_seq=16, use_fp16=True) as inf:
        inf.L.hip_gemm_profile_enable(1)
        want = np.stack([inf.forward_token(t) for t in toks])
        inf.L.hip_gemm_profile_enable(0)
        inf.reset()
        got = [np.array(inf.forward_token(t)) for t in toks[:5]]
        inf.L.hip_inference_step_wait(inf.h, 0)            # every wait is over when it begins; the kernel runs to its end
        got += [np.array(inf.forward_token(t)) for t in toks[5:]]
        assert one_launch(inf) == 5
        err = np.linalg.norm(np.stack(got) - want, axis=1) / np.linalg.norm(want, axis=1)
        assert err.max() < 200 * 2.0 ** -24, err.max()
        best = inf.generate(toks[:3], 6)
        assert one_launch(inf) == 5 and len(best) >= 1


def test_steps_are_one_launch_again_some_steps_after_a_wait_that_ran_out():
    c = SHAPES["gemma_320"].with_(weight_format="f16")
    model = make_model(c, seed=48, gamma_jitter=0.1)
    with InferenceState(c, model, max_seq=256, use_fp16=True) as inf:
        L, h, tok = inf.L, inf.h, lambda n: [inf.forward_token(t % c.V) for t in range(n)]
        tok(3)
        for rest in (64, 128):                             # twice as many after the second one
            n = one_launch(inf)
            L.hip_inference_step_wait(h, 0)
            tok(1)
            L.hip_inference_step_wait(h, 100000000)
            tok(rest)
            assert one_launch(inf) == n
            tok(2)
            assert one_launch(inf) == n + 2
        # what the steps hand out behind a failed one, and behind the pause, is what they hand out without
        got = inf.forward_token(5)
        at = inf.position() - 1
        inf.reset()
        L.hip_gemm_profile_enable(1)
        history = [t for n in (3, 1, 64, 2, 1, 128, 2) for t in range(n)]
        assert len(history) == at
        for t in history:
            inf.forward_token(t % c.V)
        want = inf.forward_token(5)
        L.hip_gemm_profile_enable(0)
        assert np.linalg.norm(got - want) < 200 * 2.0 ** -24 * np.linalg.norm(want)


# pairs of rows of a head that 80 workgroups share, 200 rows each, 80 at a time: neighbours of a unit, another wave's, another part of the workgroup's,
# another workgroup's, the first and the last
@pytest.mark.parametrize("fmt", ["f16", "q8_0"])
@pytest.mark.parametrize("rows", [(8000, 8001), (8003, 8075), (8003, 8150), (8199, 8200), (3, 12007), (0, 15999)], ids=str)
def test_the_first_of_equal_maxima(rows, fmt):
    c = SHAPES["gemma_320"].with_(weight_format=fmt, V=16000, NL=2)
    model = make_model(c, seed=51, gamma_jitter=0.1)
    toks = [5, 6, 7]                                       # (the head is the embedding: rows that no token reads are changed)
    def steps():
        with InferenceState(c, model, max_seq=8, use_fp16=fmt == "f16") as inf:
            logits = [inf.forward_token(t) for t in toks]
            inf.reset()
            best = [inf.forward_token_argmax(t) for t in toks]
            assert one_launch(inf) == 2 * len(toks)
            return logits, best
    logits, _ = steps()
    emb = model["token_emb"]
    at = 20 + int(logits[2][20:].argmax())
    emb[list(rows)] = 4 * emb[at]
    logits, best = steps()
    assert logits[2][rows[0]] == logits[2][rows[1]] == logits[2].max()       # (one step of columns: a row's sum does not depend on its place)
    assert best == [int(l.argmax()) for l in logits] and best[2] == rows[0]


def test_values_that_are_not_finite():
    """Against the steps in launches: a token whose embedding is infinite, one whose embedding overflows on the way, and rows of the head that
    are not finite.  An argmax passes over logits that are no number, and is zero where all are."""
    c = SHAPES["qwen_1344"].with_(weight_format="f16")
    model = make_model(c, seed=52, gamma_jitter=0.1)
    model["token_emb"][9] = np.inf
    model["token_emb"][10] = 1e30
    model["lm_head"][7, 3], model["lm_head"][600, 5], model["lm_head"][601] = np.inf, -np.inf, np.nan
    def steps(inf, toks):
        inf.reset()
        logits = np.stack([inf.forward_token(t) for t in toks])
        inf.reset()
        return logits, [inf.forward_token_argmax(t) for t in toks]
    for toks in ([1, 2, 3, 4], [1, 2, 9, 3, 4], [9, 1], [1, 10, 2] + list(range(11, 80))):
        with InferenceState(c, model, max_seq=80, use_fp16=True) as inf:
            got, best = steps(inf, toks)
            assert one_launch(inf) == 2 * len(toks)
            inf.L.hip_gemm_profile_enable(1)
            want, want_best = steps(inf, toks)
            inf.L.hip_gemm_profile_enable(0)
        assert best == want_best, toks
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got) * np.sign(got), np.isinf(want) * np.sign(want), equal_nan=True), toks
        ok = np.isfinite(want)
        assert np.linalg.norm(got[ok] - want[ok]) <= 200 * 2.0 ** -24 * np.linalg.norm(want[ok])
        if 9 in toks:
            assert np.isnan(got[toks.index(9):]).all() and set(best[toks.index(9):]) == {0}


def test_tags_begin_anew_before_32_bits_end():
    """A step's tags are NL + 1 numbers; zero, which words hold before they are first written, is none of them."""
    c = SHAPES["gemma_320"].with_(weight_format="f16")
    model = make_model(c, seed=50, gamma_jitter=0.1)
    toks = list(range(1, 9))
    with InferenceState(c, model, max_seq=16, use_fp16=True) as inf:
        want = [inf.forward_token(t) for t in toks]
        first = inf.L.hip_inference_step_tag(inf.h, 0)
        for below in range(4 * c.NL + 8):
            inf.reset()
            assert inf.L.hip_inference_step_tag(inf.h, 2 ** 32 - below) == 2 ** 32 - below
            for i, t in enumerate(toks[:6]):
                assert np.array_equal(inf.forward_token(t), want[i]), (below, i)
            # (nothing but these reads the words of the argmax)
            assert [inf.forward_token_argmax(t) for t in toks[6:]] == [int(w.argmax()) for w in want[6:]], below
            left = below // (c.NL + 1)                     # steps whose tags all lie below the end
            if left < 8:
                assert inf.L.hip_inference_step_tag(inf.h, 0) == 1 + (8 - left) * (c.NL + 1), below
        assert first == 1 + 8 * (c.NL + 1) and one_launch(inf) == 8 * (4 * c.NL + 9)


def test_without_memory_for_its_words_a_state_decodes_in_launches():
    c = SHAPES["gemma_320"].with_(weight_format="f16")
    model = make_model(c, seed=49, gamma_jitter=0.1)
    with InferenceState(c, model, max_seq=16, use_fp16=True) as inf:
        inf.L.hip_gemm_profile_enable(1)
        want = np.stack([inf.forward_token(t) for t in (1, 2, 3)])
        inf.L.hip_gemm_profile_enable(0)
        inf.reset()
        inf.L.hip_inference_step_memory(inf.h, 1000)
        got = np.stack([inf.forward_token(t) for t in (1, 2, 3)])
        assert one_launch(inf) == 0 and np.array_equal(got, want)
        assert inf.forward_token_argmax(4) >= 0 and one_launch(inf) == 0


@pytest.mark.parametrize("kw", [dict(D=1120), dict(IS=6880), dict(V=1002), dict(hd=64, Hq=16), dict(D=2624), dict(IS=10304)], ids=str)
def test_shapes_that_stay_with_the_launches(kw):
    base = dict(NL=1, D=1152, Hq=4, Hkv=1, hd=256, IS=2048, V=1000)
    c = SFTConfig("t", QWEN3, **{**base, **kw}).with_(weight_format="f16")
    model = make_model(c, seed=45, gamma_jitter=0.1)
    with InferenceState(c, model, max_seq=8, use_fp16=True) as inf:
        for t in (1, 2, 3):
            assert np.isfinite(inf.forward_token(t)).all()
        assert one_launch(inf) == 0


# the last that fit and the first that do not, in turn: products of heads and their size, layers, a workgroup's rows where few of them share a product,
# heads beside workgroups for the O product
@pytest.mark.parametrize("kw,taken", [
    (dict(D=1152, hd=256, Hq=4, Hkv=1), True), (dict(D=1152, hd=256, Hq=5, Hkv=1), False),
    (dict(D=1152, hd=128, Hq=32, Hkv=8), True), (dict(D=1152, hd=128, Hq=33, Hkv=11), False),
    (dict(NL=48), True), (dict(NL=49), False),
    (dict(D=64, IS=640), True), (dict(D=64, IS=704), False),
    (dict(D=64, Hq=8), True), (dict(D=64, Hq=9), False)], ids=str)
def test_on_either_side_of_what_fits(kw, taken):
    c = SFTConfig("t", QWEN3, **{**dict(NL=1, D=128, Hq=2, Hkv=1, hd=128, IS=384, V=260), **kw}).with_(weight_format="f16")
    model = make_model(c, seed=53, gamma_jitter=0.1)
    toks = list(range(8))
    with InferenceState(c, model, max_seq=8, use_fp16=True) as inf:
        got = np.stack([inf.forward_token(t) for t in toks])
        assert one_launch(inf) == (len(toks) if taken else 0)
        inf.L.hip_gemm_profile_enable(1)
        inf.reset()
        want = np.stack([inf.forward_token(t) for t in toks])
        inf.L.hip_gemm_profile_enable(0)
    # (roundings in a row grow with the layers: some 40 of each)
    assert np.linalg.norm(got - want) <= max(200, 40 * c.NL) * 2.0 ** -24 * np.linalg.norm(want)


# either side of the line: vocabularies that few workgroups read too slowly, layers of narrow Q8_0 models with heads of 128, which cost more than
# the step saves
@pytest.mark.parametrize("kw,fmt,taken", [(dict(V=516), "f16", True), (dict(V=65536), "f16", False), (dict(V=65536), "q8_0", False),
                                          (dict(model_type=QWEN3, D=512, hd=128, Hq=8, Hkv=4, V=516, NL=4), "q8_0", True),
                                          (dict(model_type=QWEN3, D=512, hd=128, Hq=8, Hkv=4, V=516, NL=20), "q8_0", False),
                                          (dict(model_type=QWEN3, D=512, hd=128, Hq=8, Hkv=4, V=516, NL=20), "f16", True)], ids=str)
def test_shapes_that_are_faster_in_launches_stay_there(kw, fmt, taken):
    c = SHAPES["gemma_320"].with_(weight_format=fmt, **kw)
    model = make_model(c, seed=47, gamma_jitter=0.1)
    with InferenceState(c, model, max_seq=8, use_fp16=fmt == "f16") as inf:
        assert np.isfinite(inf.forward_token(1)).all()
        assert one_launch(inf) == int(taken)


def test_adapters_stay_with_the_launches():
    c = SHAPES["gemma_320"].with_(weight_format="f16", batch=1, seq=8)
    model = make_model(c, seed=46, gamma_jitter=0.1)
    with SFTState(c, model) as sft, InferenceState(c, model, max_seq=8, use_fp16=True) as inf:
        inf.forward_token(1)
        assert one_launch(inf) == 1
        inf.attach_lora(sft)
        inf.forward_token(2)
        assert one_launch(inf) == 1
