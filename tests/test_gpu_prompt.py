"""Prompts taken many tokens per step (inference_forward_tokens, the prefill of inference_generate and _generate_batch) against
the same tokens one by one, which the other tests hold to the oracle.  Both keep fp32 (22 bits in the products' operands), so
they agree to about sqrt(layers) ulps of the largest logit: 2e-5 leaves a factor of ten."""
import numpy as np
import pytest

from llm_metal_amd import lib
from llm_metal_amd.configs import C1, GEMMA3, QWEN3, SFTConfig
from llm_metal_amd.sft import InferenceState, SFTState
from llm_metal_amd.synth import make_batch, make_model
from tests.decode_chain import oracle_decode
from tests.gpu_util import maxrel, rel

pytestmark = pytest.mark.gpu
TOL = 2e-5
SHAPES = [
    SFTConfig("hd32_group4", QWEN3, NL=2, D=160, Hq=8, Hkv=2, hd=32, IS=416, V=512),
    SFTConfig("hd64_group3", QWEN3, NL=2, D=192, Hq=3, Hkv=1, hd=64, IS=352, V=516),
    SFTConfig("hd128_group1", QWEN3, NL=2, D=288, Hq=2, Hkv=2, hd=128, IS=608, V=512),
    SFTConfig("hd128_group16", QWEN3, NL=1, D=256, Hq=16, Hkv=1, hd=128, IS=4224, V=512),
    SFTConfig("hd256_gemma", GEMMA3, NL=7, D=128, Hq=4, Hkv=1, hd=256, IS=256, V=512, tied=True),
    SFTConfig("hd16_one_by_one", QWEN3, NL=1, D=128, Hq=4, Hkv=2, hd=16, IS=256, V=512),
]


def tokens(c, n, seed):
    return [int(t) for t in np.random.default_rng(seed).integers(0, c.V, n)]


def one_by_one(inf, toks):
    inf.reset()
    return np.stack([inf.forward_token(t) for t in toks])


@pytest.mark.parametrize("n", [2, 7, 31, 33, 65, 130, 300])
@pytest.mark.parametrize("fmt", ["f16", "q8_0"])
@pytest.mark.parametrize("c", SHAPES, ids=lambda c: c.name)
def test_prompt_equals_tokens_one_by_one(c, fmt, n):
    print(c.name, fmt, n, flush=True)
    model, toks = make_model(c, seed=3, gamma_jitter=0.1), tokens(c, n + 3, n)
    with InferenceState(c, model, max_seq=n + 3, use_fp16=fmt == "f16") as inf:
        want = one_by_one(inf, toks)
        inf.reset()
        got = inf.forward_tokens(toks[:n], range(n))
        assert inf.position() == n and maxrel(got, want[:n]) < TOL
        # decoding goes on from the caches the prompt left, and so does a further portion
        assert maxrel(inf.forward_token(toks[n]), want[n]) < TOL
        assert maxrel(inf.forward_tokens(toks[n + 1:], [1]), want[-1:]) < TOL
        cut = max(1, n // 3)
        inf.reset()
        inf.forward_tokens(toks[:cut])
        assert maxrel(inf.forward_tokens(toks[cut:n], [n - cut - 1]), want[n - 1:n]) < TOL


@pytest.mark.parametrize("n", [5, 16, 17, 32, 64])
@pytest.mark.parametrize("fmt", ["f16", "q8_0"])
@pytest.mark.parametrize("kw", [dict(D=1184, Hq=2, Hkv=1, hd=128, IS=2080), dict(D=2560, Hq=4, Hkv=2, hd=128, IS=9728)], ids=["ragged", "many_chunks"])
@pytest.mark.parametrize("model_type", [QWEN3, GEMMA3], ids=["qwen3", "gemma3"])
def test_short_prompts_on_either_side_of_an_operand_tile(kw, fmt, n, model_type):
    """16 tokens fill the 32 rows of one operand tile with their two images, 32 those of two, 64 are two steps of a Q8_0 state; columns
    that fill no group of four Q8_0 blocks (1184), K in one chunk and in several."""
    print(kw, fmt, n, flush=True)
    c = SFTConfig("short", model_type, NL=2, V=260, tied=True, **kw)
    model, toks = make_model(c, seed=6, gamma_jitter=0.1), tokens(c, n, n)
    with InferenceState(c, model, max_seq=n, use_fp16=fmt == "f16") as inf:
        want = one_by_one(inf, toks)
        inf.reset()
        assert maxrel(inf.forward_tokens(toks, range(n)), want) < TOL


@pytest.mark.parametrize("n", [63, 64, 65])
@pytest.mark.parametrize("hd,group", [(128, 4), (256, 2), (256, 1)])
def test_attention_on_either_side_of_64_keys(hd, group, n):
    """Up to 64 keys a wave takes a token's head, beyond them the tiles do: whole prompts, and portions that end there and begin behind
    others (positions 20 and 40), seven tokens of them so that the last wave of a workgroup has nothing to do."""
    print(hd, group, n, flush=True)
    c = SFTConfig("short_keys", QWEN3, NL=1, D=128, Hq=group, Hkv=1, hd=hd, IS=96, V=260, tied=True)
    model, toks = make_model(c, seed=8, gamma_jitter=0.1), tokens(c, n, n)
    with InferenceState(c, model, max_seq=n, use_fp16=True) as inf:
        want = one_by_one(inf, toks)
        for cuts in ((), (20,), (20, 40, n - 7)):
            inf.reset()
            at = (0,) + cuts + (n,)
            got = np.concatenate([inf.forward_tokens(toks[a:b], range(b - a)) for a, b in zip(at, at[1:])])
            assert maxrel(got, want) < TOL, cuts


@pytest.mark.parametrize("n", [265, 300, 545])
def test_attention_with_workgroups_in_either_order(n):
    """Heads of 128 over eight key heads: up to 512 workgroups the second half comes shortest first, from 516 tokens on all of them longest
    first; last tiles of rows and keys full and not, a portion that begins inside a tile."""
    print(n, flush=True)
    c = SFTConfig("orders", QWEN3, NL=1, D=128, Hq=32, Hkv=8, hd=128, IS=96, V=260, tied=True)
    model, toks = make_model(c, seed=12, gamma_jitter=0.1), tokens(c, n, n)
    with InferenceState(c, model, max_seq=n, use_fp16=True) as inf:
        want = one_by_one(inf, toks)
        for cuts in ((), (77,)):
            inf.reset()
            at = (0,) + cuts + (n,)
            got = np.concatenate([inf.forward_tokens(toks[a:b], range(b - a)) for a, b in zip(at, at[1:])])
            assert maxrel(got, want) < TOL, cuts


@pytest.mark.parametrize("hd", [128, 256])
def test_infinite_values_inside_a_tile_stay_with_later_tokens(hd):
    """Tokens before one whose keys and values are not finite, in the same 32 keys and in earlier ones, do not see it."""
    c = SFTConfig("inf", QWEN3, NL=1, D=128, Hq=4, Hkv=2, hd=hd, IS=96, V=260)
    model, toks = make_model(c, seed=13), list(range(150))
    with InferenceState(c, model, max_seq=150) as inf:
        want = inf.forward_tokens(toks, range(150))
    model["token_emb"][110] = np.inf
    with InferenceState(c, model, max_seq=150) as inf:
        got = inf.forward_tokens(toks, range(150))
    assert maxrel(got[:110], want[:110]) < TOL and np.isfinite(got[:110]).all()
    assert not np.isfinite(got[110:]).any()


def test_prompt_of_several_steps():
    c = C1.with_(name="long", NL=1, V=256)
    model, toks = make_model(c, seed=4), tokens(c, 2500, 5)
    at = [0, 832, 833, 1024, 1666, 1667, 2499]
    with InferenceState(c, model, max_seq=2500) as inf:
        want = one_by_one(inf, toks)[at]
        inf.reset()
        assert maxrel(inf.forward_tokens(toks, at), want) < TOL


@pytest.mark.parametrize("fmt", ["f16", "q8_0"])
def test_prompt_with_adapters(fmt):
    """On a training state's tiles (adapter rows inside the fused matrix) and on own weights with its adapters attached."""
    c = C1.with_(weight_format=fmt)
    model, toks = make_model(c, seed=6, gamma_jitter=0.1), tokens(c, 72, 7)
    with SFTState(c, model) as sft:
        sft.train_step(*make_batch(c, seed=8), 1e-3)
        with InferenceState(sft=sft, max_seq=80) as shared, InferenceState(c, model, max_seq=80, use_fp16=fmt == "f16") as own:
            own.attach_lora(sft)
            for inf in (shared, own):
                want = one_by_one(inf, toks)
                inf.reset()
                assert maxrel(inf.forward_tokens(toks[:60], range(60)), want[:60]) < TOL
                # a further portion and single tokens go on from the caches it left
                assert maxrel(inf.forward_tokens(toks[60:70], range(10)), want[60:70]) < TOL
                assert maxrel(inf.forward_token(toks[70]), want[70]) < TOL
                assert maxrel(inf.forward_token(toks[71]), want[71]) < TOL and inf.position() == 72


def test_prompts_on_the_q8_tiles_of_a_training_state():
    """Products of gate|up go through an F16 image of the tiles from 512 rows on (160 blocks of 128 x 256), and at any length where the
    large-M kernel is asked for (1: on images, 2: on the tiles as they are); the image holds the values that a tile is unpacked to."""
    c = C1.with_(name="q8_tiles", weight_format="q8_0", IS=2464)
    model, toks, L = make_model(c, seed=9, gamma_jitter=0.1), tokens(c, 1024, 10), lib.load()
    with SFTState(c, model) as sft:
        sft.train_step(*make_batch(c, seed=8), 1e-3)
        with InferenceState(sft=sft, max_seq=1024) as inf:
            want = one_by_one(inf, toks)
            for policy, n in ((0, 6), (0, 500), (0, 511), (0, 512), (0, 513), (0, 600), (0, 1024), (1, 40), (1, 100), (2, 100)):
                print(policy, n, flush=True)
                rows = sorted({0, n // 3, n - 2, n - 1})
                L.hip_gemm_force_large_m(policy)
                try:
                    inf.reset()
                    assert maxrel(inf.forward_tokens(toks[:n], rows), want[rows]) < TOL
                finally:
                    L.hip_gemm_force_large_m(0)


def test_generation_from_prompts():
    c = C1
    model, prompt = make_model(c, seed=9, gamma_jitter=0.1), tokens(C1, 45, 10)
    with InferenceState(c, model, max_seq=64) as inf:
        inf.set_eos([c.V - 1])
        nxt, want = int(one_by_one(inf, prompt)[-1].argmax()), []
        for _ in range(10):
            want.append(nxt)
            nxt = inf.forward_token_argmax(nxt)
        assert list(inf.generate(prompt, 10)) == want
        assert [list(r) for r in inf.generate_batch(prompt, 10, 3)] == [want] * 3
        assert list(inf.generate(prompt[:5] + [c.V], 4)) == [] and inf.position() == 5


def test_infinite_values_stay_with_later_tokens():
    c = SHAPES[2].with_(NL=1)
    model, toks = make_model(c, seed=11), list(range(50))
    with InferenceState(c, model, max_seq=50) as inf:
        want = inf.forward_tokens(toks, range(50))
    model["token_emb"][20] = np.inf
    with InferenceState(c, model, max_seq=50) as inf:
        got = inf.forward_tokens(toks, range(50))
    assert maxrel(got[:20], want[:20]) < TOL and np.isfinite(got[:20]).all()
    assert not np.isfinite(got[20:]).any()


def test_q8_weights_beyond_a_half_take_tokens_one_by_one():
    c = SHAPES[2].with_(NL=1)
    model = make_model(c, seed=12)
    model["wd"][0] *= 1e7                                  # code times scale beyond 65504
    toks = tokens(c, 40, 13)
    with InferenceState(c, model, max_seq=40, use_fp16=False) as inf:
        want = one_by_one(inf, toks)
        inf.reset()
        assert np.isfinite(want).all() and np.array_equal(inf.forward_tokens(toks, range(40)), want)


@pytest.mark.parametrize("D,IS", [(32, 260), (1184, 352), (4128, 416)])
def test_norms_of_a_batch(D, IS):
    """The norm between a batch's products in pieces of four columns: a row shorter than its padding, one piece and two per
    thread.  Single sequences go another way."""
    print(D, IS, flush=True)
    c = SFTConfig("odd", QWEN3, NL=2, D=D, Hq=2, Hkv=1, hd=64, IS=IS, V=512)
    model = make_model(c, seed=13, gamma_jitter=0.1)
    seqs = np.random.default_rng(5).integers(0, c.V, (3, 4))
    with InferenceState(c, model, max_seq=8) as inf:
        got = np.stack([inf.step_batch(seqs[:, i], i) for i in range(4)], axis=1)
        for b in range(3):
            assert maxrel(got[b], one_by_one(inf, [int(t) for t in seqs[b]])) < TOL


@pytest.mark.parametrize("n", [20, 40, 100])
@pytest.mark.parametrize("c", [SFTConfig("long_k", QWEN3, NL=1, D=2560, Hq=4, Hkv=2, hd=128, IS=2560, V=512),
                               SFTConfig("gemma_hd256", GEMMA3, NL=2, D=1024, Hq=4, Hkv=1, hd=256, IS=2048, V=512, tied=True)], ids=lambda c: c.name)
def test_prompt_is_as_exact_as_single_tokens(c, n):
    """Against 64 bits, over all rows of logits: sums in the matrix cores' accumulators, rounded at every instruction, are no
    further off than the lanes' sums of the single-token kernels.  (Equal within the noise of the roundings, 3 % over these rows;
    with one accumulator per sum the prompt was 1.2 to 1.4 times as far off.)"""
    print(c.name, n, flush=True)
    model, toks = make_model(c, seed=31, gamma_jitter=0.1), tokens(c, n, n)
    want = oracle_decode(c, model, "f16", toks, n, precision="f64")
    with InferenceState(c, model, max_seq=n) as inf:
        single = one_by_one(inf, toks)
        inf.reset()
        got = inf.forward_tokens(toks, range(n))
    print(rel(got, want), rel(single, want))
    assert rel(got, want) < 1.1 * rel(single, want)


def test_prompt_tiles_kept_or_formed_per_product():
    """Without room for the tiles of its weights a state forms them in scratch for every product: the same logits, bit for bit, the
    head's included (70000 rows go in two parts; 1312 columns and 2084 rows leave padding)."""
    c = C1.with_(name="tiles", D=1312, IS=2084, NL=2, Hq=12, Hkv=4, V=70000)
    model, toks, got = make_model(c, seed=41, gamma_jitter=0.1), tokens(c, 90, 42), []
    L = lib.load()
    for mb in (0, 65536):
        L.hip_gemm_image_budget_mb(mb)
        try:
            with InferenceState(c, model, max_seq=90) as inf:
                want = one_by_one(inf, toks[:40]) if not got else None
                inf.reset()
                got.append(inf.forward_tokens(toks, range(3, 40)))
                if want is not None:
                    assert maxrel(got[0], want[3:]) < TOL
        finally:
            L.hip_gemm_image_budget_mb(65536)
    assert np.array_equal(got[0], got[1])
