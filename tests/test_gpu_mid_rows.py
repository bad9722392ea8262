"""Products of 65 to 1023 rows: the planner's choice of kernel, block and K chunks (and the stores of tiles that reach past the
matrix) against the streaming kernel alone.  Both add the same fp16 products in fp32 in another order; what that changes flips
roundings of the next operand to fp16, 2^-12 of an element here and there: 5e-4 over a tensor leaves a factor of five."""
import numpy as np
import pytest

from llm_metal_amd import lib
from llm_metal_amd.configs import C1, GEMMA3, QWEN3, SFTConfig
from llm_metal_amd.sft import InferenceState, SFTState
from llm_metal_amd.synth import make_batch, make_model
from tests.gpu_util import maxrel, rel

pytestmark = pytest.mark.gpu
# widths that no tile divides: 2084 = 65 blocks of 32 + 4, 1312 = 20.5 K steps, 8212 columns in the head
WIDE = SFTConfig("mid_qwen", QWEN3, NL=2, D=1312, Hq=12, Hkv=4, hd=64, IS=2084, V=8212)
GEMMA = SFTConfig("mid_gemma", GEMMA3, NL=2, D=608, Hq=4, Hkv=1, hd=128, IS=4128, V=6148, tied=True)


@pytest.mark.parametrize("rows", [65, 96, 129, 192, 250, 257, 511, 640, 1000, 1023])
@pytest.mark.parametrize("cfg", [WIDE, GEMMA], ids=lambda c: c.name)
def test_step_equals_streaming_kernel(cfg, rows):
    print(cfg.name, rows, flush=True)
    batch = 2 if rows % 2 == 0 else 1
    c = cfg.with_(batch=batch, seq=rows // batch)
    model = make_model(c, seed=21, gamma_jitter=0.1)
    tok, tgt = make_batch(c, seed=22)
    L, got = lib.load(), []
    for policy in (-1, 0):
        L.hip_gemm_force_large_m(policy)
        try:
            with SFTState(c, model) as st:
                loss = st.train_step(tok, tgt, 1e-4)
                got.append((loss, st.logits(), st.lora_grads()))
        finally:
            L.hip_gemm_force_large_m(0)
    (la, za, ga), (lb, zb, gb) = got
    assert np.isfinite(lb) and abs(la - lb) < 1e-5 * abs(la)
    assert rel(zb, za) < 5e-4 and rel(gb, ga) < 5e-4


@pytest.mark.parametrize("rows", [100, 250, 800])
def test_full_parameter_pass_equals_streaming_kernel(rows):
    c = WIDE.with_(NL=1, R=0, seq=rows)
    model = make_model(c, seed=23)
    tok, tgt = make_batch(c, seed=24)
    L, got = lib.load(), []
    for policy in (-1, 0):
        L.hip_gemm_force_large_m(policy)
        try:
            with SFTState(c, model) as st:
                st.alloc_grad_accum()
                st.train_step(tok, tgt, 1e-3)
                got.append([st.matrix_f16(0, k, 2).view(np.float16).astype(np.float32) for k in st.MATRICES])
        finally:
            L.hip_gemm_force_large_m(0)
    for a, b in zip(*got):
        assert rel(b, a) < 5e-3                             # the accumulators themselves are F16


@pytest.mark.parametrize("n", [33, 100, 400, 511, 513, 1000, 1024])
def test_prompt_equals_streaming_kernel(n):
    c = C1.with_(name="mid_prompt", D=1312, IS=2084, NL=2, Hq=12, Hkv=4, V=2052)
    model = make_model(c, seed=25, gamma_jitter=0.1)
    toks = np.random.default_rng(26).integers(0, c.V, n)
    L, got = lib.load(), []
    with InferenceState(c, model, max_seq=n) as inf:
        for policy in (-1, 0, 1):
            L.hip_gemm_force_large_m(policy)
            try:
                inf.reset()
                got.append(inf.forward_tokens(toks, range(0, n, 7)))
            finally:
                L.hip_gemm_force_large_m(0)
    assert rel(got[1], got[0]) < 5e-6 and rel(got[2], got[0]) < 5e-6          # operands of 22 bits


def test_rows_of_many_columns():
    """Blocks that reach past a matrix of 2.6 million columns: 256 of its rows are more bytes than one descriptor's offsets have
    bits.  Targets in the last, ragged block of columns, in the last rows of the only block of rows."""
    c = C1.with_(name="wide_head", NL=1, D=64, Hq=2, Hkv=1, hd=32, IS=64, V=2_600_004, seq=256, R=2, tied=True)
    model = make_model(c, seed=27)
    tok, _ = make_batch(c, seed=28)
    tgt = (c.V - 1 - np.arange(c.BN) % 100).astype(np.uint32)
    L, got = lib.load(), []
    for policy, block in ((-1, 0), (1, 2), (1, 1)):
        L.hip_gemm_force_large_m(policy)
        L.hip_gemm_large_m_block(block)
        try:
            with SFTState(c, model) as st:
                st.train_step(tok, tgt, 0.0)
                got.append(st.losses())
        finally:
            L.hip_gemm_force_large_m(0)
            L.hip_gemm_large_m_block(0)
    assert np.ptp(got[0]) > 0 and maxrel(got[1], got[0]) < 1e-5 and maxrel(got[2], got[0]) < 1e-5
