"""The flash launcher's choice of key splits (sca_hip_flash_split_bytes), on the CPU: a plan for 256 CUs
from the parameters alone."""

import pytest

import sca_amd
from attn_util import DTYPE_ID
from sca_amd import hip as H

MAX_BYTES = 64 << 20


def plan(B, Hq, Hkv, Sq, Skv, D, causal=True, **changes):
    """(splits, bytes); 0 splits: the call would not split."""
    p = H.FlashParams()
    p.q = p.k = p.v = p.out = 4096  # never read
    p.batch, p.num_heads, p.num_kv_heads = B, Hq, Hkv
    p.seq_q, p.seq_kv, p.head_dim = Sq, Skv, D
    p.q_sb, p.q_sh, p.q_ss = Hq * Sq * D, Sq * D, D
    p.k_sb, p.k_sh, p.k_ss = Hkv * Skv * D, Skv * D, D
    p.v_sb, p.v_sh, p.v_ss = p.k_sb, p.k_sh, p.k_ss
    p.o_sb, p.o_sh, p.o_ss = p.q_sb, p.q_sh, p.q_ss
    p.scale, p.causal, p.dtype = 0.1, int(causal), DTYPE_ID["bf16"]
    p.diagonal = Skv - Sq if causal else 0
    for name, value in changes.items():
        setattr(p, name, value)
    want = sca_amd.hip_lib().sca_hip_flash_split_bytes
    want.restype = H.c_i64
    n = want(H.ctypes.byref(p))
    state = B * Hq * Sq * (D + 2) * 4  # one fp32 O, m and l per row and split
    assert n % state == 0 and n <= MAX_BYTES
    return n // state, n


@pytest.mark.parametrize("shape,splits", [
    ((1, 32, 8, 512, 12801, 128), 2),   # a chunk: 128 row tiles for 256 CUs
    ((8, 32, 8, 6, 4102, 128), 4),      # a few tokens: 64 packed units
    ((1, 32, 8, 1000, 1000, 128), 0),   # pairs fill the GPU
    ((4, 32, 8, 8192, 8192, 128), 0),   # many row tiles
    ((24, 32, 8, 256, 1354, 128), 0),   # row tiles for every CU
    ((1, 24, 8, 256, 1354, 128), 0),    # pairs on a half-idle GPU: the merge costs more than it gives
])
def test_splits_of_known_shapes(shape, splits):
    assert plan(*shape)[0] == splits


@pytest.mark.parametrize("D", [32, 64, 96, 128, 160, 192, 256])
@pytest.mark.parametrize("causal", [True, False])
def test_bounds_over_lengths(D, causal):
    """At most 16 splits of 256 keys each, and 64 MiB; never one split; short calls never split."""
    for Sq in (1, 7, 128, 513):
        for Skv in (600, 1023, 1024, 5000, 100001):
            for B, Hq, Hkv in ((1, 8, 2), (2, 28, 4), (1, 1, 1)):
                splits, _ = plan(B, Hq, Hkv, Sq, Skv, D, causal)
                assert splits == 0 or 2 <= splits <= min(16, Skv // 256), (B, Hq, Sq, Skv)
        if Sq <= 511:
            assert plan(1, 8, 2, Sq, 511, D, causal)[0] == 0


def test_calls_the_dma_kernels_do_not_serve_do_not_split():
    few = (8, 32, 8, 6, 4102, 128)
    assert plan(*few)[0] > 0
    assert plan(*few, k_ss=-128)[0] == 0
    assert plan(*few, v_ss=1 << 20)[0] == 0       # past the 32-bit buffer offsets
    assert plan(*few, num_kv_heads=5)[0] == 0     # invalid: the launch itself says why
    assert plan(*few, dtype=DTYPE_ID["f32"])[0] == 0
