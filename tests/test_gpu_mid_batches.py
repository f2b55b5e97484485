"""GPU parity of MoE batches between the decode batch and the long prompt, bit for bit against the CPU
restatement of moe_ffn_batch (model.rs:286-371): three and four tokens (routed by a launch of their
own), 8 to 15 tokens on the decode-batch kernels by default, Q6_K down on them, groups of 16 to 191
members on average with Q6_K gate/up and down (k_gemm_r), and Q4_K groups whose member tiles of 64
hold 1 to 4 tiles of 16 (k_gemm's sweeps), skewed groups among them.
"""
import numpy as np
import pytest

from bebelm_amd import synth
from bebelm_amd.model import Context

from test_gpu_parity import Q4_K, Q6_K, check_moe

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    """A context whose batched threshold nobody set."""
    c = Context(0)
    yield c
    c.close()


# (hidden, moe_ff, experts, k, tokens, gate, down)
CASES = [
    (512, 512, 8, 2, 3, Q4_K, Q6_K), (512, 512, 8, 2, 4, Q6_K, Q4_K),
    (512, 256, 32, 4, 8, Q4_K, Q6_K), (2048, 1792, 32, 4, 11, Q4_K, Q6_K), (512, 2048, 16, 4, 15, Q4_K, Q4_K),
    (512, 1280, 7, 3, 16, Q4_K, Q6_K), (1024, 512, 16, 4, 9, Q4_K, Q4_K),   # hidden 1024: the GEMV path below 64
    (512, 768, 4, 2, 33, Q6_K, Q6_K), (512, 512, 4, 1, 100, Q6_K, Q6_K),    # groups of 16 and 25
    (256, 256, 4, 2, 129, Q6_K, Q6_K), (512, 256, 3, 1, 570, Q6_K, Q6_K),   # 64 and 190
    (512, 512, 8, 2, 64, Q4_K, Q4_K), (512, 256, 8, 2, 101, Q4_K, Q4_K), (512, 256, 8, 2, 190, Q4_K, Q4_K),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_mid_batches(ctx, oracle, case):
    hidden, ff, E, K, T, gate, down = case
    w = synth.moe_weights(T + ff, hidden=hidden, moe_ff=ff, n_experts=E, n_used=K, gate_dtype=gate, down_dtype=down)
    x = synth.hidden_states(T, T, hidden=hidden)
    x[T // 2, :256] = 0.0
    check_moe(ctx, oracle, w, x, T, f"mid batch {case}")


@pytest.mark.parametrize("gate,down", [(Q4_K, Q6_K), (Q6_K, Q4_K)])
def test_skewed_groups(ctx, oracle, gate, down):
    # a bias that sends every token to expert 0 and few to the last ones: groups of 96, 1 and 0 members
    bias = np.array([3.0] + [0.0] * 2 + [-0.4] * 3, np.float32)
    w = synth.moe_weights(5, hidden=512, moe_ff=512, n_experts=6, n_used=2, gate_dtype=gate, down_dtype=down, bias=bias)
    x = synth.hidden_states(9, 96, hidden=512)
    check_moe(ctx, oracle, w, x, 96, f"skewed groups {gate} {down}")
