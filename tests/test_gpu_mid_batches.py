"""GPU parity of MoE batches between the decode batch and the long prompt, bit for bit against the CPU
restatement of moe_ffn_batch (model.rs:286-371): three and four tokens (routed by a launch of their
own), 8 to 15 tokens on the decode-batch kernels by default, Q6_K down on them, groups of 16 to 191
members on average with Q6_K gate/up and down (k_gemm_r), and Q4_K groups whose member tiles of 64
hold 1 to 4 tiles of 16 (k_gemm's sweeps), skewed groups among them; above 16 tokens, groups averaging
fewer than 16 members on k_gemm_mid: one or two member tiles, further tiles of an expert, one member.
"""
import numpy as np
import pytest

from bebelm_amd import synth
from bebelm_amd.model import Context, MoeLayer

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


# k_gemm_mid needs 160 blocks of 256 outputs: (hidden, moe_ff, experts, k, tokens, bias of expert 0)
MID = [
    (2048, 1792, 32, 4, 17, 0.0), (2048, 1280, 32, 4, 127, 0.0), (2048, 1536, 32, 2, 255, 0.0),
    (1280, 1280, 32, 3, 33, 3.0), (1280, 1280, 32, 1, 161, 3.0),   # expert 0 chosen by every token
    (1792, 2048, 23, 2, 65, 3.0), (512, 2048, 20, 2, 150, 0.0),    # down of 512 outputs: k_gemm
]


@pytest.mark.parametrize("case", MID, ids=lambda c: "-".join(map(str, c)))
@pytest.mark.parametrize("down", [Q4_K, Q6_K])
def test_groups_of_a_few(ctx, oracle, case, down):
    hidden, ff, E, K, T, b0 = case
    bias = np.zeros(E, np.float32)
    bias[0] = b0
    w = synth.moe_weights(T, hidden=hidden, moe_ff=ff, n_experts=E, n_used=K, gate_dtype=Q4_K, down_dtype=down,
                          bias=bias)
    x = synth.hidden_states(T + 1, T, hidden=hidden)
    x[T // 2, :256] = 0.0
    check_moe(ctx, oracle, w, x, T, f"groups of a few {case} {down}")


def kernels(ctx, layer, hidden, t):
    """The kernels that a call of t tokens launches."""
    ctx.reset_stats()
    ctx.profile(True)
    layer.forward(synth.hidden_states(3, t, hidden=hidden).reshape(-1), t, np.empty(t * hidden, np.float32))
    ctx.synchronize()
    ctx.profile(False)
    return set(ctx.kernel_stats())


def test_the_default_line_can_be_set_back(ctx):
    # a layer that the decode-batch kernels serve from 32 entries, and one entry less than that line
    layer = MoeLayer(ctx, synth.moe_weights(3, hidden=512, moe_ff=1024, n_experts=32, n_used=4))
    fresh = [kernels(ctx, layer, 512, t) for t in (7, 8)]
    assert "gemm_gateup" not in fresh[0] and "gemm_gateup" in fresh[1]
    ctx.set_batched_min_entries(1 << 40)
    assert "gemm_gateup" not in kernels(ctx, layer, 512, 8)
    ctx.set_batched_min_entries(64)
    assert [kernels(ctx, layer, 512, t) for t in (7, 8)] == fresh
    layer.close()


# (hidden, moe_ff, experts, k, down, tokens on the GEMV path, tokens on the batched one)
LINES = [
    (2048, 512, 8, 4, Q4_K, 15, 16), (2048, 1024, 4, 2, Q6_K, 16, 32), (2048, 1024, 16, 8, Q4_K, 7, 8),
    (2048, 1024, 20, 4, Q4_K, 8, 9), (2048, 1792, 12, 2, Q4_K, 15, 16), (512, 1024, 8, 8, Q4_K, 4, 5),
    (512, 1024, 12, 4, Q4_K, 7, 8), (512, 1024, 12, 4, Q6_K, 11, 12), (1024, 1024, 16, 4, Q4_K, 15, 16),
]


@pytest.mark.parametrize("case", LINES, ids=lambda c: "-".join(map(str, c)))
def test_the_default_line(ctx, case):
    # layers of few gate/up blocks keep the GEMV path longer
    hidden, ff, E, K, down, t0, t1 = case
    layer = MoeLayer(ctx, synth.moe_weights(4, hidden=hidden, moe_ff=ff, n_experts=E, n_used=K, gate_dtype=Q4_K,
                                            down_dtype=down))
    assert "gemm_gateup" not in kernels(ctx, layer, hidden, t0)
    assert "gemm_gateup" in kernels(ctx, layer, hidden, t1)
    layer.close()


# Q6_K down on k_down16: 160 blocks of 256 rows and more; rows of 1 to 8 super-blocks, and one case below
@pytest.mark.parametrize("case", [(2048, 256, 20, 4, 16), (2048, 512, 23, 3, 9), (1280, 1280, 32, 4, 16),
                                  (1792, 2048, 23, 5, 12), (2048, 768, 19, 4, 16)],
                         ids=lambda c: "-".join(map(str, c)))
def test_q6_down_of_decode_batches(ctx, oracle, case):
    hidden, ff, E, K, T = case
    w = synth.moe_weights(T, hidden=hidden, moe_ff=ff, n_experts=E, n_used=K, gate_dtype=Q4_K, down_dtype=Q6_K)
    x = synth.hidden_states(T + 2, T, hidden=hidden)
    ctx.set_batched_min_entries(1)
    check_moe(ctx, oracle, w, x, T, f"decode batch {case}")
    ctx.set_batched_min_entries(64)


# (hidden, experts, k, tokens, a launch for the route): three and four tokens
@pytest.mark.parametrize("case", [(512, 8, 2, 3, False), (512, 20, 2, 4, False), (768, 8, 2, 3, True), (1024, 8, 4, 4, True)],
                         ids=lambda c: "-".join(map(str, c)))
def test_routes_of_three_and_four_tokens(ctx, oracle, case):
    hidden, E, K, T, launch = case
    w = synth.moe_weights(T + E, hidden=hidden, moe_ff=512, n_experts=E, n_used=K)
    layer = MoeLayer(ctx, w)
    assert ("route_gating" in kernels(ctx, layer, hidden, T)) == launch
    layer.close()
    check_moe(ctx, oracle, w, synth.hidden_states(T + 3, T, hidden=hidden), T, f"routes {case}")
