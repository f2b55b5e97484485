"""GPU parity of batched projections (k_proj, tiled Q8 activations; the grouped GEMM past 768
tokens) against the CPU restatement: the dense FFN (matmul, kernels/matmul.rs:908-991), the conv
operator and an attention operator whose k and v have no packed form (64 rows: their input then
stays row-major). Sizes at the edges of its cuts: one to three member tiles of 16 tokens and past
each group of four, rows of 1 to 10 super-blocks over 2 to 8 waves, 768 and 769 tokens. Outputs are
bit-identical: the integer parts are exact and every f32 operation is in the reference's order.
"""
import numpy as np
import pytest

from bebelm_amd import synth
from bebelm_amd.model import AttnOp, ConvOp, DenseLayer

from test_gpu_parity import Q4_K, Q6_K, assert_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [Q4_K, Q6_K])
@pytest.mark.parametrize("hidden,ff,ts", [
    (256, 768, (2, 15, 16, 17, 768, 769)),      # rows of 1 and 3 super-blocks
    (512, 1792, (3, 31, 33, 48, 65, 129)),      # 2 and 7
    (1024, 2560, (2, 49, 64, 112, 257)),        # 4 and 10 (long rows of few row tiles)
])
def test_dense_batches(gpu_ctx, oracle, hidden, ff, ts, dtype):
    w = synth.dense_weights(hidden + dtype, hidden=hidden, ff=ff, dtype=dtype)
    layer = DenseLayer(gpu_ctx, w)
    for t in ts:
        x = synth.hidden_states(hidden + t, t, hidden=hidden)
        x[t // 2] = 0.0                      # a zero row: scale 0
        x[t - 1, :256] *= np.float32(1e4)
        got = layer.forward(x.reshape(-1), t, np.empty(t * hidden, np.float32))
        assert_bits(got, oracle.dense_ffn(w, x.reshape(-1), t), f"dense {hidden}x{ff} dtype {dtype} t={t}")
    layer.close()


# past 768 tokens, one group of the grouped GEMM: Q4_K tiles of 80 (783 and 1025 tokens) and of 64 (1281),
# Q6_K gate/up in tiles of 64, Q6_K down in k_gemm_wide's chunks (16, 8, 4, 2 and 1 member tiles), the
# last tile of each partly empty
@pytest.mark.parametrize("t", [783, 1025, 1281])
@pytest.mark.parametrize("dtype", [Q4_K, Q6_K])
def test_one_group(gpu_ctx, oracle, dtype, t):
    w = synth.dense_weights(21 + dtype, hidden=256, ff=768, dtype=dtype)
    layer = DenseLayer(gpu_ctx, w)
    x = synth.hidden_states(t, t, hidden=256).reshape(-1)
    got = layer.forward(x, t, np.empty(t * 256, np.float32))
    assert_bits(got, oracle.dense_ffn(w, x, t), f"dense one group dtype {dtype} t={t}")
    layer.close()
    w = synth.conv_weights(22, hidden=256, in_dtype=dtype, out_dtype=Q4_K + Q6_K - dtype)
    op = ConvOp(gpu_ctx, w)
    state = op.new_state()
    want, new = oracle.conv_forward(w, state, x, t)
    assert_bits(op.forward(state, x, t, np.empty(t * 256, np.float32)), want, f"conv one group dtype {dtype} t={t}")
    assert_bits(state, new, f"conv state after t={t}")
    op.close()


@pytest.mark.parametrize("dtypes", [(Q4_K, Q6_K), (Q6_K, Q4_K)])
def test_conv_batches(gpu_ctx, oracle, dtypes):
    w = synth.conv_weights(11, hidden=512, in_dtype=dtypes[0], out_dtype=dtypes[1])
    op = ConvOp(gpu_ctx, w)
    state = op.new_state()
    for t in (2, 16, 31, 66):                # one conversation: the conv cache carries over
        x = synth.hidden_states(80 + t, t, hidden=512).reshape(-1)
        want, new = oracle.conv_forward(w, state, x, t)
        got = op.forward(state, x, t, np.empty(t * 512, np.float32))
        assert_bits(got, want, f"conv t={t}")
        assert_bits(state, new, f"conv state t={t}")
    op.close()


def test_attention_with_unpacked_projections(gpu_ctx, oracle):
    w = synth.attn_weights(12, hidden=256, n_heads=4, n_kv_heads=1, head_dim=64)
    op = AttnOp(gpu_ctx, w)
    kv, okv, pos = op.new_cache(128), oracle.KvCache(w.kv_dim, 128), 0
    for t in (5, 40, 1, 17):
        x = synth.hidden_states(90 + t, t, hidden=256).reshape(-1)
        want = oracle.attn_forward(w, okv, pos, x, t)
        got = op.forward(kv, pos, x, t, np.empty(t * 256, np.float32))
        assert_bits(got, want, f"attention t={t}")
        pos += t
    kv.close()
    op.close()


@pytest.mark.parametrize("taps", [2, 3, 6, 16, 17])
def test_conv_one_launch(gpu_ctx, oracle, taps):
    # k_conv_q8: batches shorter and longer than the state, whole and partial groups of tokens (17 taps
    # keep the separate kernels), each batch continuing from the state of the one before
    w = synth.conv_weights(91 + taps, hidden=256, l_cache=taps, in_dtype=Q6_K, out_dtype=Q4_K)
    op = ConvOp(gpu_ctx, w)
    state = op.new_state()
    for i, t in enumerate((2, 3, 1, 4, 5, 17, 8, 33)):
        x = synth.hidden_states(50 + i, t, hidden=256).reshape(-1)
        want, new = oracle.conv_forward(w, state, x, t)
        assert_bits(op.forward(state, x, t, np.empty(t * 256, np.float32)), want, f"{taps} taps, {t} tokens")
        assert_bits(state, new, f"{taps} taps, state after {t} tokens")
    op.close()


@pytest.mark.parametrize("taps", [3, 4, 5, 8, 9, 16])
def test_conv_in_groups_of_tokens(gpu_ctx, oracle, taps):
    # one and four tokens a wave, filters shorter than their kernel's longest, blocks partly past the batch
    w = synth.conv_weights(120 + taps, hidden=512, l_cache=taps, in_dtype=Q4_K, out_dtype=Q6_K)
    op = ConvOp(gpu_ctx, w)
    state = op.new_state()
    for i, t in enumerate((15, 1, 64, 16, 301)):
        x = synth.hidden_states(60 + i, t, hidden=512).reshape(-1)
        want, new = oracle.conv_forward(w, state, x, t)
        assert_bits(op.forward(state, x, t, np.empty(t * 512, np.float32)), want, f"{taps} taps, {t} tokens")
        assert_bits(state, new, f"{taps} taps, state after {t} tokens")
    op.close()
