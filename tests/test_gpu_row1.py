"""GPU parity of one token through the kernels that prepare their activations themselves
(csrc/bb_row1.hip) against the CPU restatement, bit for bit: the dense FFN (gate, up and SwiGLU,
down), the conv operator (projection, conv and state), the attention operator's projections, and
FFN stacks in which a dense layer follows a dense layer, an MoE layer and nothing. Rows of 1 to 32
super-blocks, output counts that leave a block partly empty, both weight types, filters of 2 to 4
taps (and 5, which keeps the separate kernels). The rmsnorm's f64 sum is a tree (about one f32
result in 1e9 may differ from the reference's left-to-right sum); these inputs have none.
"""
import numpy as np
import pytest

from bebelm_amd import synth
from bebelm_amd.model import AttnOp, ConvOp, DenseLayer, FfnStack, MoeLayer

from test_gpu_parity import Q4_K, Q6_K, assert_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [Q4_K, Q6_K])
@pytest.mark.parametrize("hidden,ff", [(256, 256), (512, 2304), (768, 1792), (2048, 8192), (1024, 8448)])
def test_dense_one_token(gpu_ctx, oracle, hidden, ff, dtype):
    w = synth.dense_weights(hidden + ff, hidden=hidden, ff=ff, dtype=dtype)
    layer = DenseLayer(gpu_ctx, w)
    for seed in (1, 2):
        x = synth.hidden_states(seed, 1, hidden=hidden).reshape(-1)
        x[:256] *= np.float32(0.0 if seed == 2 else 1.0)  # a zero block: scale 0
        assert_bits(layer.dense_ffn(x), oracle.dense_ffn(w, x, 1), f"dense {hidden}x{ff} dtype {dtype}")
    layer.close()


@pytest.mark.parametrize("hidden,taps,dtypes", [(256, 2, (Q4_K, Q6_K)), (768, 3, (Q6_K, Q4_K)), (2048, 4, (Q4_K, Q4_K)),
                                                (512, 5, (Q6_K, Q6_K))])
def test_conv_steps(gpu_ctx, oracle, hidden, taps, dtypes):
    w = synth.conv_weights(31 + taps, hidden=hidden, l_cache=taps, in_dtype=dtypes[0], out_dtype=dtypes[1])
    op = ConvOp(gpu_ctx, w)
    state = op.new_state()
    for i in range(taps + 2):
        x = synth.hidden_states(40 + i, 1, hidden=hidden).reshape(-1)
        want, new = oracle.conv_forward(w, state, x, 1)
        assert_bits(op.forward(state, x, 1, np.empty(hidden, np.float32)), want, f"conv step {i}")
        assert_bits(state, new, f"conv state {i}")
    op.close()


@pytest.mark.parametrize("hidden,heads,kv_heads,dtypes", [
    (256, 4, 1, (Q4_K, Q6_K, Q4_K, Q6_K)), (1024, 20, 4, (Q6_K, Q4_K, Q6_K, Q4_K)), (2048, 32, 8, (Q4_K,) * 4)])
def test_attention_steps(gpu_ctx, oracle, hidden, heads, kv_heads, dtypes):
    w = synth.attn_weights(heads, hidden=hidden, n_heads=heads, n_kv_heads=kv_heads, head_dim=64, dtypes=dtypes)
    op = AttnOp(gpu_ctx, w)
    kv, okv = op.new_cache(8), oracle.KvCache(w.kv_dim, 8)
    for i in range(4):
        x = synth.hidden_states(60 + i, 1, hidden=hidden).reshape(-1)
        want = oracle.attn_forward(w, okv, i, x, 1)
        assert_bits(op.forward(kv, i, x, 1, np.empty(hidden, np.float32)), want, f"attention step {i}")
    kv.close()
    op.close()


def test_stack_orders(gpu_ctx, oracle):
    def dense(i, dt):
        return synth.dense_weights(70, i, hidden=512, ff=768, dtype=dt)

    def moe(i, dt):
        return synth.moe_weights(70, i, hidden=512, moe_ff=256, n_experts=8, n_used=2, down_dtype=dt)

    gain = [(1 + 0.1 * synth.hidden_states(71, 1, hidden=512, stream=i)).astype(np.float32).reshape(-1) for i in range(6)]
    for order in ("d", "dd", "dm", "md", "mdmdd", "ddmmdm"):
        spec = [(gain[i], (dense if k == "d" else moe)(i, Q4_K if i % 2 else Q6_K)) for i, k in enumerate(order)]
        layers = [(g, (DenseLayer if isinstance(w, synth.DenseWeights) else MoeLayer)(gpu_ctx, w)) for g, w in spec]
        stack = FfnStack(gpu_ctx, layers)
        x = synth.hidden_states(72, 1, hidden=512).reshape(-1)
        before = x.copy()
        assert_bits(stack.run_layers(x), oracle.ffn_stack(spec, x, 1), f"stack {order}")
        assert_bits(x, before, "the input")
        stack.close()
        for _, layer in layers:
            layer.close()


@pytest.mark.parametrize("kind", ["dense", "moe"])
@pytest.mark.parametrize("t,shift", [(1, 4), (5, 512), (5, -512), (3, 0)])
def test_stack_of_one_layer_in_overlapping_rows(gpu_ctx, oracle, kind, t, shift):
    # the output may lie over the input, at another place too (device pointers, shift floats apart)
    import torch

    h = 512
    w = (synth.dense_weights(73, hidden=h, ff=768) if kind == "dense" else
         synth.moe_weights(73, hidden=h, moe_ff=256, n_experts=8, n_used=2))
    gain = np.ones(h, np.float32)
    layer = (DenseLayer if kind == "dense" else MoeLayer)(gpu_ctx, w)
    stack = FfnStack(gpu_ctx, [(gain, layer)])
    x = synth.hidden_states(74, t, hidden=h).reshape(-1)
    buf = torch.zeros(1024 + t * h, device="cuda")
    at = 512
    xv, ov = buf[at:at + t * h], buf[at + shift:at + shift + t * h]
    xv.copy_(torch.from_numpy(x))
    torch.cuda.synchronize()
    stack.forward(xv, t, ov)
    gpu_ctx.synchronize()
    assert_bits(ov.cpu().numpy(), oracle.ffn_stack([(gain, w)], x, t), f"{kind} t={t} shift {shift}")
    stack.close()
    layer.close()
