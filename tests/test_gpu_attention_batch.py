"""GPU parity of the attention operator's batched path (batches of 8 tokens and more: scores and P·V
on f32 MFMA, 16-item tiles, the softmax of each row in registers) against the CPU restatement of
attn_batch (model.rs:222-259), bit for bit: group sizes G = heads per kv head that divide a tile of
16 items and that do not, batches whose last tile is partly empty, histories that end at every place
of a 16-position piece and a 64-position chunk, rows of every size of softmax block, and a batch
large enough for the two-position P·V form. Every f32 operation is the reference's, in its order.
"""
import ctypes

import numpy as np
import pytest

from bebelm_amd import kernels as K
from bebelm_amd import synth
from bebelm_amd.model import AttnOp

from test_gpu_parity import assert_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv_heads,steps", [
    (4, 4, (8, 9, 23, 1, 15)),          # G = 1: 16 tokens a tile
    (8, 4, (17, 8, 31)),
    (12, 4, (11, 20, 64)),              # G = 3: 5 tokens, 15 items a tile
    (20, 4, (13, 8)),                   # G = 5: 3 tokens a tile
    (16, 1, (8, 30, 2, 9)),             # G = 16: one token a tile
    (32, 8, (512, 33)),                 # 2048 waves: two positions an MFMA in P·V
    (4, 1, (1000, 30, 1100, 40)),       # rows past 1024 and 2048 positions
    (4, 2, (4090, 16, 4100, 9)),        # ... 4096 and 8192
])
def test_attention_batches(gpu_ctx, oracle, heads, kv_heads, steps):
    w = synth.attn_weights(heads * 100 + kv_heads, hidden=256, n_heads=heads, n_kv_heads=kv_heads, head_dim=64)
    op, cap = AttnOp(gpu_ctx, w), sum(steps)
    kv, okv, pos = op.new_cache(cap), oracle.KvCache(w.kv_dim, cap), 0
    for t in steps:
        x = synth.hidden_states(pos + t, t, hidden=256).reshape(-1)
        want = oracle.attn_forward(w, okv, pos, x, t)
        got = op.forward(kv, pos, x, t, np.empty(t * 256, np.float32))
        assert_bits(got, want, f"attention {heads}/{kv_heads} t={t} at {pos}")
        pos += t
    kv.close()
    op.close()


def identity_op():
    """Attention weights of F32 identities: q, k and v are columns of the input row, the output row the
    attention itself, so its bits are seen as they are."""
    eye = np.eye(512, dtype=np.float32)
    ones = np.ones(64, np.float32)
    return synth.AttnWeights(512, 8, 2, 64, 0, 0, 0, 0, eye.reshape(-1), eye[128:256].reshape(-1),
                             eye[256:384].reshape(-1), eye.reshape(-1), ones, ones)


@pytest.mark.parametrize("scale", [1.0, 1e-36, 2e-38, 3e-40, 1e-44])
def test_attention_of_subnormal_values(gpu_ctx, oracle, scale):
    # the MFMA's products round as fmaf's do and the sums as the adds do where they are subnormal or zero:
    # values (columns 256..383 of x) of every size down to the smallest subnormal
    w = identity_op()
    op = AttnOp(gpu_ctx, w)
    kv, okv, pos = op.new_cache(80), oracle.KvCache(w.kv_dim, 80), 0
    for t in (33, 16, 31):
        x = synth.hidden_states(pos + t, t, hidden=512).astype(np.float32)
        x[:, 256:384] *= np.float32(scale)
        x[1, 256:384] = 0.0
        want = oracle.attn_forward(w, okv, pos, x.reshape(-1), t)
        assert scale > 1e-37 or np.any((want != 0) & (np.abs(want) < 1.1e-38))
        got = op.forward(kv, pos, x.reshape(-1), t, np.empty(t * 512, np.float32))
        assert_bits(got, want, f"values of {scale}, t={t} at {pos}")
        pos += t
    kv.close()
    op.close()


@pytest.mark.parametrize("n", [900, 1025, 3000, 8000, 16384])
def test_softmax_rows_that_need_the_chain(gpu_ctx, oracle, n):
    # scores of two values, as many of each as leaves the sum of exps so near a rounding boundary of
    # (float)(1 / sum) that the interval test cannot settle it: the block then runs the reference's
    # chain of adds
    expf = ctypes.CDLL("libm.so.6").expf
    expf.restype, expf.argtypes = ctypes.c_float, [ctypes.c_float]

    a = np.arange(1, n)
    for low in np.linspace(-3, -0.1, 4000, dtype=np.float32):
        s = a + (n - a) * float(expf(float(low)))
        b = (n + 64) * 2.0 ** -51 * s
        found = a[(1.0 / (s - b)).astype(np.float32) != (1.0 / (s + b)).astype(np.float32)]
        if len(found):
            break
    ones = found[0]
    g = np.random.default_rng(n)
    k = np.zeros((n, 64), np.float32)
    k[g.permutation(n)[ones:], 0] = low      # score = 8·k[0] / sqrt(64)
    q = np.zeros(64, np.float32)
    q[0] = 8.0
    v = g.standard_normal(n * 64).astype(np.float32)
    out = np.zeros(64, np.float32)
    K.attention_decode(gpu_ctx, q, k.reshape(-1), v, n, 1, 1, 64, out)
    assert_bits(out, oracle.attention_decode(q, k.reshape(-1), v, n, 1, 1, 64), f"softmax chain n={n}")
