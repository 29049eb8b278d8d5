"""The f16 expert products of K-quant swiglu layers (moe_f16.hip) at the sizes
where they can go wrong: every weight type on either side, one and several
chunks of hidden and ffn, chunks of one to 32 pairs, a shared expert of another
width, batches on both sides of each launch shape, and a layer just past what
they take (ffn 768: the bf16 pipelines).  Bound of the outputs: the parity
bound of the layer (check_layer); a token's bits are the same in every batch of
two or more tokens."""
import dataclasses

import numpy as np
import pytest

from llambda_amd import ggml, synthetic
from llambda_amd.moe import HipMoeSession, synthetic_qwen3next

from test_moe_gpu import check_layer

pytestmark = pytest.mark.gpu

Q4, Q6 = ggml.Q4_K, ggml.Q6_K


@pytest.mark.parametrize("up,down,hidden,experts,top_k,ffn,shared,tokens", [
    (Q4, Q6, 256, 4, 1, 256, 0, 2), (Q6, Q4, 512, 6, 2, 512, 256, 17),
    (Q4, Q4, 768, 16, 3, 256, 512, 33), (Q6, Q6, 2304, 8, 2, 256, 256, 9),
    (Q4, Q6, 256, 4, 2, 512, 512, 130), (Q4, Q6, 512, 64, 4, 512, 512, 48),
    (Q4, Q6, 512, 8, 2, 768, 256, 20),
    # all of hidden staged at once (few workgroups): 4, 5 and 8 chunks, the last
    # two against the bits of a batch that stages chunk by chunk
    (Q6, Q6, 1024, 8, 2, 256, 256, 3), (Q4, Q4, 2048, 8, 2, 256, 0, 2),
    (Q6, Q4, 1280, 64, 4, 512, 0, 48), (Q4, Q6, 2048, 64, 4, 512, 512, 48)])
def test_layers(hip, up, down, hidden, experts, top_k, ffn, shared, tokens):
    rng = np.random.default_rng(hidden + tokens)
    layer = synthetic_qwen3next(rng, hidden=hidden, experts=experts, top_k=top_k, ffn=ffn,
                                shared_ffn=shared, gate_type=up, down_type=down)
    x = synthetic.activations(rng, tokens, hidden)
    y, _ = check_layer(layer, x, f"{ggml.NAMES[up]}/{ggml.NAMES[down]} {hidden}x{ffn} T={tokens}")
    session = HipMoeSession(layer)
    try:
        np.testing.assert_array_equal(session.run(x[:2]), y[:2])
        first = (tokens - 2) // 2  # at least two tokens: one alone runs another pipeline
        np.testing.assert_array_equal(session.run(x[first:]), y[first:])
    finally:
        session.close()


def test_tokens_of_every_magnitude(hip):
    """Tokens 2^40 apart in one batch: each is held to its own bound (a linear
    router keeps its experts; silu saturates), a zero token gives zeros, and a
    NaN token leaves its neighbours' bits alone."""
    rng = np.random.default_rng(3)
    layer = synthetic_qwen3next(rng, hidden=512, experts=16, top_k=2, ffn=256, shared_ffn=256)
    x = synthetic.activations(rng, 12, 512)
    x[1] *= np.float32(2.0 ** -20)
    x[2] *= np.float32(2.0 ** 20)
    x[3, ::2] *= np.float32(2.0 ** -14)
    x[4] = 0.0
    y, _ = check_layer(layer, x, "magnitudes")
    assert not y[4].any()
    bad = x.copy()
    bad[6, 5] = np.nan
    session = HipMoeSession(layer)
    try:
        import torch
        xd = torch.from_numpy(bad).cuda()
        yd = torch.zeros_like(xd)
        torch.cuda.synchronize()
        session.run_device(xd.data_ptr(), yd.data_ptr(), 12)
        torch.cuda.synchronize()
        keep = [t for t in range(12) if t != 6]
        np.testing.assert_array_equal(yd.cpu().numpy()[keep], y[keep])
    finally:
        session.close()


def test_shared_expert_of_another_type(hip):
    """Types that differ between routed and shared rows keep the other pipelines."""
    rng = np.random.default_rng(4)
    layer = synthetic_qwen3next(rng, hidden=256, experts=8, top_k=2, ffn=256, shared_ffn=256)
    layer = dataclasses.replace(layer, shared_down=(Q4, synthetic.packed(Q4, rng, 256, 256)))
    check_layer(layer, synthetic.activations(rng, 11, 256), "shared down of another type")
