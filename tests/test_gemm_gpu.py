"""Multi-token projections (gemm.hip) against 64-bit products of the oracle's
dequantised weights.

Bounds.  Every output's error is at most 2^-20 of its sum of |terms|: the
activations carry 2^-23 relative error, and the longest run of fp32 adds into
one sum is 8 chunks x (about 40 roundings in a chunk) with partial sums below
the sum of |terms|, whose roundings add up at random (sqrt(320) 2^-24 < 2^-19,
and the partial sums average half of the bound).  A Q4_K term counts as
three products, sc (q - 8) d, 8 sc d and m dmin, more than the two it is formed
from (test_one_large_activation takes these two).  The 2-norm
error of N(0, 1) activations stays below 3e-7 (an fp32 evaluation: 1.2e-7 to
2.4e-7).
"""
import numpy as np
import pytest

import oracle
from llambda_amd import ggml, synthetic
from llambda_amd.hip_backend import make_hip_session_packed

pytestmark = pytest.mark.gpu

TYPES = [ggml.Q4_K, ggml.Q6_K, ggml.Q5_0, ggml.Q8_0]


def _weights(type_tag, w, rows, columns):
    if type_tag == ggml.F32:
        return w.view(np.float32).reshape(rows, columns).astype(np.float64)
    return oracle.dequantize(type_tag, w, rows * columns).reshape(rows, columns).astype(np.float64)


def _terms(type_tag, w, wd, rows, columns):
    """|weight| per element as the kernel forms it."""
    if type_tag != ggml.Q4_K:
        return np.abs(wd)
    b = w.reshape(-1, 144)
    d = b[:, 0:2].copy().view(np.float16).astype(np.float64)
    m = b[:, 2:4].copy().view(np.float16).astype(np.float64)
    return np.abs(wd) + np.repeat(np.abs(d) * 63 * 16 + np.abs(m) * 63, 256, axis=1).reshape(rows, columns)


def _run(s, x):
    y = np.empty((x.shape[0], s.output_element_count), dtype=np.float32)
    return s.run_batch_into(y, x, x.shape[0])


def _check(type_tag, w, rows, columns, x, y, label, norm=True):
    wd = _weights(type_tag, w, rows, columns)
    ref = x.astype(np.float64) @ wd.T
    bound = 2.0 ** -20 * (np.abs(x.astype(np.float64)) @ _terms(type_tag, w, wd, rows, columns).T)
    err = np.abs(y - ref)
    assert np.all(err <= bound), (label, float((err / bound).max()))
    if norm:
        rel = np.linalg.norm(y - ref) / np.linalg.norm(ref)
        assert rel < 3e-7, (label, rel)


# rows, columns (K-quants; block types), tokens: one row and one chunk, ragged
# rows and tokens on both sides of every tile (16 x 16 to 256 x 64), one to
# several chunks per wave group, more than eight chunks in one run of totals,
# a last chunk of one 32-block, and grids that each tile shape serves
SHAPES = [
    (1, 256, 32, 2), (17, 512, 288, 3), (515, 2048, 1056, 16), (515, 2304, 1856, 17),
    (1024, 2560, 2688, 33), (4096, 256, 544, 31), (4000, 768, 480, 65), (14000, 512, 96, 7),
    (14000, 512, 320, 63), (14000, 256, 256, 130), (14300, 256, 224, 200), (1000, 5120, 4640, 300),
    (70, 32768, 32736, 20),  # the widest rows
]


@pytest.mark.parametrize("type_tag", TYPES)
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_matches_64_bit_products(hip, type_tag, shape):
    rows, wide, narrow, tokens = shape
    columns = wide if type_tag in (ggml.Q4_K, ggml.Q6_K) else narrow
    rng = np.random.default_rng(rows + tokens)
    w = synthetic.packed(type_tag, rng, rows, columns)
    x = synthetic.activations(rng, tokens, columns)
    s = make_hip_session_packed(w, type_tag, rows, columns)
    try:
        y = _run(s, x)
    finally:
        s.close()
    _check(type_tag, w, rows, columns, x, y, f"{ggml.NAMES[type_tag]} {shape}")


@pytest.mark.parametrize("type_tag", TYPES)
def test_extreme_activations_and_scales(hip, type_tag):
    """Tokens of every magnitude beside each other, each exact to its own; an
    infinity or a NaN stays in its token, and finite outputs that an infinity
    reaches with a nonzero weight are infinite or NaN, never finite."""
    rows, columns = 160, 1280
    rng = np.random.default_rng(5)
    w = synthetic.packed(type_tag, rng, rows, columns)
    bb = ggml.block_bytes(type_tag)
    blocks = w.reshape(-1, bb)
    at = 208 if type_tag == ggml.Q6_K else 0
    scales = np.array([2000.0, 256.0, -300.0, 6e-8, 0.0, 1e-5], dtype=np.float16)
    blocks[:, at:at + 2] = rng.choice(scales, size=blocks.shape[0]).view(np.uint8).reshape(-1, 2)
    x = synthetic.activations(rng, 23, columns)
    for t, f in enumerate((1e-33, 1e-30, 1e28, 1e-20, 1e20, 0.0)):
        x[t] = (x[t] * np.float32(f)).astype(np.float32)
    x[7, ::3] *= np.float32(2.0 ** -12)
    x[8, 5], x[9, 300], x[10, 700] = np.inf, -np.inf, np.nan
    s = make_hip_session_packed(w, type_tag, rows, columns)
    try:
        with np.errstate(all="ignore"):
            for first in (0, 3):  # both sides of the 16-token tiles
                y = _run(s, np.ascontiguousarray(x[first:]))
                fine = [t for t in range(first, 23) if t not in (8, 9, 10)]
                _check(type_tag, w, rows, columns, x[fine], y[[t - first for t in fine]],
                       f"extremes {ggml.NAMES[type_tag]}", norm=False)
                wd = _weights(type_tag, w, rows, columns)
                for t, k in ((8, 5), (9, 300), (10, 700)):
                    reached = wd[:, k] != 0 if t < 10 else slice(None)
                    assert not np.isfinite(y[t - first][reached]).any(), t
                for t, k in ((8, 5), (9, 300)):
                    if type_tag == ggml.Q4_K:  # its offset products may meet as inf - inf
                        continue
                    alone = (wd[:, k] != 0) & ~np.isnan(y[t - first])
                    assert np.array_equal(np.sign(y[t - first][alone]), np.sign(x[t, k] * wd[alone, k]))
    finally:
        s.close()


@pytest.mark.parametrize("type_tag", [ggml.Q5_0, ggml.Q8_0], ids=["Q5_0", "Q8_0"])
@pytest.mark.parametrize("shape", [(40, 480, 3), (515, 1056, 16), (4000, 480, 65), (14000, 320, 63),
                                   (14300, 256, 200), (14300, 2336, 200)],
                         ids=lambda s: "x".join(map(str, s)))
def test_large_scales_leave_small_ones_exact(hip, type_tag, shape):
    """Scales of 256 and more beside scales of 1e-5 to 1e-3: in another row of
    the tile, and in another block of the same row where the large block's
    weights are zero.  Each row is held to its own bound."""
    rows, columns, tokens = shape
    rng = np.random.default_rng(rows)
    w = synthetic.packed(type_tag, rng, rows, columns)
    blocks = w.reshape(rows, columns // 32, ggml.block_bytes(type_tag))
    small = rng.choice(np.array([1e-3, 1e-4, -1e-5, 5e-6], dtype=np.float16), size=blocks.shape[:2])
    blocks[:, :, 0:2] = small.view(np.uint8).reshape(*blocks.shape[:2], 2)
    large = np.array([256.0, -2000.0, 65504.0], dtype=np.float16).view(np.uint8).reshape(3, 2)
    zero = np.zeros(ggml.block_bytes(type_tag) - 2, dtype=np.uint8)
    if type_tag == ggml.Q5_0:
        zero[:4] = 0xFF  # fifth bits: code 16 is weight 0
    for i, at in enumerate(range(0, rows, 16)):  # one row of each tile: one zero block of a large scale
        r, b = at + i % min(16, rows - at), i % blocks.shape[1]
        blocks[r, b, 0:2], blocks[r, b, 2:] = large[i % 3], zero
        if i % 2:  # and every other tile a row of large scales among its own small ones
            r = at + (i + 7) % min(16, rows - at)
            blocks[r, ::3, 0:2] = large[i % 3]
    x = synthetic.activations(rng, tokens, columns)
    s = make_hip_session_packed(w, type_tag, rows, columns)
    try:
        y = _run(s, x)
    finally:
        s.close()
    _check(type_tag, w, rows, columns, x, y, f"{ggml.NAMES[type_tag]} {shape}", norm=False)


@pytest.mark.parametrize("shape", [(40, 512, 3), (515, 2048, 16), (4000, 768, 65), (1024, 2560, 33),
                                   (14300, 256, 200)], ids=lambda s: "x".join(map(str, s)))
def test_one_large_activation(hip, shape):
    """An activation 2^22 times the others leaves its hold on the rows where its
    Q4_K weight is zero (code and minimum) at what the split of x loses beside
    it: 2^-39 of it per activation of its 256, whose lo parts are f16 subnormals
    then.  Otherwise each row is held to 2^-20 of the products it is formed
    from, sc q d and m dmin."""
    rows, columns, tokens = shape
    rng = np.random.default_rng(rows)
    w = synthetic.packed(ggml.Q4_K, rng, rows, columns)
    b = w.reshape(rows, columns // 256, 144)
    at = 256 * (columns // 256 // 2) + 100  # sub-block 3 of a chunk: high nibbles of qs[32:64]
    zeroed = b[::2, at // 256]
    zeroed[:, 11] &= 0xC0  # its minimum
    zeroed[:, 52] &= 0x0F  # the element's code
    x = synthetic.activations(rng, tokens, columns)
    x[:, at] = np.float32(2.0 ** 22)
    s = make_hip_session_packed(w, ggml.Q4_K, rows, columns)
    try:
        y = _run(s, x)
    finally:
        s.close()
    wd = _weights(ggml.Q4_K, w, rows, columns)
    assert not wd[::2, at].any()
    m = np.concatenate([b[:, :, 8:12] & 63, (b[:, :, 12:16] >> 4) | (b[:, :, 8:12] >> 6 << 4)], axis=2)
    low = b[:, :, 2:4].copy().view(np.float16).astype(np.float64) * m
    low = np.repeat(np.abs(low), 32, axis=2).reshape(rows, columns)
    x = x.astype(np.float64)
    terms = np.abs(wd + low) + low
    chunk = slice(at // 256 * 256, at // 256 * 256 + 256)
    bound = 2.0 ** -20 * (np.abs(x) @ terms.T) + 2.0 ** (22 - 39) * terms[:, chunk].sum(axis=1)
    err = np.abs(y - x @ wd.T)
    assert np.all(err <= bound), float((err / bound).max())


@pytest.mark.parametrize("type_tag", TYPES)
def test_ordinary_scales_at_every_magnitude(hip, type_tag):
    """Tokens from 1e-36 to 1e34, scales of 1e-4 to 1e-3: neither 1 / s nor its
    product with a scale may reach the subnormals or overflow."""
    rows, columns = 160, 1280
    rng = np.random.default_rng(11)
    w = synthetic.packed(type_tag, rng, rows, columns)
    x = synthetic.activations(rng, 24, columns).astype(np.float64)
    x = (x * 10.0 ** np.linspace(-36, 34, 24)[:, None]).astype(np.float32)
    s = make_hip_session_packed(w, type_tag, rows, columns)
    try:
        for batch in (x, x[:9], x[9:]):  # both kernels
            _check(type_tag, w, rows, columns, batch, _run(s, np.ascontiguousarray(batch)),
                   ggml.NAMES[type_tag], norm=False)
    finally:
        s.close()


@pytest.mark.parametrize("shape", [(1, 4, 2), (33, 260, 16), (515, 1028, 17), (512, 2048, 33),
                                   (96, 4100, 130)], ids=lambda s: "x".join(map(str, s)))
def test_f32_rows(hip, shape):
    rows, columns, tokens = shape
    rng = np.random.default_rng(rows)
    w = synthetic.packed(ggml.F32, rng, rows, columns)
    x = synthetic.activations(rng, tokens, columns)
    s = make_hip_session_packed(w, ggml.F32, rows, columns)
    try:
        y = _run(s, x)
        again = _run(s, np.ascontiguousarray(x[:2]))
        first = _run(s, np.ascontiguousarray(x[:5]))
    finally:
        s.close()
    wd = w.view(np.float32).reshape(rows, columns).astype(np.float64)
    bound = 2.0 ** -20 * (np.abs(x.astype(np.float64)) @ np.abs(wd).T)
    assert np.all(np.abs(y - x.astype(np.float64) @ wd.T) <= bound)
    # one order of sums up to four tokens, one from five on
    assert np.all(np.abs(again - x[:2].astype(np.float64) @ wd.T) <= bound[:2])
    assert np.array_equal(*((first, y[:5]) if tokens > 4 else (again, y[:2])))


@pytest.mark.parametrize("shape", [(1, 4, 3), (33, 1028, 4), (515, 4100, 3), (512, 2048, 4), (7, 1020, 2)],
                         ids=lambda s: "x".join(map(str, s)))
def test_f32_rows_of_two_to_four_tokens(hip, shape):
    """The kernel of few tokens: tokens and rows short of a workgroup's, columns
    short of and past a turn of 1024; neighbours of y stay untouched."""
    import torch
    rows, columns, tokens = shape
    rng = np.random.default_rng(rows)
    w = synthetic.packed(ggml.F32, rng, rows, columns)
    x = synthetic.activations(rng, tokens, columns)
    xd = torch.from_numpy(x).cuda()
    yd = torch.full((tokens * rows + 6,), 7.0, device="cuda")
    torch.cuda.synchronize()
    s = make_hip_session_packed(w, ggml.F32, rows, columns)
    try:
        s.run_device(xd.data_ptr(), yd[3:].data_ptr(), tokens)
        torch.cuda.synchronize()
    finally:
        s.close()
    y = yd.cpu().numpy()
    assert np.all(y[:3] == 7.0) and np.all(y[-3:] == 7.0)
    _check(ggml.F32, w, rows, columns, x, y[3:-3].reshape(tokens, rows), shape)


@pytest.mark.parametrize("type_tag,rows,columns,tokens", [
    (ggml.Q8_0, 16, 32, 16 * 65535 + 20), (ggml.Q5_0, (1 << 20) + 40, 32, 3),
    (ggml.F32, (1 << 20) + 5, 4, 5), (ggml.F32, 7, 8, 16 * 65535 + 9)],
    ids=lambda v: str(v))
def test_more_rows_or_tokens_than_one_grid_takes(hip, type_tag, rows, columns, tokens):
    import torch
    rng = np.random.default_rng(9)
    w = synthetic.packed(type_tag, rng, rows, columns)
    x = synthetic.activations(rng, tokens, columns)
    wd = torch.from_numpy(_weights(type_tag, w, rows, columns)).cuda()
    xd = torch.from_numpy(x).cuda()
    yd = torch.full((tokens, rows), float("nan"), device="cuda")
    torch.cuda.synchronize()
    s = make_hip_session_packed(w, type_tag, rows, columns)
    try:
        s.run_device(xd.data_ptr(), yd.data_ptr(), tokens)
        torch.cuda.synchronize()
    finally:
        s.close()
    bound = 2.0 ** -20 * (xd.double().abs() @ wd.abs().T.contiguous())
    assert bool(((yd.double() - xd.double() @ wd.T.contiguous()).abs() <= bound).all())


def test_device_rows_on_any_float(hip):
    """x and y need float alignment only; neighbours of y stay untouched."""
    import torch
    rows, columns, tokens = 300, 768, 21
    rng = np.random.default_rng(6)
    for type_tag in TYPES + [ggml.F32]:
        w = synthetic.packed(type_tag, rng, rows, columns)
        x = synthetic.activations(rng, tokens, columns)
        s = make_hip_session_packed(w, type_tag, rows, columns)
        try:
            xd = torch.zeros(x.size + 3, device="cuda")
            xd[1:1 + x.size] = torch.from_numpy(x.reshape(-1)).cuda()
            yd = torch.full((tokens * rows + 6,), 7.0, device="cuda")
            torch.cuda.synchronize()
            s.run_device(xd[1:].data_ptr(), yd[3:].data_ptr(), tokens)
            torch.cuda.synchronize()
            y = yd.cpu().numpy()
            assert np.all(y[:3] == 7.0) and np.all(y[-3:] == 7.0)
            _check(type_tag, w, rows, columns, x, y[3:-3].reshape(tokens, rows), "offset rows")
        finally:
            s.close()


def test_replays_in_a_graph(hip):
    """A captured call replays with new activations, eager calls in between
    (no memory is allocated by the call)."""
    import torch
    rows, columns, tokens = 515, 1024, 40
    rng = np.random.default_rng(8)
    w = synthetic.packed(ggml.Q4_K, rng, rows, columns)
    s = make_hip_session_packed(w, ggml.Q4_K, rows, columns)
    try:
        xd = torch.zeros((tokens, columns), device="cuda")
        yd = torch.zeros((tokens, rows), device="cuda")
        ye = torch.zeros((tokens, rows), device="cuda")
        graph = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph):
            s.run_device(xd.data_ptr(), yd.data_ptr(), tokens,
                         torch.cuda.current_stream().cuda_stream)
        for _ in range(3):
            xd.copy_(torch.from_numpy(synthetic.activations(rng, tokens, columns)))
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            s.run_device(xd.data_ptr(), ye.data_ptr(), tokens)
            torch.cuda.synchronize()
            assert torch.equal(yd, ye)
    finally:
        s.close()
