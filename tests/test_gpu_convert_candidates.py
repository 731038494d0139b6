"""The converter's shortcut over the candidate scales, byte for byte against the oracle (needs an MI355X).

Data on which the shortcut could go wrong: scales at both ends of the range it serves,
integers and codebook values (elements exactly on midpoints), elements that change
their entry exactly at a candidate, equal magnitudes, sparse and heavy-tailed blocks,
blocks outside the range, NaN and infinities.
The sizes are the smallest calls, a partly filled wave and both sides of the launch
rule (768 workgroups of 256 blocks).
"""
import numpy as np
import pytest

import oracle as O
import qe_moe

pytestmark = pytest.mark.gpu
KV = np.array([-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113], np.float64)
MID = (KV[1:] + KV[:-1]) / 2


def blocks(rng, n):
    m = n // 10 + 1
    z = lambda: rng.standard_normal((m, 32))  # noqa: E731
    p = [z() * 10.0 ** rng.uniform(-8, 6, (m, 1)),                          # across both ends of [1e-6, 1e4]
         z() * 10.0 ** rng.uniform(-6.3, -5.7, (m, 1)),
         rng.integers(-127, 128, (m, 32)) * 2.0 ** rng.integers(-12, 3, (m, 1)),
         rng.integers(-5, 6, (m, 32)) * rng.uniform(0.001, 1, (m, 1)),
         rng.choice(np.concatenate([MID, KV]), (m, 32)) * rng.uniform(-0.1, 0.1, (m, 1)),
         rng.standard_t(1.5, (m, 32)) * 0.02,
         np.sign(z()) * rng.uniform(0.1, 2, (m, 1)),
         z() * (rng.random((m, 32)) < 0.2)]
    b = z()
    b[:, 1:] *= rng.uniform(0.02, 0.12, (m, 1))                             # one large element
    p.append(b)
    top = rng.uniform(0.01, 1, (m, 1))
    b = -rng.choice(MID, (m, 32)) * top / rng.integers(120, 135, (m, 32))   # on a midpoint at a candidate
    b = np.where(np.abs(b) <= top, b, 0.0)
    b[:, 0] = top[:, 0]
    p.append(b)
    x = np.concatenate(p).astype(np.float32)
    return x[rng.permutation(len(x))[:n]]


def convert(torch, src, src_type, rows):
    dev = torch.from_numpy(np.ascontiguousarray(src).view(np.uint8).reshape(-1).copy()).cuda()
    out = torch.full((rows * O.nl4_row_bytes(256),), 0xEE, dtype=torch.uint8, device="cuda")
    qe_moe.nl4_quantize_rows(dev, src_type, rows, 256, out)
    torch.cuda.synchronize()
    return out.cpu().numpy().reshape(rows, -1)


@pytest.mark.parametrize("src_type", [O.SRC_F32, O.SRC_F16, O.SRC_BF16, O.SRC_Q8_0])
@pytest.mark.parametrize("rows", [1, 37, 24576, 24577])
def test_candidates_byte_exact(torch_cuda, src_type, rows):
    torch = torch_cuda
    print(f"converter candidates: type {src_type}, {rows} x 256", flush=True)
    rng = np.random.default_rng(rows + src_type)
    x = blocks(rng, rows * 8)
    if src_type == O.SRC_F32:
        src = x
    elif src_type == O.SRC_F16:
        src = np.clip(x, -60000, 60000).astype(np.float16)
    elif src_type == O.SRC_BF16:
        src = (x.view(np.uint32) >> 16).astype(np.uint16)
    else:
        d = np.abs(rng.standard_normal(len(x)) * 0.01).astype(np.float16)
        q = rng.integers(-128, 128, (len(x), 32)).astype(np.int8)
        q[::3] = rng.integers(-9, 10, q[::3].shape)
        src = np.concatenate([d.view(np.uint8).reshape(-1, 2), q.view(np.uint8)], axis=1)
    want = O.nl4_quantize_rows(np.ascontiguousarray(src), src_type, rows, 256)
    assert np.array_equal(convert(torch, src, src_type, rows), want)


# blocks out of the shortcut's range keep all fifteen candidates: in all lanes of a wave, in
# about as many as decide between the two ways of evaluating them (48 of 64), or in half;
# 37 rows end in a wave of 40 blocks
@pytest.mark.parametrize("rows", [37, 24577])
@pytest.mark.parametrize("scale,share", [(3e-8, 1.0), (2e-7, 1.0), (1e5, 1.0), (1e-7, 0.75), (1e5, 0.74), (1e-7, 0.5)])
def test_blocks_out_of_range(torch_cuda, scale, share, rows):
    print(f"converter out of range: {scale}, {share} of the blocks, {rows} x 256", flush=True)
    rng = np.random.default_rng(rows)
    n = rows * 8
    x = rng.standard_normal((n, 32)) * np.where(rng.random((n, 1)) < share, scale, 0.02)
    x = x.astype(np.float32)
    want = O.nl4_quantize_rows(x, O.SRC_F32, rows, 256)
    assert np.array_equal(convert(torch_cuda, x, O.SRC_F32, rows), want)


def test_smallest_change_beside_the_largest_sum(torch_cuda):
    """31 elements (or 24 to 30) of the largest magnitude, and a few that change their entry
    at the smallest midpoint, -4.5, at one of the candidates or an ulp or two beside it: the
    change is 1e-7 of the sum, and which side of it wins is a matter of roundings."""
    rows = 513
    print(f"converter smallest change, {rows} x 256", flush=True)
    rng = np.random.default_rng(5)
    n = rows * 8
    m = (rng.uniform(0.5, 1, (n, 1)) * 10.0 ** rng.uniform(-5, 3, (n, 1))).astype(np.float32)
    x = np.repeat(m, 32, axis=1)
    k = rng.choice([1, 1, 2, 4, 8], n)
    small = (4.5 * m.astype(np.float64) / rng.integers(119, 136, (n, 32))).astype(np.float32)
    small = (small.view(np.int32) + rng.integers(-2, 3, (n, 32), dtype=np.int32)).view(np.float32)
    x = np.where(np.arange(32)[None, :] >= 32 - k[:, None], small, x)
    x *= rng.choice([-1, 1], (n, 1)).astype(np.float32)
    want = O.nl4_quantize_rows(x, O.SRC_F32, rows, 256)
    assert np.array_equal(convert(torch_cuda, x, O.SRC_F32, rows), want)


@pytest.mark.parametrize("rows", [37, 24577])
def test_nan_and_infinities(torch_cuda, rows):
    """A block with a NaN or an infinity has a NaN scale (its codes are not defined), and
    leaves its neighbours in the wave as they are."""
    print(f"converter NaN and infinities: {rows} x 256", flush=True)
    rng = np.random.default_rng(rows)
    n = rows * 8
    x = (rng.standard_normal((n, 32)) * 0.02).astype(np.float32)
    for step, first, value in ((5, 0, np.nan), (7, 1, np.inf), (11, 2, -np.inf)):
        at = np.arange(first, n, step)
        x[at, rng.integers(0, 32, at.size)] = value
    bad = ~np.isfinite(x).all(axis=1)
    with np.errstate(all="ignore"):
        want = O.nl4_quantize_rows(x, O.SRC_F32, rows, 256)
    got = convert(torch_cuda, x, O.SRC_F32, rows)
    codes = [r[:, :128].reshape(n, 16) for r in (got, want)]
    scales = [np.ascontiguousarray(r[:, 128:]).view(np.float16).reshape(n) for r in (got, want)]
    assert np.array_equal(codes[0][~bad], codes[1][~bad])
    assert np.array_equal(scales[0][~bad].view(np.uint16), scales[1][~bad].view(np.uint16))
    assert np.isnan(scales[1][bad]).all() and np.isnan(scales[0][bad]).all()
