"""The prefill router and shared gate/up tiles at the sizes where their plan changes (needs an MI355X).

Router logits are compared bit for bit with the oracle's canonical order on every
token; the shared expert's output, on a sample of tokens, to fp32 rounding.
"""
import numpy as np
import pytest

import oracle as O
import qe_moe

pytestmark = pytest.mark.gpu
SEED = 0x70C7E5


@pytest.fixture(scope="module")
def ctx(torch_cuda):
    m = qe_moe.MoE(n_layers=1, t_max=4161)
    yield m
    m.close()


def run(torch, ctx, x):
    T = x.shape[0]
    xd = torch.from_numpy(x).cuda()
    y = torch.empty_like(xd)
    ctx.forward_normed(0, xd, y, T)
    torch.cuda.synchronize()
    return ctx.logits(T), ctx.routing(T)["sd"]


# token tiles of 64 (router, large shared tiles) and 32 (small shared tiles); 32 K
# splits below 256 tokens, 16 below 1280 (the end of the fused launch), 8 below 4096
# (two K groups of the shared tiles), 4 from there
@pytest.mark.parametrize("T", [9, 32, 63, 65, 255, 256, 1279, 1280, 1345, 4095, 4096, 4161])
def test_tiles_at_plan_edges(ctx, torch_cuda, T):
    print(f"router and shared tiles, T={T}", flush=True)
    bias = O.gen_zipf_bias(SEED, 0, 1.0)
    L = O.SynthLayer(SEED, 0, bias=bias)
    ctx.synth_layer(0, SEED, bias)
    x = O.gen_x(SEED, T, T)
    lg, sd = run(torch_cuda, ctx, x)
    ref = O.router(x, L.router, L.bias)
    assert np.array_equal(lg.view(np.uint32), ref.view(np.uint32))
    pick = np.unique(np.concatenate([np.arange(0, T, max(1, T // 60)), [T - 1]]))
    ref_sd = O.shared(np.ascontiguousarray(x[pick]), L.sh_gu, L.sh_dn)
    # each product of the two fp16 halves is exact; the sums of 2048 and 512 terms
    # differ from the oracle's by a few fp32 roundings each (about 1e-6 in all)
    assert np.linalg.norm(sd[pick] - ref_sd) <= 1e-5 * np.linalg.norm(ref_sd)


@pytest.mark.parametrize("t_max,T", [(224, 223), (256, 255), (1280, 1279), (4096, 4095)])
def test_call_that_needs_more_than_the_largest(torch_cuda, t_max, T):
    """Contexts whose last call but one writes more items or router partials than the last
    (the sizes themselves: test_plan_sizes.py)."""
    print(f"t_max={t_max}, T={T}", flush=True)
    L = O.SynthLayer(SEED, 0, bias=None)
    m = qe_moe.MoE(n_layers=1, t_max=t_max)
    try:
        m.synth_layer(0, SEED, None)
        for n in (T, t_max):
            x = O.gen_x(SEED, 3000 + n, n)
            lg, _ = run(torch_cuda, m, x)
            ref = O.router(x, L.router, None)
            assert np.array_equal(lg.view(np.uint32), ref.view(np.uint32))
            m.check()
    finally:
        m.close()


def q8_rows(raw, cols):
    raw = np.ascontiguousarray(raw).view(np.uint8).reshape(-1, cols + cols // 16)
    scale = np.ascontiguousarray(raw[:, cols:]).view(np.float16).astype(np.float64)
    return (raw[:, :cols].view(np.int8).reshape(len(raw), -1, 32) * scale[:, :, None]).reshape(len(raw), cols)


@pytest.mark.parametrize("T", [100, 1279, 1280, 1999, 2047])
def test_shared_error_against_64_bits(ctx, torch_cuda, T):
    """Below 2048 tokens no sum of the shared gate/up is a chain of more than 16 blocks.
    The output's relative 2-norm from 64 bits is 1.88e-7 with chains of 8 blocks, 1.98e-7
    with 16 and 2.22e-7 with 32, each within 1 % over seeds and sizes; the bound lies
    between the last two."""
    print(f"shared expert against 64 bits, T={T}", flush=True)
    L = O.SynthLayer(SEED, 0, bias=None)
    ctx.synth_layer(0, SEED, None)
    x = O.gen_x(SEED, 2000 + T, T)
    _, sd = run(torch_cuda, ctx, x)
    gu, dn = q8_rows(L.sh_gu, 2048), q8_rows(L.sh_dn, 512)
    g, u = np.split(x.astype(np.float64) @ gu.T, 2, axis=1)
    ref = (g / (1.0 + np.exp(-g)) * u) @ dn.T
    err = np.linalg.norm(sd - ref) / np.linalg.norm(ref)
    print(f"  {err:.3e}", flush=True)
    assert err <= 2.1e-7


@pytest.mark.parametrize("T", [70, 300, 1300, 4100])
def test_router_extreme_rows(ctx, torch_cuda, T):
    """Rows whose products and sums are subnormal, overflow, or hold infinities and
    NaN: the matrix cores' chain rounds as the scalar one does.  (Which NaN comes
    out is not defined, so only its place is compared.)"""
    print(f"router on extreme rows, T={T}", flush=True)
    L = O.SynthLayer(SEED, 0, bias=None)
    ctx.synth_layer(0, SEED, None)
    x = O.gen_x(SEED, 1000 + T, T)
    x[0] *= np.float32(1e-38)
    x[1] *= np.float32(3e-37)
    x[2] *= np.float32(1e37)
    x[3, ::3] = -0.0
    x[4] = 0.0
    x[T - 1] *= np.float32(1e-42)
    x[5, 7] = np.inf
    x[6, 100] = -np.inf
    x[T - 2, 2047] = np.nan
    with np.errstate(all="ignore"):
        lg, _ = run(torch_cuda, ctx, x)
        ref = O.router(x, L.router, None)
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(lg), nan)
    assert np.array_equal(lg.view(np.uint32)[~nan], ref.view(np.uint32)[~nan])
