"""GPU parity of the single operators against the C oracle (same seeded inputs).

Scaffold accumulators and the RMSNorm/quantizer outputs must be bit-exact; the conv + SSM
recurrence is compared after 128 steps with max|d| / max|ref| <= 1e-3 (fp32 state), the
tolerance that the whole decode's state is held to.
"""
import numpy as np
import pytest
import torch

from dfssm import ops
from dfssm.format import unpack_sign_bits
from oracle import oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _h(a):  # numpy fp16 -> torch fp16 on the GPU
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).to(DEV).view(torch.float16)


def _np16(t):
    return t.cpu().view(torch.int16).numpy().view(np.float16)


def _tiled(bits_np, N, K):
    return ops.tile_bits(torch.from_numpy(bits_np.view(np.int32)).to(DEV), N, K)


# N picks 16, 32 or 64 output rows per matrix-core workgroup (N <= 4096, <= 8192, above)
@pytest.mark.parametrize("N,K", [(8512, 2048), (2048, 4096), (10576, 2560), (2048, 5120), (2320, 512), (6144, 1024)])
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 16, 32, 64])
def test_scaffold_acc_bit_exact(N, K, M):
    """Config 1: in_proj 2048->8512, out_proj 4096->2048 (+2.7B and tiny shapes), int8 ~N(0,40)."""
    print(f"scaffold N={N} K={K} M={M}", flush=True)
    rng = np.random.default_rng([1, N, K, M])
    bits = rng.integers(0, 2 ** 32, (N, K // 32), dtype=np.uint32)
    q = np.clip(np.rint(rng.normal(0, 40, (M, K))), -127, 127).astype(np.int8)
    xs = rng.uniform(0.01, 0.05, M).astype(np.float16)
    ws = rng.uniform(0.01, 0.05, N).astype(np.float16)
    acc, y = ops.scaffold_gemm(_tiled(bits, N, K), torch.from_numpy(q).to(DEV), N, _h(xs), _h(ws), want_y=True)
    ref = O.scaffold_acc(bits, q)
    np.testing.assert_array_equal(acc.cpu().numpy(), ref)
    yref = O.dequant_lora(ref, xs, ws, np.zeros((M, 16), np.float16), np.zeros((N, 16), np.int8),
                          np.zeros(N, np.float16))
    np.testing.assert_array_equal(_np16(y).view(np.uint16), yref.view(np.uint16))


@pytest.mark.parametrize("M", [1, 4, 32])
def test_scaffold_extremes(M):
    """All +127 / all -128 activations against all-set / all-clear / random bits: +-K*127, etc."""
    N, K = 192, 2048
    rng = np.random.default_rng(7)
    bits = np.concatenate([np.full((64, K // 32), 0xFFFFFFFF, np.uint32), np.zeros((64, K // 32), np.uint32),
                           rng.integers(0, 2 ** 32, (64, K // 32), dtype=np.uint32)])
    q = np.where(np.arange(M)[:, None] % 2 == 0, 127, -128).astype(np.int8).repeat(K, axis=1).reshape(M, K)
    acc = ops.scaffold_gemm(_tiled(bits, N, K), torch.from_numpy(q).to(DEV), N).cpu().numpy()
    ref = q.astype(np.int64) @ unpack_sign_bits(bits).astype(np.int64).T
    np.testing.assert_array_equal(acc, ref)
    assert acc[0, 0] == 127 * K and acc[0, 64] == -127 * K


@pytest.mark.parametrize("K", [512, 2048, 4096, 5120])
@pytest.mark.parametrize("scale", [1.0, 1e-3, 300.0])
def test_rmsnorm_quantize_bit_exact(K, scale):
    M = 4
    rng = np.random.default_rng([2, K, int(scale * 1000)])
    x = (rng.normal(0, 1, (M, K)) * scale).astype(np.float16)
    x[1, :] = 0                      # all-zero row: amax clamps to 1e-4
    x[2, ::7] = np.float16(scale * 9)  # outliers
    w = (1 + rng.uniform(-0.1, 0.1, K)).astype(np.float32)
    xn, q, s = ops.rmsnorm_quantize(_h(x), torch.from_numpy(w).to(DEV))
    xn_ref = O.rmsnorm(x, w)
    q_ref, s_ref = O.quantize(xn_ref)
    np.testing.assert_array_equal(_np16(xn).view(np.uint16), xn_ref.view(np.uint16))
    np.testing.assert_array_equal(_np16(s).view(np.uint16), s_ref.view(np.uint16))
    np.testing.assert_array_equal(q.cpu().numpy(), q_ref)


@pytest.mark.parametrize("B", [1, 32])
def test_conv_ssm_128_steps(B):
    """Config 2: 64 heads x 64, d_state 128, conv channels 4352, 128 sequential steps."""
    H, P, N = 64, 64, 128
    DI = H * P
    C = DI + 2 * N
    steps = 128
    print(f"conv+ssm B={B}", flush=True)
    rng = np.random.default_rng([3, B])
    conv0 = rng.normal(0, 1, (B, C, 3)).astype(np.float16)
    conv_w = rng.normal(0, 0.5, (C, 4)).astype(np.float16)
    conv_b = rng.normal(0, 0.1, C).astype(np.float16)
    A_log = rng.uniform(0, np.log(16), H).astype(np.float32)
    Dp = np.ones(H, np.float32)
    dt_bias = np.zeros(H, np.float32)
    xbc_seq = rng.normal(0, 1, (steps, B, C)).astype(np.float16)
    dt_seq = rng.normal(-2, 1, (steps, B, H)).astype(np.float16)

    g_conv = _h(conv0)
    g_h = torch.zeros(B, H, P, N, dtype=torch.float32, device=DEV)
    g_y = torch.empty(B, DI, dtype=torch.float16, device=DEV)
    tw, tb = _h(conv_w), _h(conv_b)
    tA, tD, tdb = (torch.from_numpy(a).to(DEV) for a in (A_log, Dp, dt_bias))
    r_conv = conv0.copy()
    r_h = np.zeros((B, H, P, N), np.float32)
    ys = []
    for t in range(steps):
        gx = _h(xbc_seq[t])
        ops.conv_step(g_conv, gx, tw, tb)
        ops.ssm_step(g_h, gx, _h(dt_seq[t]), tdb, tA, tD, g_y)
        rx = xbc_seq[t].copy()
        O.conv_step(r_conv, rx, conv_w, conv_b)
        r_y = O.ssm_step(r_h, rx, dt_seq[t], dt_bias, A_log, Dp)
        if t in (0, steps - 1):
            ys.append((_np16(g_y).astype(np.float32), r_y.astype(np.float32)))
    gh = g_h.cpu().numpy()
    rel = np.abs(gh - r_h).max() / np.abs(r_h).max()
    print(f"B={B} state max rel err {rel:.3e}, bit-exact {np.array_equal(gh, r_h)}")
    assert rel <= 1e-3                      # the tolerance of the state
    # the state update uses only correctly rounded elementwise operations on identical inputs,
    # so it is in fact bit-exact
    np.testing.assert_array_equal(gh, r_h)
    np.testing.assert_array_equal(_np16(g_conv).view(np.uint16), r_conv.view(np.uint16))
    for gy, ry in ys:
        assert np.abs(gy - ry).max() <= 1e-3 * np.abs(ry).max() + 1e-3


@pytest.mark.parametrize("w3", [1.0, 37.0, 65504.0])
def test_silu_all_halves(w3):
    """SiLU of every fp16 value (times a conv weight: sums up to 4.3e9, infinities and NaN) against the
    oracle's formula, bit for bit: the clamped exponential and the reciprocal of the kernels."""
    x = np.arange(65536, dtype=np.uint16).view(np.float16).reshape(1, -1)
    C = x.shape[1]
    w = np.zeros((C, 4), np.float16)
    w[:, 3] = w3
    b = np.zeros(C, np.float16)
    st = np.zeros((1, C, 3), np.float16)
    print(f"silu of all halves times {w3}", flush=True)
    gx = _h(x)
    ops.conv_step(_h(st), gx, _h(w), _h(b))
    rx = x.copy()
    O.conv_step(st.copy(), rx, w, b)
    got = _np16(gx)
    nan = np.isnan(rx)
    np.testing.assert_array_equal(np.isnan(got), nan)
    np.testing.assert_array_equal(got.view(np.uint16)[~nan], rx.view(np.uint16)[~nan])


def _silu_inputs():
    """fp32 values o for the kernels' o sigmoid(o): every float within 2000 steps of the ends of its exponential's
    range; the floats within two steps of each point where o sigmoid(o) changes its fp16 rounding, on each of its
    three monotonic branches; and values spread over the logarithm of [2^-14, 104]."""
    ends = np.array([86.0, 87.0, 88.0, 88.72284, 89.0, 103.97], np.float32).view(np.int32)
    edge = (ends[:, None] + np.arange(-2000, 2001)[None]).astype(np.int32).view(np.float32).ravel()
    halves = np.arange(1, 31743, dtype=np.uint16).view(np.float16).astype(np.float64)
    mid = (halves[:-1] + halves[1:]) / 2
    bottom = -1.2784645427610738  # the minimum of o sigmoid(o), -0.27846
    points = []
    for lo, hi, v in ((0.0, 66000.0, mid), (bottom, 0.0, -mid[mid < 0.2784]), (-30.0, bottom, -mid[mid < 0.2784])):
        lo, hi = np.full_like(v, lo), np.full_like(v, hi)
        rising = hi[0] > bottom
        for _ in range(60):
            c = (lo + hi) / 2
            below = c / (1 + np.exp(-c)) < v
            lo, hi = np.where(below == rising, c, lo), np.where(below == rising, hi, c)
        points.append(lo[np.abs(lo) >= 2.0 ** -14])
    p = np.concatenate(points).astype(np.float32).view(np.int32)
    near = (p[:, None] + np.arange(-2, 3)[None]).astype(np.int32).view(np.float32).ravel()
    rng = np.random.default_rng(33)
    spread = np.exp(rng.uniform(np.log(2.0 ** -14), np.log(104.0), 400000)).astype(np.float32)
    return np.concatenate([edge, -edge, near, spread, -spread])


def test_silu_sweep():
    """SiLU at fp32 inputs, where the clamps and roundings of the kernels' sigmoid could show (the conv feeds it
    fp32 sums), against the oracle's formula, bit for bit. Each input is the exact sum of three taps: the
    bytes of its 24-bit integer times powers of two."""
    o = _silu_inputs()
    m, e = np.frexp(np.abs(o).astype(np.float64))
    m = (m * 2 ** 24).astype(np.int64)
    e = e - 24  # |o| = m 2^e
    taps, weights = [], []
    for sh in (16, 8, 0):
        t = e + sh
        k = np.clip(t, -24, 15)  # the weight's exponent; the rest goes to the byte
        taps.append(np.ldexp(((m >> sh) & 255).astype(np.float64) * np.sign(o), t - k).astype(np.float16))
        weights.append(np.ldexp(1.0, k).astype(np.float16))
    total = sum(a.astype(np.float64) * b.astype(np.float64) for a, b in zip(taps, weights))
    np.testing.assert_array_equal(total, o.astype(np.float64))
    C = o.size
    w = np.zeros((C, 4), np.float16)
    st = np.zeros((1, C, 3), np.float16)
    for i in range(2):
        st[0, :, 1 + i], w[:, 1 + i] = taps[i], weights[i]
    w[:, 3] = weights[2]
    x, b = taps[2].reshape(1, C), np.zeros(C, np.float16)
    print(f"silu at {C} fp32 inputs", flush=True)
    gx = _h(x)
    ops.conv_step(_h(st), gx, _h(w), _h(b))
    rx = np.ascontiguousarray(x)
    O.conv_step(st.copy(), rx, w, b)
    np.testing.assert_array_equal(_np16(gx).view(np.uint16), rx.view(np.uint16))


def _strided(a):
    """The same values as every second element of a larger tensor."""
    big = torch.zeros(*a.shape[:-1], 2 * a.shape[-1], dtype=a.dtype, device=a.device)
    big[..., ::2] = a
    return big[..., ::2]


def test_strided_arguments():
    """Several arguments that are not contiguous in one call: each operator's copies are all alive until its
    launch, so no copy takes another's memory."""
    rng = np.random.default_rng(31)
    N, K, M = 256, 512, 2
    packed = rng.integers(0, 1 << 32, (N, K // 32), dtype=np.uint32).view(np.int32)
    bits = ops.tile_bits(torch.from_numpy(packed).to(DEV), N, K)
    f = lambda *sh: _h(rng.uniform(0.5, 1.5, sh).astype(np.float16))
    i8 = lambda *sh: torch.from_numpy(rng.integers(-127, 128, sh, dtype=np.int8)).to(DEV)
    ws, q, xs, xn, lA, lAs, lBq = f(N), i8(M, K), f(M), f(M, K), i8(N, 16), f(N), f(16, K)
    print("strided scaffold", flush=True)
    ref = ops.scaffold_lora_gemm(bits, ws, q, xs, xn, lA, lAs, lBq, N)
    got = ops.scaffold_lora_gemm(bits, *map(_strided, (ws, q, xs, xn, lA, lAs, lBq)), N)
    for r, t in zip(ref, got):
        assert torch.equal(r, t)

    print("strided norm", flush=True)
    x, w = f(M, K), torch.from_numpy(rng.uniform(0.5, 1.5, K).astype(np.float32)).to(DEV)
    for r, t in zip(ops.rmsnorm_quantize(x, w), ops.rmsnorm_quantize(_strided(x), _strided(w))):
        assert torch.equal(r, t)

    print("strided conv", flush=True)
    C = 512
    cw, cb, st, xbc = f(C, 4), f(C), f(M, C, 3), f(M, C)
    st2, xbc2 = st.clone(), xbc.clone()
    ops.conv_step(st, xbc, cw, cb)
    ops.conv_step(st2, xbc2, _strided(cw), _strided(cb))
    assert torch.equal(st, st2) and torch.equal(xbc, xbc2)

    print("strided ssm", flush=True)
    H, P = 8, 16
    h = torch.from_numpy(rng.normal(0, 1, (M, H, P, 128)).astype(np.float32)).to(DEV)
    xbc, dt = f(M, H * P + 256), f(M, H)
    v = [torch.from_numpy(rng.uniform(0.1, 2.0, H).astype(np.float32)).to(DEV) for _ in range(3)]
    h2, y = h.clone(), torch.empty(M, H * P, dtype=torch.float16, device=DEV)
    y2 = torch.empty_like(y)
    ops.ssm_step(h, xbc, dt, *v, y)
    ops.ssm_step(h2, xbc, dt, *map(_strided, v), y2)
    assert torch.equal(h, h2) and torch.equal(y, y2)


def test_rmsnorm_quantize_transposed_input():
    """Rows that lie side by side in memory (a transposed tensor): the values of the row-major copy."""
    x = _h(np.random.default_rng(32).normal(0, 1, (512, 3)).astype(np.float16)).t()
    w = torch.ones(512, device=DEV)
    print("transposed norm", flush=True)
    for r, t in zip(ops.rmsnorm_quantize(x.contiguous(), w), ops.rmsnorm_quantize(x, w)):
        assert torch.equal(r, t)
