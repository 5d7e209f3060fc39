"""Prompt prefill (dfssm_prefill) against step-by-step ingestion and the oracle.

The layer-major prefill must give, bit for bit, what T decode steps give: the fp32 SSM state,
the conv state, the residual row handed to the next step, the greedy token and the logits of the
last prompt token. Covered: batch 1 (one-launch decode layer) and >= 5 (matrix-core path),
prompt lengths below, at and across the kernel's 16-token staging rounds, prompts split into
several chunks, head dimensions 16 / 32 / 64 (one, two and four 16-row state blocks per scan
workgroup), the 1.3B shape and the 2.7B layer shapes.
"""
import numpy as np
import pytest
import torch

from df_ssm_inference import DFSSMModel
from dfssm import _C
from dfssm.format import DFSSMConfig
from dfssm.synth import config_1p3b, config_tiny, make_prompts, make_weights
from oracle import oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _twins(w, B):
    return (DFSSMModel.from_weights(w, device=DEV, batch_size=B),
            DFSSMModel.from_weights(w, device=DEV, batch_size=B))


def _assert_same(a: DFSSMModel, b: DFSSMModel, la, lb):
    torch.cuda.synchronize()
    assert torch.equal(a.h_state, b.h_state), "SSM state differs"
    assert torch.equal(a.conv_state.view(torch.int16), b.conv_state.view(torch.int16)), "conv state differs"
    assert torch.equal(a.x.view(torch.int16), b.x.view(torch.int16)), "next-step input differs"
    assert torch.equal(a._next, b._next), "greedy token differs"
    if la is not None:
        assert torch.equal(la.view(torch.int16), lb.view(torch.int16)), "logits differ"
    assert a.error_flag() == 0 and b.error_flag() == 0


def _prefill_vs_steps(w, B, T, max_rows=None, steps_first=0):
    prompts = torch.from_numpy(make_prompts(B, w.cfg.vocab_size, T + steps_first))
    pf, st = _twins(w, B)
    if max_rows is not None:
        pf.PREFILL_MAX_ROWS = max_rows
    if steps_first:  # a state that is not zero when the prefill starts
        pf.ingest(prompts[:, :steps_first], step_by_step=True)
        st.ingest(prompts[:, :steps_first], step_by_step=True)
    lp = pf.prefill(prompts[:, steps_first:], want_logits=True)
    if T > 1:
        st.ingest(prompts[:, steps_first:-1], step_by_step=True)
    # the last prompt token through forward(): logits, greedy token and its embedding in x
    ls = st.forward(prompts[:, -1].to(DEV))
    _assert_same(pf, st, lp, ls)
    # continuing from both: the same greedy tokens
    gp = pf.decode(5)
    gs = st.decode(5)
    assert torch.equal(gp, gs)


@pytest.fixture(scope="module")
def tiny_weights():
    return make_weights(config_tiny(n_layer=3), seed=0)


@pytest.mark.parametrize("B,T", [(1, 1), (1, 17), (3, 40), (5, 16), (16, 9), (64, 3), (5, 61), (64, 9)])
def test_prefill_equals_steps_tiny(tiny_weights, B, T):
    print(f"prefill tiny B={B} T={T}", flush=True)
    _prefill_vs_steps(tiny_weights, B, T)


@pytest.mark.parametrize("B,T,rows", [(2, 37, 2 * 5), (8, 20, 8 * 7), (5, 33, 5 * 16)])
def test_prefill_chunks(tiny_weights, B, T, rows):
    """Prompts longer than one chunk (chunks of rows / B tokens), from a non-zero state."""
    print(f"prefill chunks B={B} T={T} rows={rows}", flush=True)
    _prefill_vs_steps(tiny_weights, B, T, max_rows=rows, steps_first=3)


@pytest.mark.parametrize("nheads,headdim", [(32, 32), (64, 16)])
def test_prefill_headdims(nheads, headdim):
    """Head dimensions 32 and 16 (two and one 16-row state blocks per scan workgroup), against
    step-by-step ingestion and the oracle's greedy tokens."""
    c = DFSSMConfig(n_layer=2, d_model=512, d_inner=1024, d_state=128, nheads=nheads, headdim=headdim,
                    ngroups=1, vocab_size=1000, kw=4)
    w = make_weights(c, seed=7)
    print(f"prefill heads {nheads} x {headdim}", flush=True)
    _prefill_vs_steps(w, 6, 21)
    B, T, n = 6, 21, 4
    prompts = make_prompts(B, c.vocab_size, T)
    ref, _ = O.OracleModel(w, B).generate(prompts, n)
    gpu = DFSSMModel.from_weights(w, device=DEV, batch_size=B)
    got = gpu.generate(n_tokens=n, prompt=torch.from_numpy(prompts), return_tokens=True, verbose=False)
    np.testing.assert_array_equal(got.cpu().numpy(), ref)


def test_prefill_1p3b():
    """1.3B shape, batch 4, 32-token prompts: prefill == 32 decode steps."""
    w = make_weights(config_1p3b(), seed=0)
    print("prefill 1.3B B=4 T=32", flush=True)
    _prefill_vs_steps(w, 4, 32)


def test_prefill_2p7b_layer_shapes():
    """Config 4's layer shapes (d_model 2560, d_inner 5120, 80 heads) at batch 64, 4 layers."""
    c = DFSSMConfig(n_layer=4, d_model=2560, d_inner=5120, d_state=128, nheads=80, headdim=64, ngroups=1,
                    vocab_size=4096, kw=4)
    w = make_weights(c, seed=5)
    print("prefill 2.7B layers B=64 T=20", flush=True)
    _prefill_vs_steps(w, 64, 20)


def _many_row_forms(dm, di, rows):
    """The forms that the many-row prologue (rows per workgroup, the same for both projections) and the wide GEMM
    (outputs per workgroup, in_proj and out_proj) take at a chunk of `rows` rows: the rules of launch_prep and
    launch_gemm_wide_mode."""
    assert rows > 64
    wide = lambda n: 256 if -(-rows // 64) * -(-n // 256) >= 640 else 128
    return 4 if rows <= 1024 else 16, wide(2 * di + 2 * 128 + di // 64), wide(dm)


@pytest.mark.parametrize("dm,di,B,T,forms", [
    # up to 1024 rows: four rows per workgroup of the prologue
    (1536, 3072, 5, 27, (4, 128, 128)),
    (1536, 3072, 5, 13, (4, 128, 128)),      # 65 rows: the smallest chunk of these kernels
    (4608, 512, 6, 43, (4, 128, 128)),
    (512, 512, 64, 16, (4, 128, 128)),       # 1024 rows
    # more: 16 rows per workgroup
    (2048, 4096, 5, 205, (16, 128, 128)),    # 1025 rows: one live row in the last workgroup; the 1.3B shape
    (512, 3584, 64, 19, (16, 128, 128)),
    (1536, 3072, 33, 33, (16, 128, 128)),    # 1089 rows; the LoRA contraction in one pass (3) and in two (6)
    # the wide tile of the GEMM, rows that no tile divides
    (2048, 4096, 37, 33, (16, 256, 128)),    # 1221 rows
    (4608, 512, 33, 69, (16, 128, 256)),     # 2277 rows: 648 tiles of out_proj
    (2560, 5120, 63, 65, (16, 256, 256)),    # 4095 rows: the 2.7B shape in the forms of its largest chunks
])
def test_prefill_many_rows(dm, di, B, T, forms):
    """The many-row prologue and GEMM (more than 64 rows) in each of their forms: both row counts of the
    prologue's workgroups and both sides of the switch, both widths of the GEMM's tile in both projections, odd
    multiples of 512 columns, one and two passes of the LoRA contraction, row counts that neither divides."""
    assert _many_row_forms(dm, di, B * T) == forms
    c = DFSSMConfig(n_layer=2 if dm < 2048 else 1, d_model=dm, d_inner=di, d_state=128, nheads=di // 64, headdim=64,
                    ngroups=1, vocab_size=1000, kw=4)
    print(f"prefill rows {B * T} of {dm} / {di}", flush=True)
    _prefill_vs_steps(make_weights(c, seed=11), B, T)


def test_prefill_rejects_bad_prompts(tiny_weights):
    gpu = DFSSMModel.from_weights(tiny_weights, device=DEV, batch_size=2)
    with pytest.raises(ValueError):
        gpu.prefill(torch.zeros(3, 4, dtype=torch.int64))
    with pytest.raises(IndexError):
        gpu.prefill(torch.full((2, 4), tiny_weights.cfg.vocab_size, dtype=torch.int64))


@pytest.mark.parametrize("B,T,heads,headdim", [(5, 18, 8, 64), (8, 37, 32, 16), (5, 21, 16, 64), (64, 6, 32, 16),
                                               (5, 4, 16, 64), (17, 9, 16, 64), (24, 7, 32, 32), (64, 13, 16, 64),
                                               (64, 1, 16, 64)])
def test_prefill_readout_order(B, T, heads, headdim):
    """The scan's C.h sums are added in the order of the batched decode step, in each of its forms (eight,
    four, two and one waves per 16-row block: up to 256 blocks, under 1024, under 4096, more). A state of large
    values that cancel in pairs (C constant, B zero) makes every fp64 sum depend on its order, by far
    more than the fp16 rounding of y."""
    di = heads * headdim
    c = DFSSMConfig(n_layer=1, d_model=512, d_inner=di, d_state=128, nheads=heads, headdim=headdim, ngroups=1,
                    vocab_size=1000, kw=4)
    w = make_weights(c, seed=3)
    L = w.layers[0]
    L["conv_w"][di:] = 0
    L["conv_b"][di:di + 128] = 0        # B = silu(0) = 0
    L["conv_b"][di + 128:] = 1.5        # C = one constant
    rng = np.random.default_rng(4)
    P = headdim
    big = (rng.uniform(1, 2, (B, heads, P, 32)) * 2.0 ** 50).astype(np.float32)
    h = np.concatenate([big, -big, rng.normal(0, 1, (B, heads, P, 64)).astype(np.float32)], axis=-1)
    h = np.take_along_axis(h, rng.permuted(np.tile(np.arange(128), (B, heads, P, 1)), axis=-1), axis=-1)
    # the sum does depend on the order: 64-bit sums of two orders differ by more than fp16 resolves
    d = h.astype(np.float64)
    assert np.median(np.abs(d.cumsum(-1)[..., -1] - d[..., ::-1].cumsum(-1)[..., -1])) > 0.01
    print(f"readout order B={B} T={T} {heads} x {headdim}", flush=True)
    pf, st = _twins(w, B)
    for m in (pf, st):
        m.h_state[0].copy_(torch.from_numpy(h))
    prompts = torch.from_numpy(make_prompts(B, c.vocab_size, T))
    lp = pf.prefill(prompts, want_logits=True)
    st.ingest(prompts[:, :-1], step_by_step=True)
    ls = st.forward(prompts[:, -1].to(DEV))
    _assert_same(pf, st, lp, ls)


def _norm_order_weights(chunk, small):
    """A one-layer model whose tokens all embed to one row of 2560 columns with a sum of squares that rounds to fp32
    one way or the other by the order of its fp64 sum. The large columns (2^15 and 8, the first two of a
    512-column chunk; n of 32) make 2^30 + 64 + 1024 n, in the middle of two fp32 values; the small ones (2^-12)
    count only if at least 2^-22 of their squares is added up before it meets the 2^30. The norm weights put
    the normalized values of the n columns where the two results round to different halves."""
    K, f4 = 2560, np.float32
    x = np.zeros(K, np.float16)
    x[512 * chunk:512 * chunk + 2] = 2.0 ** 15, 8.0
    assert not x[small].any()
    x[small] = 2.0 ** -12

    def scale(ss):  # 1 / sqrt(ss / K + 1e-5) as the kernels round it
        var = f4(f4(ss) * (f4(1) / f4(K)))
        return f4(1) / np.sqrt(var + f4(1e-5))

    for n in range(200, 400):
        lost = 2.0 ** 30 + 64 + 1024 * n
        r0, r1 = scale(lost), scale(lost + 2.0 ** -22)
        if r0 != r1:
            break
    assert r0 != r1 and lost + 2.0 ** -23 == lost
    fill = np.arange(600, 600 + n)
    x[fill] = 32.0
    w = np.ones(K, f4)
    w[512 * chunk] = 0.01
    halves = np.arange(0x3c00, 0x3c00 + n, dtype=np.uint16).view(np.float16).astype(np.float64)
    near = ((halves + 2.0 ** -11) / (32.0 * float(r0))).astype(f4).view(np.int32)
    w[fill] = near.view(f4)
    for d in range(-8, 9):  # the weight's last bits
        c = (near + d).astype(np.int32).view(f4)
        differ = ((f4(32) * r0) * c).astype(np.float16) != ((f4(32) * r1) * c).astype(np.float16)
        w[fill[differ]] = c[differ]
    flips = (((f4(32) * r0) * w[fill]).astype(np.float16) != ((f4(32) * r1) * w[fill]).astype(np.float16)).sum()
    assert flips > n // 2
    c = DFSSMConfig(n_layer=1, d_model=K, d_inner=512, d_state=128, nheads=8, headdim=64, ngroups=1, vocab_size=1000,
                    kw=4, emb_code=0)
    wt = make_weights(c, seed=2)
    wt.emb[:] = x
    wt.layers[0]["ln_w"][:] = w
    return wt


@pytest.mark.parametrize("chunk,lanes", [(0, None), (0, (2, 3)), (0, (1, 2)), (3, (4, 8)), (3, (8, 12)), (3, (16, 32)),
                                         (4, (32, 48))])
def test_prefill_norm_order(chunk, lanes):
    """The prefill's prologue adds its squares in the order of the decode step's (prep_kernel) in each of its forms:
    60, 65 and 1025 rows. The small columns lie 2048 columns behind the large one (None), or two each in two
    lanes of its chunk (8 columns a lane), which the tree adds to each other first or to the large one."""
    small = np.arange(2048, 2056) if lanes is None else np.concatenate([512 * chunk + 8 * l + np.arange(2, 4) for l in lanes])
    w = _norm_order_weights(chunk, small)
    for B, T in ((5, 12), (5, 13), (5, 205)):
        print(f"norm order chunk {chunk} lanes {lanes} B={B} T={T}", flush=True)
        _prefill_vs_steps(w, B, T)


def _gate_weights(z):
    """A one-layer model whose gate gets the halves z in every row and whose SSM readout is 1: the embedding is
    all ones, LoRA ranks 0 and 1 of in_proj carry 16 and 1, so that an integer 16 a + b times a power of two,
    any fp16 value, comes from the int8 factors a and b and the row scale; no scaffold term; x = silu of the
    conv bias, B = C = 0 and D = 1 / x."""
    c = DFSSMConfig(n_layer=1, d_model=512, d_inner=z.size, d_state=128, nheads=z.size // 64, headdim=64, ngroups=1,
                    vocab_size=1000, kw=4)
    w = make_weights(c, seed=1)
    w.emb[:], w.emb_scale[:] = 1, 1
    L = w.layers[0]
    L["ln_w"][:] = 1
    L["in_scale"][:] = 0
    L["in_lB"][:], L["in_lB_s"][:] = 0, 1
    L["in_lB"][0, 0], L["in_lB"][1, 0] = 16, 1
    m, e = np.frexp(z.astype(np.float64))
    e = np.maximum(e - 11, -24)  # z = m 2^e with |m| < 2048
    inf, nan = np.isinf(z), np.isnan(z)
    m = np.ldexp(np.where(inf | nan, 0, z.astype(np.float64)), -e).astype(np.int64)
    a, b, s = np.abs(m) // 16 * np.sign(m), np.abs(m) % 16 * np.sign(m), np.ldexp(1.0, e)
    a = np.where(inf, np.where(z > 0, 127, -127), np.where(nan, 127, a))
    b, s = np.where(nan, -127, b), np.where(inf | nan, 65504.0, s)  # inf - inf
    L["in_lA"][:], L["in_lA_s"][:] = 0, 1
    L["in_lA"][:z.size, 0], L["in_lA"][:z.size, 1], L["in_lA_s"][:z.size] = a, b, s
    L["conv_w"][:] = 0
    L["conv_b"][:z.size], L["conv_b"][z.size:] = 2, 0
    x = np.zeros((1, 1), np.float16)
    O.conv_step(np.zeros((1, 1, 3), np.float16), x, np.zeros((1, 4), np.float16), np.full(1, 2, np.float16))
    L["D"][:] = 1 / np.float32(x[0, 0])
    return w


def test_gate_all_halves():
    """The gate fp16(z fp16(sigmoid(z))) of every fp16 z but -0 (all finite values, the infinities, one NaN) in the
    batched decode step and in the prefill scan, as both leave it in their workspaces' g rows, against the
    oracle's formula, bit for bit."""
    bits = np.concatenate([np.arange(0, 0x7c02), np.arange(0x8001, 0xfc01)]).astype(np.uint16)
    B, DI = 5, 5120
    n = -(-bits.size // DI)
    bits = np.concatenate([bits, np.zeros(n * DI - bits.size, np.uint16)]).reshape(n, DI)
    align = lambda v: -(-v // 256) * 256
    for i in range(n):
        z = bits[i].view(np.float16)
        ref = O.gate(np.ones((1, DI), np.float16), z.reshape(1, DI))[0]
        w = _gate_weights(z)
        gpu = DFSSMModel.from_weights(w, device=DEV, batch_size=B)
        ld = w.cfg.in_proj_out
        print(f"gate of halves {i + 1} / {n}", flush=True)
        gpu.prefill(torch.zeros(B, 1, dtype=torch.int64))
        proj = align(B * w.cfg.d_model * 2)                      # rows of x, then of in_proj, then of g
        pf = gpu._pf_ws[proj:].view(torch.float16)[:B * ld].view(B, ld)[:, :DI].cpu().numpy()
        nan = np.isnan(z)
        np.testing.assert_array_equal(pf[0].view(np.uint16)[~nan], z.view(np.uint16)[~nan])  # the gate's input
        rows = [gpu._pf_ws[proj + align(B * ld * 2):]]
        x = torch.ones(B, w.cfg.d_model, dtype=torch.float16, device=DEV)
        gpu.reset_state()
        for ph in range(3):  # in_proj's prologue, in_proj + conv, SSM + gate
            _C.check(_C.lib().dfssm_layer_phase(gpu._model, 0, ph, x.data_ptr(), gpu._state, gpu.workspace.data_ptr(),
                                                _C.stream()))
        rows.append(gpu.workspace[align(B * ld * 2):])           # rows of in_proj, then of g
        for r in rows:
            got = r.view(torch.float16)[:B * DI].view(B, DI).cpu().numpy()
            assert np.isnan(got[:, nan]).all()
            for b in range(B):
                np.testing.assert_array_equal(got[b].view(np.uint16)[~nan], ref.view(np.uint16)[~nan])
