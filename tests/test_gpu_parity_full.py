"""Parity at the benchmark configurations' full shapes, and the drop-in surfaces called the way the
reference calls them.

* config 1: the scaffold projection with its rank-16 int8 LoRA as one operator
  (dfssm_scaffold_lora_gemm) at in_proj / out_proj shapes (and the 2.7B and edge shapes),
  M in {1, 2, 3, 4, 16, 32}, with and without the exchange workspace: int32 accumulators, LoRA
  intermediates and y bit-exact against the oracle; one workspace shared by consecutive calls of
  different shapes;
* config 3 at batch 32: the 1.3B model (48 layers, vocab 50288) greedy, identical tokens and
  logits at every step (the batched exact head at 32 rows);
* config 4's dimensions at batch 64 with the full 50288-token vocabulary (2 layers so that the
  oracle stays fast): tokens and logits identical;
* config 4's layer shapes through a 300-token prompt prefill split into chunks, against
  step-by-step ingestion at batch 4;
* DFSSMModel(path) on files written by the exporter (fp16 and int8 tables);
* the b2 module df_ssm_kernels called as df_ssm_inference.py:177-191 calls it, for 16 steps;
* the reference-shaped embedding attribute.
"""
import numpy as np
import pytest
import torch

from df_ssm_inference import DFSSMModel
from dfssm import _C, ops
from dfssm.format import EMB_F16, EMB_I8, DFSSMConfig
from dfssm.synth import config_1p3b, make_prompts, make_weights
from oracle import oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _h(a):  # numpy fp16 -> torch fp16 on the GPU
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).to(DEV).view(torch.float16)


def _np16(t):
    return t.detach().cpu().view(torch.int16).numpy().view(np.float16)


# ------------------------------------------------------------------------------ config 1
def _lora_op_case(N, K, M, seed):
    """Inputs of one scaffold + LoRA call (the benchmark's distributions) and its oracle outputs."""
    rng = np.random.default_rng([1, N, K, M, seed])
    bits = rng.integers(0, 2**32, (N, K // 32), dtype=np.uint64).astype(np.uint32)
    ws = rng.uniform(0.01, 0.05, N).astype(np.float16)
    xn = rng.normal(0, 1, (M, K)).astype(np.float16)
    q, xs = O.quantize(xn)   # the activations the scaffold sees are xn's quantization
    lA = np.clip(np.rint(rng.normal(0, 20, (N, 16))), -127, 127).astype(np.int8)
    lAs = (1.7e-3 * rng.uniform(0.5, 1.5, N)).astype(np.float16)
    lB = np.clip(np.rint(rng.normal(0, 20, (16, K))), -127, 127).astype(np.int8)
    lBs = (rng.uniform(0.5, 1.5, 16) / (20 * np.sqrt(K))).astype(np.float16)
    tb = ops.tile_bits(torch.from_numpy(bits.view(np.int32)).to(DEV), N, K)
    lBq = torch.empty(16, K, dtype=torch.float16, device=DEV)
    tB, tBs = torch.from_numpy(lB).to(DEV), _h(lBs)  # kept alive until the kernel has run
    _C.check(_C.lib().dfssm_dequant_lora_b(tB.data_ptr(), tBs.data_ptr(), K, lBq.data_ptr(), _C.stream()))
    torch.cuda.synchronize()
    args = (tb, _h(ws), torch.from_numpy(q).to(DEV), _h(xs), _h(xn), torch.from_numpy(lA).to(DEV), _h(lAs), lBq, N)
    acc_r = O.scaffold_acc(bits, q)
    h_r = O.lora_h(xn, lB, lBs)
    y_r = O.dequant_lora(acc_r, xs, ws, h_r, lA, lAs)
    assert np.abs(y_r.astype(np.float32)).max() > 0
    return args, (acc_r, h_r, y_r)


def _check_lora_op(out, ref):
    acc, y, h = out
    acc_r, h_r, y_r = ref
    np.testing.assert_array_equal(acc.cpu().numpy(), acc_r)
    np.testing.assert_array_equal(_np16(h).view(np.uint16), h_r.view(np.uint16))
    np.testing.assert_array_equal(_np16(y).view(np.uint16), y_r.view(np.uint16))


@pytest.mark.parametrize("N,K", [(8512, 2048), (2048, 4096), (10576, 2560), (2560, 5120), (64, 512)])
@pytest.mark.parametrize("M", [1, 2, 3, 4, 16, 32])
@pytest.mark.parametrize("xchg", [True, False])
def test_scaffold_lora_op_bit_exact(N, K, M, xchg):
    """Packed bits with fp16 row scales ~U(0.01, 0.05), int8 activations
    ~N(0, 40) clipped with fp16 per-token scales, rank-16 int8 LoRA A/B; xn is the fp16 vector
    the activations quantize (the LoRA reads it, df_ssm_inference.py:173). xchg: with the exchange
    workspace (one launch at M <= 4), else without."""
    print(f"scaffold+lora N={N} K={K} M={M} xchg={xchg}", flush=True)
    args, ref = _lora_op_case(N, K, M, 0)
    wsx = torch.zeros(ops.SCAFFOLD_WORKSPACE_BYTES // 4, dtype=torch.int32, device=DEV) if xchg else None
    _check_lora_op(ops.scaffold_lora_gemm(*args, workspace=wsx), ref)
    if xchg:
        assert ops.scaffold_error(wsx) == 0


def test_scaffold_lora_op_shared_workspace():
    """One exchange workspace across consecutive calls whose grids cover different numbers of output
    rows, batches and K (every call must find the words of its own call, not of an earlier one), the
    same call twice in a row, and calls in between that take the matrix-core path (M K > 8192) and
    leave the workspace alone."""
    wsx = torch.zeros(ops.SCAFFOLD_WORKSPACE_BYTES // 4, dtype=torch.int32, device=DEV)
    cases = [(8512, 2048, 1), (2048, 4096, 1), (64, 512, 4), (10576, 2560, 2), (8512, 2048, 1),
             (2048, 4096, 3), (2048, 4096, 3)]
    for i, (N, K, M) in enumerate(cases):
        print(f"shared workspace call {i}: N={N} K={K} M={M}", flush=True)
        args, ref = _lora_op_case(N, K, M, i)
        _check_lora_op(ops.scaffold_lora_gemm(*args, workspace=wsx), ref)
    assert ops.scaffold_error(wsx) == 0
    counts = wsx[:256].cpu().numpy()
    one_launch = sum(M <= 4 and M * K <= 8192 for N, K, M in cases)
    assert one_launch == 5
    assert (counts == one_launch).all()  # every workgroup index counted every one-launch call


def test_scaffold_lora_op_tags_wrap():
    """The 16-bit tag of a call's words comes round after 65 536 calls: a call of four rows with the tag of an
    earlier one, calls of one row between them (the counts are set forward in place of most of these, but not
    past one that 2^14 divides), waits for its own words."""
    wsx = torch.zeros(ops.SCAFFOLD_WORKSPACE_BYTES // 4, dtype=torch.int32, device=DEV)
    for i, (M, count) in enumerate([(4, 5), (1, 16384), (1, 65540), (4, 65541), (2, 81920), (3, 131077),
                                          (2, 147456), (4, 196613)]):
        print(f"tag wrap: call {count + 1} with {M} rows", flush=True)
        wsx[:256] = count
        args, ref = _lora_op_case(8512, 2048, M, 30 + i)
        _check_lora_op(ops.scaffold_lora_gemm(*args, workspace=wsx), ref)
    assert ops.scaffold_error(wsx) == 0


def test_scaffold_lora_op_streams_and_graphs():
    """Calls with the automatic workspace on two streams that may overlap, and in a captured graph replayed
    between eager calls: every result is the oracle's."""
    cases = [_lora_op_case(8512, 2048, 1, 20), _lora_op_case(2048, 2048, 4, 21)]
    print("scaffold+lora on two streams", flush=True)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    outs = []
    for _ in range(8):
        for s, (args, _) in zip(streams, cases):
            with torch.cuda.stream(s):
                outs.append(ops.scaffold_lora_gemm(*args))
    torch.cuda.synchronize()
    for i, out in enumerate(outs):
        _check_lora_op(out, cases[i % 2][1])
    print("scaffold+lora in a graph", flush=True)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        captured = [ops.scaffold_lora_gemm(*args) for args, _ in cases]
    for _ in range(4):
        g.replay()
        torch.cuda.synchronize()
        for out, (_, ref) in zip(captured, cases):
            _check_lora_op(out, ref)
            out[1].zero_()
        for args, ref in cases:
            _check_lora_op(ops.scaffold_lora_gemm(*args), ref)


# ------------------------------------------------------------------------------ config 3, B = 32
@pytest.fixture(scope="module")
def w13():
    return make_weights(config_1p3b(), seed=0)


def test_1p3b_batch32_stepwise(w13):
    """1.3B at batch 32: 8 prompt tokens then 4 greedy steps through forward(), logits identical to
    the oracle at every step, then the state within 1e-3."""
    w, B = w13, 32
    print("1.3B B=32 stepwise", flush=True)
    prompts = make_prompts(B, w.cfg.vocab_size, 8)
    gpu = DFSSMModel.from_weights(w, device=DEV, batch_size=B)
    orc = O.OracleModel(w, B)
    tok = prompts[:, 0]
    for t in range(12):
        lg = _np16(gpu.forward(torch.from_numpy(tok).to(DEV))).astype(np.float32)
        lo, nxt = orc.step(tok)
        assert np.abs(lg - lo.astype(np.float32)).max() == 0.0, f"step {t}: logits differ"
        np.testing.assert_array_equal(lg.argmax(axis=1), nxt)
        tok = prompts[:, t + 1] if t + 1 < prompts.shape[1] else nxt
        print(f"  step {t} ok", flush=True)
    rel = np.abs(gpu.h_state.cpu().numpy() - orc.h).max() / np.abs(orc.h).max()
    assert rel <= 1e-3
    assert gpu.error_flag() == 0


# ------------------------------------------------------------------------------ config 4 dims
def test_2p7b_dims_full_vocab_batch64():
    """Config 4's dimensions (d_model 2560, d_inner 5120, 80 heads) at batch 64 with the full
    50288-token vocabulary (the batched exact head at D 2560): 2 layers, 2 prompt tokens and 2
    generated, tokens and final logits identical to the oracle."""
    c = DFSSMConfig(n_layer=2, d_model=2560, d_inner=5120, d_state=128, nheads=80, headdim=64, ngroups=1,
                    vocab_size=50288, kw=4)
    w = make_weights(c, seed=7)
    B = 64
    print("2.7B dims, V=50288, B=64", flush=True)
    prompts = make_prompts(B, c.vocab_size, 2)
    orc = O.OracleModel(w, B)
    ref, _ = orc.generate(prompts, 2)
    gpu = DFSSMModel.from_weights(w, device=DEV, batch_size=B)
    got = gpu.generate(n_tokens=2, prompt=torch.from_numpy(prompts), return_tokens=True, verbose=False)
    np.testing.assert_array_equal(got.cpu().numpy(), ref)
    lg = _np16(gpu.forward(torch.from_numpy(ref[:, -1]).to(DEV))).astype(np.float32)
    lo, _ = orc.step(ref[:, -1])
    assert np.abs(lg - lo.astype(np.float32)).max() == 0.0
    assert np.abs(gpu.h_state.cpu().numpy() - orc.h).max() <= 1e-3 * np.abs(orc.h).max()
    assert gpu.error_flag() == 0


@pytest.mark.parametrize("B", [1, 5])
def test_largest_vocab_head(B):
    """The largest supported vocabulary (65536 = 1024 table groups: the most per-workgroup argmax
    pairs the heads' last workgroup reduces) at B = 1 (head_i8_kernel) and B = 5 (head_i8s_kernel):
    tokens and final logits identical to the oracle."""
    c = DFSSMConfig(n_layer=1, d_model=512, d_inner=1024, d_state=128, nheads=16, headdim=64, ngroups=1,
                    vocab_size=65536, kw=4)
    w = make_weights(c, seed=11)
    print(f"V=65536 head, B={B}", flush=True)
    prompts = make_prompts(B, c.vocab_size, 3)
    orc = O.OracleModel(w, B)
    ref, _ = orc.generate(prompts, 3)
    gpu = DFSSMModel.from_weights(w, device=DEV, batch_size=B)
    got = gpu.generate(n_tokens=3, prompt=torch.from_numpy(prompts), return_tokens=True, verbose=False)
    np.testing.assert_array_equal(got.cpu().numpy(), ref)
    lg = _np16(gpu.forward(torch.from_numpy(ref[:, -1]).to(DEV))).astype(np.float32)
    lo, _ = orc.step(ref[:, -1])
    assert np.abs(lg - lo.astype(np.float32)).max() == 0.0
    assert gpu.error_flag() == 0


def test_2p7b_layers_prefill_300_chunked():
    """A 300-token prompt through config 4's layer shapes at batch 4, prefilled in chunks of 128
    tokens (two chunk boundaries), against 300 decode steps: state, conv state, next-step input,
    greedy token and last logits bit-identical, and 4 continued tokens equal."""
    c = DFSSMConfig(n_layer=2, d_model=2560, d_inner=5120, d_state=128, nheads=80, headdim=64, ngroups=1,
                    vocab_size=4096, kw=4)
    w = make_weights(c, seed=8)
    B, T = 4, 300
    print("2.7B layers, prefill 300 tokens in chunks of 128", flush=True)
    prompts = torch.from_numpy(make_prompts(B, c.vocab_size, T))
    pf = DFSSMModel.from_weights(w, device=DEV, batch_size=B)
    st = DFSSMModel.from_weights(w, device=DEV, batch_size=B)
    pf.PREFILL_MAX_ROWS = B * 128
    lp = pf.prefill(prompts, want_logits=True)
    st.ingest(prompts[:, :-1], step_by_step=True)
    ls = st.forward(prompts[:, -1].to(DEV))
    torch.cuda.synchronize()
    assert torch.equal(pf.h_state, st.h_state)
    assert torch.equal(pf.conv_state.view(torch.int16), st.conv_state.view(torch.int16))
    assert torch.equal(pf.x.view(torch.int16), st.x.view(torch.int16))
    assert torch.equal(pf._next, st._next)
    assert torch.equal(lp.view(torch.int16), ls.view(torch.int16))
    assert torch.equal(pf.decode(4), st.decode(4))


# ------------------------------------------------------------------------------ wide prefill vs the oracle
@pytest.mark.parametrize("case", ["tiny_b16_t33", "2p7b_layers_b64_t6", "d512_di5120_b64_t18", "d4608_di512_b64_t37"])
def test_generate_wide_prefill_vs_oracle(case):
    """generate(prompt=...) whose prefill takes the many-row kernels (one chunk of more than 64 rows), against
    the oracle's step-by-step ingestion: greedy tokens and the logits of one more step identical, state within
    1e-3. Up to 1024 rows (prep_few_rows_kernel, the GEMM's narrow tile): the tiny model at batch 16 with a
    33-token prompt (512 prefill rows); the 2.7B layer shapes with the full vocabulary at batch 64 with a
    6-token prompt (320 rows). More (prep_rows_kernel): 1088 rows with the wide tile in in_proj, 2304 rows
    with the wide tile in out_proj."""
    if case == "tiny_b16_t33":
        from dfssm.synth import config_tiny
        c, B, T, n = config_tiny(n_layer=3), 16, 33, 4
    elif case == "2p7b_layers_b64_t6":
        c = DFSSMConfig(n_layer=2, d_model=2560, d_inner=5120, d_state=128, nheads=80, headdim=64, ngroups=1,
                        vocab_size=50288, kw=4)
        B, T, n = 64, 6, 2
    else:
        dm, di, T = (512, 5120, 18) if case.startswith("d512") else (4608, 512, 37)
        c = DFSSMConfig(n_layer=1, d_model=dm, d_inner=di, d_state=128, nheads=di // 64, headdim=64, ngroups=1,
                        vocab_size=1000, kw=4)
        B, n = 64, 2
        tiles = -(-B * (T - 1) // 64) * -(-(c.in_proj_out if dm == 512 else dm) // 256)
        assert B * (T - 1) > 1024 and tiles >= 640  # 16 rows per prologue workgroup, the GEMM's wide tile
    assert B * (T - 1) > 64  # the many-row kernels
    w = make_weights(c, seed=21)
    print(f"wide prefill vs oracle: {case}", flush=True)
    prompts = make_prompts(B, c.vocab_size, T, base_seed=4000)
    orc = O.OracleModel(w, B)
    ref, _ = orc.generate(prompts, n)
    gpu = DFSSMModel.from_weights(w, device=DEV, batch_size=B)
    got = gpu.generate(n_tokens=n, prompt=torch.from_numpy(prompts), return_tokens=True, verbose=False)
    np.testing.assert_array_equal(got.cpu().numpy(), ref)
    lg = _np16(gpu.forward(torch.from_numpy(ref[:, -1]).to(DEV))).astype(np.float32)
    lo, _ = orc.step(ref[:, -1])
    assert np.abs(lg - lo.astype(np.float32)).max() == 0.0
    assert np.abs(gpu.h_state.cpu().numpy() - orc.h).max() <= 1e-3 * np.abs(orc.h).max()
    gpu.check_errors()


@pytest.mark.parametrize("B,chunk_rows", [(4, 256), (64, 512)])
def test_config4_full_depth_vs_oracle_fixture(B, chunk_rows):
    """The whole config-4 model (2.7B shape, 64 layers, vocabulary 50288; bench.py's weights)
    against the oracle's runs committed in tests/golden/oracle_2p7b_64layer_b{4,64}.npz
    (tests/golden/make_config4_golden.py): at batch 4 a 129-token prompt prefilled in two chunks of
    64 tokens, at batch 64 (the benchmark's batch) a 17-token prompt in two chunks of 8 tokens
    (256 and 512 rows per chunk: the wide kernels and a chunk boundary), 4 greedy tokens, then one
    more step: tokens identical, and the SHA-256 of its fp16 logits, of the fp32 SSM state and of
    the conv state equal to the oracle's."""
    import hashlib
    import os
    from dfssm.synth import config_2p7b

    def sha(a):
        return hashlib.sha256(np.ascontiguousarray(a).tobytes()).hexdigest()

    g = np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", f"oracle_2p7b_64layer_b{B}.npz"))
    w = make_weights(config_2p7b(), seed=0)
    assert g["prompt"].shape[0] == B
    print(f"config 4 full depth (64 layers) vs oracle fixture, batch {B}", flush=True)
    gpu = DFSSMModel.from_weights(w, device=DEV, batch_size=B)
    gpu.PREFILL_MAX_ROWS = chunk_rows
    got = gpu.generate(n_tokens=g["tokens"].shape[1], prompt=torch.from_numpy(g["prompt"]), return_tokens=True,
                       verbose=False)
    np.testing.assert_array_equal(got.cpu().numpy(), g["tokens"])
    lg = _np16(gpu.forward(torch.from_numpy(g["tokens"][:, -1]).to(DEV)))
    np.testing.assert_array_equal(lg[:, :8].view(np.uint16), g["logits_head"].view(np.uint16))
    assert sha(lg) == str(g["logits_sha256"])
    np.testing.assert_array_equal(gpu._next.cpu().numpy(), g["next_token"])
    assert sha(gpu.h_state.cpu().numpy()) == str(g["state_sha256"])
    assert sha(_np16(gpu.conv_state)) == str(g["conv_sha256"])
    gpu.check_errors()


# ------------------------------------------------------------------------------ files from the exporter
@pytest.mark.parametrize("emb_code", [EMB_F16, EMB_I8])
@pytest.mark.parametrize("B", [1, 5])
def test_model_from_exported_file(tmp_path, emb_code, B):
    """DFSSMModel(path) (the reference's constructor, df_ssm_inference.py:48) on a .dfssm file the
    exporter wrote from a float student state dict: greedy tokens equal the oracle's on the same
    file, and the reference-shaped embedding attribute equals the file's table."""
    from dfssm.export import export_dfssm
    from dfssm.format import read_dfssm
    from test_export import _student_sd
    path = str(tmp_path / f"student_{emb_code}.dfssm")
    export_dfssm(_student_sd(), path, emb_code=emb_code)
    w = read_dfssm(path)
    print(f"exported file emb_code={emb_code} B={B}", flush=True)
    gpu = DFSSMModel(path, device=DEV, batch_size=B)
    prompts = make_prompts(B, w.cfg.vocab_size, 5)
    got = gpu.generate(n_tokens=6, prompt=torch.from_numpy(prompts), return_tokens=True, verbose=False)
    ref, _ = O.OracleModel(w, B).generate(prompts, 6)
    np.testing.assert_array_equal(got.cpu().numpy(), ref)
    emb = gpu.embedding
    assert tuple(emb.shape) == (w.cfg.vocab_size, w.cfg.d_model) and emb.dtype == torch.float16
    np.testing.assert_array_equal(_np16(emb).view(np.uint16), w.emb_f16().view(np.uint16))


# ------------------------------------------------------------------------------ b2 module
@pytest.mark.parametrize("B", [1, 32])
def test_df_ssm_kernels_reference_call_pattern(B):
    """df_ssm_kernels.conv_step / ssm_step called exactly as df_ssm_inference.py:177-191 calls them
    (xBC a contiguous copy of the projection slice, mutated in place by conv_step; y_buf zeroed,
    then written by ssm_step) at config 2's shapes for 16 steps: conv state and fp32 state
    bit-identical to the oracle, y within the operator test's tolerance."""
    import df_ssm_kernels
    H, P, N = 64, 64, 128
    D_INNER = H * P
    D_XBC = D_INNER + 2 * N
    print(f"df_ssm_kernels B={B}", flush=True)
    rng = np.random.default_rng([9, B])
    conv_w = rng.normal(0, 0.5, (D_XBC, 4)).astype(np.float16)
    conv_b = rng.normal(0, 0.1, D_XBC).astype(np.float16)
    A_log = rng.uniform(0, np.log(16), H).astype(np.float32)
    Dp = np.ones(H, np.float32)
    dt_bias = rng.normal(-3, 0.5, H).astype(np.float32)
    conv_states = torch.zeros(B, D_XBC, 3, dtype=torch.float16, device=DEV)
    h_states = torch.zeros(B, H, P, N, dtype=torch.float32, device=DEV)
    y_buf = torch.empty(B, D_INNER, dtype=torch.float16, device=DEV)
    tw, tb = _h(conv_w), _h(conv_b)
    tdb, tA, tD = (torch.from_numpy(a).to(DEV) for a in (dt_bias, A_log, Dp))
    r_conv = np.zeros((B, D_XBC, 3), np.float16)
    r_h = np.zeros((B, H, P, N), np.float32)
    for t in range(16):
        proj = rng.normal(0, 1, (B, D_INNER + D_XBC + H)).astype(np.float16)
        proj[:, D_INNER + D_XBC:] = rng.normal(-2, 1, (B, H)).astype(np.float16)
        tproj = _h(proj)
        xBC = tproj[:, D_INNER:D_INNER + D_XBC].contiguous()
        dt = tproj[:, D_INNER + D_XBC:D_INNER + D_XBC + H].contiguous()
        df_ssm_kernels.conv_step(conv_states, xBC, tw, tb, D_XBC)
        y_buf.zero_()
        df_ssm_kernels.ssm_step(h_states, xBC, dt, tdb, tA, tD, y_buf)
        rx = np.ascontiguousarray(proj[:, D_INNER:D_INNER + D_XBC])
        O.conv_step(r_conv, rx, conv_w, conv_b)
        r_y = O.ssm_step(r_h, rx, np.ascontiguousarray(proj[:, D_INNER + D_XBC:]), dt_bias, A_log, Dp)
        np.testing.assert_array_equal(_np16(xBC).view(np.uint16), rx.view(np.uint16))
        # y: the C.h readout is an fp64 sum whose order differs (tree on the GPU, sequential in
        # the oracle); the tolerance of the conv + SSM operator test
        gy, ry = _np16(y_buf).astype(np.float32), r_y.astype(np.float32)
        assert np.abs(gy - ry).max() <= 1e-3 * np.abs(ry).max() + 1e-3
    np.testing.assert_array_equal(_np16(conv_states).view(np.uint16), r_conv.view(np.uint16))
    np.testing.assert_array_equal(h_states.cpu().numpy(), r_h)
