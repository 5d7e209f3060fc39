"""Host-side logic of the drop-in API, checked without a GPU: the one-launch layer's residency
rule (dfssm_one_launch_plan), the decoding of the workspace error flag, and token range checks that
must fire before any kernel reads the ids."""
import os

import numpy as np
import pytest
import torch

from dfssm import _C, ops
from dfssm.synth import config_tiny
import df_ssm_inference as dfi


def _dims(**kw):
    base = dict(n_layer=48, d_model=2048, d_inner=4096, d_state=128, nheads=64, headdim=64, ngroups=1,
                vocab_size=50288, batch=1, emb_code=1)
    base.update(kw)
    return _C.Dims(*[base[f] for f, _ in _C.Dims._fields_])


@pytest.mark.parametrize("kw,cus,per_cu,grid", [
    ({}, 256, 1, 256),                 # MI355X: one 1024-thread workgroup per CU
    ({}, 256, 2, 256),
    ({}, 256, 0, 0),                   # the instantiation does not fit a CU: five kernels
    ({"batch": 4}, 256, 1, 256),
    ({"batch": 5}, 256, 1, 0),         # batch >= 5 always runs five kernels
    ({}, 140, 1, 0),                   # 133 in_proj groups + 16 LoRA workgroups do not fit
    ({}, 2048, 1, 1024),               # one workgroup per CU, at most 1024
    ({"d_model": 2560, "d_inner": 5120, "nheads": 80}, 256, 1, 256),
    ({"batch": 65}, 256, 1, 0),
])
def test_one_launch_plan(kw, cus, per_cu, grid):
    assert _C.lib().dfssm_one_launch_plan(_dims(**kw), cus, per_cu) == grid


def test_describe_error_flag():
    """Every bit names its own source (the launch whose bounded wait gave up), as include/dfssm.h
    defines them."""
    assert dfi.describe_error_flag(0) == ""
    assert (dfi.ERR_TOKEN_RANGE, dfi.ERR_WAIT_LAYER, dfi.ERR_WAIT_SSM_PROLOGUE, dfi.ERR_WAIT_OUT_PROLOGUE) == \
        (1, 4, 8, 16)
    assert "token id out of range" in dfi.describe_error_flag(dfi.ERR_TOKEN_RANGE)
    layer = dfi.describe_error_flag(dfi.ERR_WAIT_LAYER)
    ssm = dfi.describe_error_flag(dfi.ERR_WAIT_SSM_PROLOGUE)
    out = dfi.describe_error_flag(dfi.ERR_WAIT_OUT_PROLOGUE)
    assert "one-launch layer" in layer and "timed out" in layer
    assert "SSM" in ssm and "timed out" in ssm and "one-launch" not in ssm
    assert "out_proj" in out and "timed out" in out and "one-launch" not in out
    assert len({layer, ssm, out}) == 3
    every = dfi.describe_error_flag(1 | 4 | 8 | 16 | 64)
    assert all(x in every for x in ("out of range", layer, ssm, out, "0x40"))


def test_error_bits_match_header():
    """The Python constants are the C header's DFSSM_ERR_* values."""
    import os
    import re
    hdr = open(os.path.join(os.path.dirname(__file__), "..", "include", "dfssm.h")).read()
    vals = dict(re.findall(r"#define DFSSM_ERR_(\w+) (\d+)", hdr))
    assert {k: int(v) for k, v in vals.items()} == {
        "TOKEN_RANGE": dfi.ERR_TOKEN_RANGE, "WAIT_LAYER": dfi.ERR_WAIT_LAYER,
        "WAIT_SSM_PROLOGUE": dfi.ERR_WAIT_SSM_PROLOGUE, "WAIT_OUT_PROLOGUE": dfi.ERR_WAIT_OUT_PROLOGUE}


def _hostless_model(B=2):
    """A DFSSMModel shell with no device state: any kernel launch or device access would fail
    with AttributeError, so a test that expects IndexError shows the check ran first."""
    m = dfi.DFSSMModel.__new__(dfi.DFSSMModel)
    m.batch_size = B
    m.cfg = config_tiny(n_layer=1)
    return m


@pytest.mark.parametrize("bad", [-1, "V"])
def test_generate_checks_prompt_range_before_launch(bad):
    m = _hostless_model()
    V = m.cfg.vocab_size
    tok = V if bad == "V" else bad
    prompt = torch.tensor([[1, 2], [3, tok]])
    with pytest.raises(IndexError):
        m.generate(n_tokens=4, prompt=prompt, verbose=False)
    with pytest.raises(IndexError):
        m.generate(n_tokens=4, prompt=prompt, temperature=0.7, verbose=False)
    with pytest.raises(IndexError):
        m.ingest(prompt)
    with pytest.raises(IndexError):
        m.prefill(prompt)
    with pytest.raises(IndexError):
        m.forward(torch.tensor([0, tok]))


def test_generate_checks_prompt_shape():
    m = _hostless_model(B=2)
    with pytest.raises(ValueError):
        m.generate(n_tokens=4, prompt=torch.zeros(3, 2, dtype=torch.int64), verbose=False)


def test_stream_in_forked_child_asks_torch_again(monkeypatch):
    """A process that has launched work asks torch's C layer for the stream directly; a child forked from it
    goes through torch.cuda again, whose error for a forked GPU context must reach the caller."""
    class Stream:
        cuda_stream = 7

    monkeypatch.setattr(_C, "_get_raw_stream", None)
    monkeypatch.setattr(torch.cuda, "current_stream", Stream)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda device: 9, raising=False)
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: 0, raising=False)
    assert (_C.stream(), _C.stream()) == (7, 9)

    def refuse():
        raise RuntimeError("Cannot re-initialize CUDA in forked subprocess")

    monkeypatch.setattr(torch.cuda, "current_stream", refuse)
    assert _C.stream() == 9
    pid = os.fork()
    if pid == 0:
        try:
            _C.stream()
            os._exit(1)
        except RuntimeError:
            os._exit(0)
    assert os.waitstatus_to_exitcode(os.waitpid(pid, 0)[1]) == 0


@pytest.fixture
def host_workspaces(monkeypatch):
    """scaffold_workspace without a GPU: an empty cache, buffers on the host, a settable stream handle."""
    real, env = torch.zeros, {"stream": 1, "capturing": False}
    monkeypatch.setattr(torch, "zeros", lambda *a, device=None, **k: real(
        *a, device=device if torch.device(device).type == "meta" else None, **k))
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: env["capturing"])
    monkeypatch.setattr(_C, "stream", lambda: env["stream"])
    monkeypatch.setattr(ops, "_scaffold_ws", type(ops._scaffold_ws)())
    return env


def test_scaffold_workspace_of_another_device_type(host_workspaces):
    """A workspace asked for on another device type is not handed to the GPU's calls, nor the other way round."""
    host = ops.scaffold_workspace("cpu")
    assert host.device.type == "cpu" and ops.scaffold_workspace("cpu") is host
    assert ops.scaffold_workspace(torch.device("meta")).device.type == "meta"


def test_scaffold_workspace_per_stream(host_workspaces):
    """Calls on two streams may overlap and calls that share a workspace must not: every stream has its own,
    every call of a capture too (its graph may be replayed on any stream), and the number kept is bounded."""
    first = ops.scaffold_workspace("cuda:0")
    assert ops.scaffold_workspace("cuda") is first
    host_workspaces["stream"] = 2
    second = ops.scaffold_workspace("cuda:0")
    assert second.data_ptr() != first.data_ptr()
    assert ops.scaffold_workspace("cuda:1").data_ptr() != second.data_ptr()
    host_workspaces["capturing"] = True
    captured = [ops.scaffold_workspace("cuda:0") for _ in range(2)]
    assert len({t.data_ptr() for t in captured + [first, second]}) == 4
    host_workspaces["capturing"] = False
    assert ops.scaffold_workspace("cuda:0") is second
    for host_workspaces["stream"] in range(100, 400):
        ops.scaffold_workspace("cuda:0")
    assert len(ops._scaffold_ws) <= 64
