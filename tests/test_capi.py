"""The ctypes binding's host side: what it needs of torch, and the workspaces
that it allocates for a call on another stream."""
import subprocess
import sys
import types

import numpy as np
import pytest

from conftest import ROOT


def test_host_only_calls_need_no_torch():
    code = ("import sys; sys.modules['torch'] = None\n"
            "from vm_c_amd import capi\n"
            "assert capi.version() and capi.kv_entry_bytes(capi.KV_Q8_0, 128) == 136\n"
            "assert capi.tq_config(128, 'turboquant_3bit_nc').slot_size_aligned == 102\n"
            "assert len(capi.tq_host_tables(128, 3)[0]) == 8\n")
    subprocess.run([sys.executable, "-c", code], check=True, cwd=ROOT)


@pytest.mark.parametrize("raw", [True, False])
def test_current_stream(monkeypatch, raw):
    """With torch's raw query and, where a torch has none, by the public one."""
    import torch
    from vm_c_amd import capi
    monkeypatch.setattr(capi, "_current_stream", capi._bind_current_stream)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 3)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(cuda_stream=7))
    if raw:
        monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda d: 100 + d, raising=False)
    else:
        monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    assert [capi._stream(), capi._stream()] == [103 if raw else 7] * 2
    assert capi._stream(types.SimpleNamespace(cuda_stream=11)) == 11


@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 128, 256])
def test_own_workspace_on_another_stream(dev, d):
    """A decode on a busy side stream without a workspace: memory that the
    current stream gets after the call is not the one the call still writes its
    partial rows to."""
    import torch
    from vm_c_amd import capi
    B, H, L = 2, 8, 4096
    q = torch.randn(B, H, d, device=dev).half()
    kc, vc = (torch.randn(B * L * H * d, device=dev).half().view(torch.uint8) for _ in range(2))
    bt = torch.from_numpy(np.arange(B * L // 16, dtype=np.int32).reshape(B, -1)).to(dev)
    lens = torch.full((B,), L, dtype=torch.int32, device=dev)
    out, ref = torch.empty_like(q), torch.empty_like(q)

    def run(o, stream=None):
        capi.paged_attention_decode(o, q, kc, vc, bt, lens, H, d ** -0.5, stream=stream)

    run(ref)
    size = capi.paged_decode_workspace_size(B, H, H, d, L // 16)
    a = torch.randn(8192, 8192, device=dev).half()
    c = a @ a
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    with torch.cuda.stream(side):
        for _ in range(20):  # about 1 ms each
            torch.matmul(a, a, out=c)
    run(out, side)
    mine = torch.full((size,), 0xff, dtype=torch.uint8, device=dev)
    torch.cuda.synchronize()
    assert (mine == 0xff).all() and torch.equal(out, ref)
