"""The ctypes binding's host side: what it needs of torch."""
import subprocess
import sys
import types

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
