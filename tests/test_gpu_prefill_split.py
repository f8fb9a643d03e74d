"""Prefill whose tiles' keys are split between two waves (steps that would
leave compute units idle) against steps that are not.

A row's result does not depend on the rest of the step, so the rows of a short
step (split) are compared with the same rows of a long one (whole): the step's
tokens repeated as further sequences until the launch passes the split's
bound.  Both round each weight to fp16 (2^-11 relative, against another
running max), which moves a row by at most 2^-11 max |v - out| <= 2^-10 max |v|
on either side, and the output to 16 bits (one unit apart).
"""
import numpy as np
import pytest

import oracle_lib as O
from kvgen import BS, make_workload

pytestmark = pytest.mark.gpu


def _close(a, b, bf16):
    a, b = a.float().cpu().numpy(), b.float().cpu().numpy()
    err = np.abs(a - b) - (2.0 ** (-7 if bf16 else -10)) * np.abs(b)
    assert np.isfinite(a).all() and err.max() <= 2.0 ** -9 * 5, f"max err {err.max()}"  # |v| < 5


@pytest.mark.parametrize("heads", [(8, 2), (6, 3), (7, 1)])  # 4, 2 and 1 heads a workgroup
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("ws", [False, True])
def test_local(dev, heads, bf16, ws):
    import torch
    from vm_c_amd import capi
    hq, hkv = heads
    dt = torch.bfloat16 if bf16 else torch.float16
    lens = [1, 31, 32, 33, 63, 64, 65, 129, 200]
    t = sum(lens)
    g = torch.Generator(device=dev).manual_seed(4)
    q, k, v = (torch.randn(t, h, 128, generator=g, device=dev).to(dt) for h in (hq, hkv, hkv))
    pos = torch.cat([torch.arange(n, dtype=torch.int32, device=dev) for n in lens])
    reps = 257 * 256 * 8 // (t * hq) + 2

    def run(n):
        qq, kk, vv, pp = (x.repeat((n,) + (1,) * (x.dim() - 1)).contiguous() for x in (q, k, v, pos))
        out = torch.full_like(qq, float("nan"))
        w = torch.empty(max(16, capi.flash_attention_prefill_workspace_size(n * t, hkv, 128)), dtype=torch.uint8,
                        device=dev)
        capi.flash_attention_prefill(out, qq, kk, vv, pp, hkv, 128 ** -0.5, workspace=w if ws else None)
        torch.cuda.synchronize()
        return out

    _close(run(1), run(reps)[:t], bf16)


@pytest.mark.parametrize("fmt", [O.KV_F16, O.KV_BF16, O.KV_Q8_0, O.KV_Q4_0, "turboquant_3bit_nc",
                                 "turboquant_4bit_nc", "turboquant_k3v4_nc", "turboquant_k8v4"])
@pytest.mark.parametrize("heads", [(8, 2), (6, 3), (7, 1)])
def test_paged(dev, fmt, heads):
    import torch
    from vm_c_amd import capi
    hq, hkv = heads
    prefix, new = np.array([0, 31, 100, 513]), np.array([33, 17, 64, 30])
    lens = prefix + new
    w = make_workload(lens, Hq=hq, Hkv=hkv, seed=9, holes=3)
    tq = isinstance(fmt, str)
    bf16 = fmt == O.KV_BF16
    dt = torch.bfloat16 if bf16 else torch.float16
    K, V, slots = (torch.from_numpy(x).to(dev) for x in (w.K, w.V, w.slots))
    bt = torch.from_numpy(w.bt).to(dev)
    if tq:
        cfg = capi.tq_config(128, fmt)
        cache = torch.zeros(w.num_blocks * BS * hkv * cfg.slot_size_aligned, dtype=torch.uint8, device=dev)
        capi.turboquant_store(K, V, cache, slots, BS, cfg)
    else:
        kc, vc = (torch.zeros(w.num_blocks * BS * hkv * O.entry_bytes(fmt, 128), dtype=torch.uint8, device=dev)
                  for _ in range(2))
        capi.reshape_and_cache(K.to(dt), V.to(dt), kc, vc, slots, BS, kv_format=fmt)
    seq = torch.from_numpy(np.repeat(np.arange(4), new).astype(np.int32)).to(dev)
    pos = torch.from_numpy(np.concatenate([np.arange(a, b) for a, b in zip(prefix, lens)]).astype(np.int32)).to(dev)
    t = len(pos)
    q = torch.randn(t, hq, 128, generator=torch.Generator(device=dev).manual_seed(5), device=dev).to(dt)
    reps = 257 * 256 * 8 // (t * hq) + 2

    def run(n):
        qq, ss, pp = q.repeat(n, 1, 1), seq.repeat(n), pos.repeat(n)
        out = torch.full_like(qq, float("nan"))
        if tq:
            capi.turboquant_prefill_attention(out, qq, cache, bt, ss, pp, hkv, float(w.scale), cfg, block_size=BS)
        else:
            capi.flash_attention_prefill_v2(out, qq, kc, vc, bt, ss, pp, hkv, float(w.scale), block_size=BS,
                                            kv_format=fmt)
        torch.cuda.synchronize()
        return out

    _close(run(1), run(reps)[:t], bf16)
