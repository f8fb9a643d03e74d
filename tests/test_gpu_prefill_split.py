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


# one block of rows and one head a workgroup (128 rows or fewer: the keys stay
# whole over this step's K/V and 4-bit values), and one row more, against fp64;
# tolerance as the oracle comparisons of the two paths
@pytest.mark.parametrize("t", [1, 33, 128, 129])
@pytest.mark.parametrize("fmt", [None, "turboquant_4bit_nc", "turboquant_3bit_nc"])
def test_one_block(dev, fmt, t):
    import torch
    from kvgen import close_report
    from vm_c_amd import capi
    hq, hkv, prefix = 7, 1, 0 if fmt is None else 300
    t = max(t, 17) if fmt else t  # shorter steps over slots take decode rows
    w = make_workload([prefix + t], Hq=hq, Hkv=hkv, seed=t)
    K, V = (torch.from_numpy(x.astype(np.float32)).to(dev).half() for x in (w.K, w.V))
    pos = torch.arange(prefix, prefix + t, dtype=torch.int32, device=dev)
    q = torch.randn(t, hq, 128, generator=torch.Generator(device=dev).manual_seed(6), device=dev).half()
    out = torch.full_like(q, float("nan"))
    bits = lambda x: np.ascontiguousarray(x.cpu().numpy().view(np.uint16))  # noqa: E731
    if fmt is None:
        capi.flash_attention_prefill(out, q, K, V, pos, hkv, float(w.scale))
        ex = O.prefill_exact_rows(bits(q), bits(K), bits(V), np.asarray([0, t]), hkv, float(w.scale),
                                  np.repeat(np.arange(t), hq), np.tile(np.arange(hq), t), is_bf16=False)
    else:
        cfg, L = capi.tq_config(128, fmt), O.tq_layout(fmt)
        cache = torch.zeros(w.num_blocks * BS * hkv * cfg.slot_size_aligned, dtype=torch.uint8, device=dev)
        capi.turboquant_store(K, V, cache, torch.from_numpy(w.slots).to(dev), BS, cfg)
        capi.turboquant_prefill_attention(out, q, cache, torch.from_numpy(w.bt).to(dev),
                                          torch.zeros(t, dtype=torch.int32, device=dev), pos, hkv, float(w.scale), cfg,
                                          block_size=BS)
        c, _ = O.tq_tables(128, cfg.key_quant_bits)
        ex = O.tq_decode_exact(bits(q), cache.cpu().numpy(), np.repeat(w.bt, t, 0), pos.cpu().numpy() + 1, hkv,
                               float(w.scale), BS, L, c, bf16=False)
    torch.cuda.synchronize()
    ok, err = close_report(out.float().cpu().numpy().reshape(ex.shape), ex, 2e-3, 1e-2)
    assert ok, f"max err {err}"
