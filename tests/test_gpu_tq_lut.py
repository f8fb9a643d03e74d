"""Tiled prefill over TurboQuant slots of arbitrary codes: the byte-permute
tables that turn a row's codes into fp16 (tq_lut.hpp).

The slots are written here byte by byte, so that every code meets every
position and rows of one code only (the largest and smallest sums of squares
of the norm correction, 128 equal centroids) are among them, with zero norms
and scales.  Checked against the oracle's fp64 attention over the same bytes.
Tolerance as for encoded rows (K, V and the weights are rounded to fp16, 2^-11
relative each, and the rows' values are of the same size): 2e-3 + 1e-2 |ref|.
"""
import numpy as np
import pytest

import oracle_lib as O
from kvgen import BS, close_report, f32_to_bf16_bits, make_workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method", ["turboquant_3bit_nc", "turboquant_4bit_nc", "turboquant_k3v4_nc"])
@pytest.mark.parametrize("bf16,norm_corr", [(False, 1), (True, 1), (False, 0)])
def test_any_codes(dev, method, bf16, norm_corr):
    import torch
    from vm_c_amd import capi
    prefix, new, Hq, Hkv = 307, 33, 8, 2
    w = make_workload([prefix + new], Hq=Hq, Hkv=Hkv, seed=3)
    cfg, L = capi.tq_config(128, method), O.tq_layout(method)
    cfg.norm_correction = L.norm_correction = norm_corr
    rng = np.random.default_rng(17)
    n, kb, vb = w.num_blocks * BS * Hkv, cfg.key_quant_bits, cfg.value_quant_bits
    half = f32_to_bf16_bits if bf16 else (lambda x: x.astype(np.float16).view(np.uint16))

    def put(x):
        return half(x.astype(np.float32))[:, None].view(np.uint8)

    codes = [rng.integers(0, 256, (n, 16 * b), dtype=np.uint8) for b in (kb, vb)]
    for c, b in zip(codes, (kb, vb)):  # rows of one code: bits repeat with the period of a code
        for i, code in enumerate(rng.permutation(1 << b)):
            row = np.tile([(code >> k) & 1 for k in range(b)], 128)
            c[i::41] = np.packbits(row.astype(np.uint8), bitorder="little")
    norm, scale, zero = rng.uniform(0, 16, n), rng.uniform(0, 0.3, n), rng.uniform(-2, 2, n)
    norm[::29], scale[::31] = 0, 0
    slots = np.concatenate([codes[0], put(norm), codes[1], put(scale), put(zero)], 1)
    assert slots.shape[1] == cfg.slot_size_aligned
    cache = np.ascontiguousarray(slots.reshape(-1))
    pos = np.arange(prefix, prefix + new, dtype=np.int32)
    qf = rng.standard_normal((new, Hq, 128)).astype(np.float32)
    qbits = np.ascontiguousarray(half(qf))
    q = torch.from_numpy(qbits.view(np.int16)).to(dev).view(torch.bfloat16 if bf16 else torch.float16)
    out = torch.full_like(q, float("nan"))
    capi.turboquant_prefill_attention(out, q, torch.from_numpy(cache).to(dev), torch.from_numpy(w.bt).to(dev),
                                      torch.zeros(new, dtype=torch.int32, device=dev), torch.from_numpy(pos).to(dev),
                                      Hkv, float(w.scale), cfg, block_size=BS)
    torch.cuda.synchronize()
    c, _ = O.tq_tables(128, kb)
    ex = O.tq_decode_exact(qbits, cache, np.repeat(w.bt, new, 0), pos + 1, Hkv, float(w.scale), BS, L, c, bf16=bf16)
    ok, err = close_report(out.float().cpu().numpy(), ex, 2e-3, 1e-2)
    assert ok, f"max err {err}"
