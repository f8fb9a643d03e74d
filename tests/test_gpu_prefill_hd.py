"""Local prefill of head_dim 64 and 256 on MFMA (prefill_hd.hip) against the
one-wave-per-row kernel (generic_attn.hip), which an output that is not
16-byte aligned still takes, and against fp64 attention.  Both kernels hold
weights and sums to fp32, so the rows may differ by one rounding of the 16-bit
output (2^-10 fp16, 2^-7 bf16, relative) plus fp32 noise near zero (2e-5 of
values of order 1).
"""
import numpy as np
import pytest

import oracle_lib as O
from kvgen import BS, f32_to_bf16_bits, prefill_inputs
from test_gpu_decode_hd import _both, _close

pytestmark = pytest.mark.gpu


def _inputs(dev, d, heads, seq_lens, bf16, seed=0):
    import torch
    qb, kb, vb, pos, cu = prefill_inputs(seq_lens, *heads, D=d, seed=seed, bf16=bf16)
    dt = torch.bfloat16 if bf16 else torch.float16
    q, k, v = (torch.from_numpy(x.view(np.int16)).to(dev).view(dt) for x in (qb, kb, vb))
    return q, k, v, torch.from_numpy(pos).to(dev), (qb, kb, vb, cu)


# tile and block edges (keys 64, rows 32 .. 256), one-token sequences, several
# sequences in a block and sequences of several tiles; 1, 2, 4, 7 and 8 query
# heads per KV head (head splits 1, 2 and 4 of a workgroup)
@pytest.mark.parametrize("d", [64, 256])
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("heads", [(2, 2), (4, 2), (8, 2), (7, 1), (16, 2)])
@pytest.mark.parametrize("seq_lens", [[1], [17], [25], [64], [65, 63, 1, 1, 200], [31, 300, 33]])
def test_prefill(dev, d, bf16, heads, seq_lens):
    from vm_c_amd import capi
    q, k, v, pos, (qb, kb, vb, cu) = _inputs(dev, d, heads, seq_lens, bf16, seed=d + sum(seq_lens))
    sc = 1 / np.sqrt(d)
    got, ref, ulp = _both(q, lambda o: capi.flash_attention_prefill(o, q, k, v, pos, heads[1], sc))
    _close(got, ref, ulp)
    T = q.shape[0]
    toks, hds = np.repeat(np.arange(T), heads[0]), np.tile(np.arange(heads[0]), T)
    ex = O.prefill_exact_rows(qb, kb, vb, cu, heads[1], sc, toks, hds, is_bf16=bf16).reshape(T, heads[0], d)
    err = np.abs(got.cpu().numpy() - ex)
    assert (err <= 2e-5 + ulp / 2 * np.abs(ex)).all(), float(err.max())


# steps of enough workgroups for the eight-wave kernel (4, 2 and 1 heads a
# workgroup), with an infinity in V of one KV head's early sequence
@pytest.mark.parametrize("d", [64, 256])
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("heads", [(16, 2), (36, 6), (28, 4)])
def test_prefill_long_steps(dev, d, bf16, heads):
    from vm_c_amd import capi
    hw = {8: 4, 6: 2, 7: 1}[heads[0] // heads[1]]
    per_cu = 4 if d == 64 else 1
    rows = (256 * per_cu + 1) * 32 * 4 // heads[0] + 64  # rows x heads / 128 workgroups of four waves
    lens = [31, 300, 33, 65, 1, 200] * (rows // 630 + 1)
    q, k, v, pos, _ = _inputs(dev, d, heads, lens, bf16, seed=hw)
    v[40, 0, 3] = float("inf")
    got, ref, ulp = _both(q, lambda o: capi.flash_attention_prefill(o, q, k, v, pos, heads[1], 1 / np.sqrt(d)))
    _close(got, ref, ulp)


# positions that are not 0 .. n-1 of contiguous sequences: every row's window
# is [t - pos, t], empty below 0
@pytest.mark.parametrize("d", [64, 256])
def test_prefill_any_positions(dev, d):
    import torch
    from vm_c_amd import capi
    q, k, v, pos, _ = _inputs(dev, d, (4, 1), [330], True, seed=5)
    rng = np.random.default_rng(d)
    p = np.minimum(rng.integers(-1, 200, 330), np.arange(330)).astype(np.int32)
    pos = torch.from_numpy(p).to(dev)
    for sc in (1 / np.sqrt(d), -1 / np.sqrt(d), 0.0):
        got, ref, ulp = _both(q, lambda o: capi.flash_attention_prefill(o, q, k, v, pos, 1, sc))
        _close(got, ref, ulp)
        assert (got[torch.from_numpy(p).to(dev) < 0] == 0).all()


# infinities and NaNs in q, K and V (a row sees only its own window's), values
# near the largest of the type (v_late: the sums stay below it only with weights
# of at most 1, and the scores rise by 5 after the first tile, less than moves
# the kernel's reference max), scores far apart
@pytest.mark.parametrize("d", [64, 256])
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("what", ["v_inf", "k_nan", "q_inf", "v_large", "v_late", "spread"])
def test_prefill_specials(dev, d, bf16, what):
    from vm_c_amd import capi
    q, k, v, pos, _ = _inputs(dev, d, (4, 2), [90, 150], bf16, seed=6)
    big = 1e30 if bf16 else 60000.0
    if what == "v_late":
        big = 2.0 ** 121 if bf16 else 60000.0
        v.copy_(big / 8 * v.abs().clamp_(0.5, 8))
        q[:, :, 0], k[:, :, 0], k[90 + 64:, :, 0] = d ** 0.5, 0, 5
    if what == "v_inf":
        v[100, 0, 3] = float("inf")
    elif what == "k_nan":
        k[130, 1, 7] = float("nan")
    elif what == "q_inf":
        q[95, 2, 1] = float("inf")
    elif what == "v_large":
        v.mul_(big / 8).clamp_(-big, big)
    elif what == "spread":
        q.mul_(8.0)
    got, ref, ulp = _both(q, lambda o: capi.flash_attention_prefill(o, q, k, v, pos, 2, 1 / np.sqrt(d)))
    # scores of order 100: their fp32 sums differ by up to 2^-24 * 2^7 * a few, and so do the weights, relatively
    if what == "v_late":
        assert ref.isfinite().all()
    _close(got, ref, ulp, atol=2e-5 * big / 8 if what in ("v_large", "v_late") else 2e-4 if what == "spread" else 2e-5)
