"""Paged decode of head_dim 64 and 256 on MFMA (paged_decode_hd.hip) against the
one-wave-per-row kernel (generic_attn.hip), which an output that is not
16-byte aligned still takes.  Both hold weights and sums to fp32, so the rows
may differ by one rounding of the 16-bit output (2^-10 fp16, 2^-7 bf16,
relative) plus fp32 noise near zero (2e-5 of values of order 1).
"""
import numpy as np
import pytest

from kvgen import BS, make_workload

pytestmark = pytest.mark.gpu

F16, BF16, Q8, Q4 = 0, 1, 2, 3
# (format, q type): the combinations the MFMA kernel takes
TYPES = [(F16, "f16"), (BF16, "bf16"), (Q8, "f16"), (Q8, "bf16"), (Q4, "f16"), (Q4, "bf16")]
# page edges, one-token and empty sequences, one long enough for several ranges and block-table chunks
LENS = [1, 16, 0, 17, 31, 33, 1500, 64, 0, 257]


def _setup(dev, d, heads, fmt, qt, hnd, lens=LENS, seed=0, edit=None):
    import torch
    from vm_c_amd import capi
    dt = torch.bfloat16 if qt == "bf16" else torch.float16
    Hq, Hkv = heads
    lens = np.asarray(lens, np.int32)
    w = make_workload(lens, Hq=Hq, Hkv=Hkv, D=d, seed=seed + d, holes=1, pool_slack=2)
    K, V, Q = (torch.from_numpy(np.asarray(x).astype(np.float32)).to(dev).to(dt) for x in (w.K, w.V, w.Q))
    if edit:
        edit(w, K, V, Q)
    layout = capi.LAYOUT_HND if hnd else capi.LAYOUT_NHD
    n = w.num_blocks * BS * Hkv * capi.kv_entry_bytes(fmt, d)
    kc, vc = (torch.full((n,), 0xff, dtype=torch.uint8, device=dev) for _ in range(2))  # unwritten bytes are NaNs
    capi.reshape_and_cache(K, V, kc, vc, torch.from_numpy(w.slots).to(dev), BS, kv_format=fmt, layout=layout)
    args = (kc, vc, torch.from_numpy(w.bt).to(dev))
    kw = dict(block_size=BS, kv_format=fmt, layout=layout)
    return w, Q, args, torch.from_numpy(lens).to(dev), Hkv, float(w.scale), kw


def _both(Q, run):
    """run(out) into an aligned output (MFMA) and into one 8 bytes past a 16-byte boundary (one wave per row)."""
    import torch
    out = torch.full_like(Q, float("nan"))
    flat = torch.full((Q.numel() + 8,), float("nan"), dtype=Q.dtype, device=Q.device)
    ref = flat[4:4 + Q.numel()].view(Q.shape)
    assert out.data_ptr() % 16 == 0 and ref.data_ptr() % 16 == 8
    run(out)
    run(ref)
    torch.cuda.synchronize()
    return out.float(), ref.float(), 2.0 ** (-7 if Q.dtype == torch.bfloat16 else -10)


def _close(got, ref, ulp, atol=2e-5):
    import torch
    bad = ~((got - ref).abs() <= atol + ulp * ref.abs())  # a NaN or an infinity on one side is bad too
    bad &= ~((got == ref) | (got.isnan() & ref.isnan()))
    assert not bad.any(), f"{int(bad.sum())} values differ, first at {torch.nonzero(bad)[0].tolist()}: " \
                          f"{got[bad][0].item()} vs {ref[bad][0].item()}"


@pytest.mark.parametrize("d", [64, 256])
@pytest.mark.parametrize("fmt,qt", TYPES)
@pytest.mark.parametrize("hnd", [False, True])
@pytest.mark.parametrize("splits", [0, 1, 3])
def test_decode_formats(dev, d, fmt, qt, hnd, splits):
    from vm_c_amd import capi
    w, Q, pages, lens, Hkv, scale, kw = _setup(dev, d, (14, 2), fmt, qt, hnd, seed=fmt)
    got, ref, ulp = _both(Q, lambda o: capi.paged_attention_decode(o, Q, *pages, lens, Hkv, scale, max_splits=splits,
                                                                   **kw))
    _close(got, ref, ulp)
    assert (got[2] == 0).all() and (got[8] == 0).all()


# the smallest and largest group of query heads, KV head counts that are not a
# power of two or pass the tuned d = 128 kernels' 8; a negative scale
@pytest.mark.parametrize("d", [64, 256])
@pytest.mark.parametrize("heads", [(1, 1), (16, 1), (3, 3), (40, 10)])
def test_decode_heads(dev, d, heads):
    from vm_c_amd import capi
    w, Q, pages, lens, Hkv, scale, kw = _setup(dev, d, heads, BF16, "bf16", False, seed=9)
    for sc in (scale, -scale):
        got, ref, ulp = _both(Q, lambda o: capi.paged_attention_decode(o, Q, *pages, lens, Hkv, sc, **kw))
        _close(got, ref, ulp)


# no workspace, and one with room for a few ranges only: accepted as before
@pytest.mark.parametrize("d", [64, 256])
@pytest.mark.parametrize("rows", [0, 1, 7, 24])
def test_decode_small_workspace(dev, d, rows):
    import torch
    from vm_c_amd import capi
    w, Q, pages, lens, Hkv, scale, kw = _setup(dev, d, (8, 2), F16, "f16", False, seed=11)
    ws = torch.empty(max(1, rows * 2 * 8 * (d + 4) * 4), dtype=torch.uint8, device=dev)
    got, ref, ulp = _both(Q, lambda o: capi.paged_attention_decode(o, Q, *pages, lens, Hkv, scale, workspace=ws, **kw))
    _close(got, ref, ulp)


# prefill rows: many rows of one sequence
@pytest.mark.parametrize("d", [64, 256])
@pytest.mark.parametrize("splits", [0, 1])
def test_prefill_rows(dev, d, splits):
    import torch
    from vm_c_amd import capi
    w, _, pages, lens, Hkv, scale, kw = _setup(dev, d, (8, 2), Q8, "bf16", True, seed=12)
    seq = np.repeat([6, 9, 0], [70, 5, 1]).astype(np.int32)
    pos = np.concatenate([np.arange(1430, 1500), np.arange(252, 257), [0]]).astype(np.int32)
    g = torch.Generator().manual_seed(d)
    Q = torch.randn((len(seq), 8, d), generator=g).to(dev).to(torch.bfloat16)
    ts, tp = torch.from_numpy(seq).to(dev), torch.from_numpy(pos).to(dev)
    got, ref, ulp = _both(Q, lambda o: capi.paged_attention_prefill(o, Q, *pages, ts, tp, Hkv, scale,
                                                                    max_splits=splits, **kw))
    _close(got, ref, ulp)


# rows enough that a merge workgroup takes several heads and scans more than 256
# lengths, and the last and first counts on either side of one range per row
@pytest.mark.parametrize("d", [64, 256])
@pytest.mark.parametrize("rows", [300, 1023, 1024])
def test_many_rows(dev, d, rows):
    import torch
    from vm_c_amd import capi
    w, _, pages, _, Hkv, scale, kw = _setup(dev, d, (14, 2), BF16, "bf16", False, lens=[300, 150, 7], seed=14)
    rng = np.random.default_rng(rows)
    seq = np.sort(rng.integers(0, 3, rows)).astype(np.int32)
    pos = (rng.random(rows) * np.asarray([300, 150, 7])[seq]).astype(np.int32)
    pos[::50] = -1  # rows without keys
    g = torch.Generator().manual_seed(d)
    Q = torch.randn((rows, 14, d), generator=g).to(dev).to(torch.bfloat16)
    ts, tp = torch.from_numpy(seq).to(dev), torch.from_numpy(pos).to(dev)
    got, ref, ulp = _both(Q, lambda o: capi.paged_attention_prefill(o, Q, *pages, ts, tp, Hkv, scale, max_splits=0,
                                                                    **kw))
    _close(got, ref, ulp)
    assert (got[::50] == 0).all()


# tables of as many pages as one wave takes without a split, and one more
@pytest.mark.parametrize("d,wide", [(64, 8), (64, 9), (256, 4), (256, 5)])
def test_narrow_table(dev, d, wide):
    from vm_c_amd import capi
    w, Q, pages, lens, Hkv, scale, kw = _setup(dev, d, (8, 2), F16, "f16", False, lens=[16 * wide, 1, 0, 16 * wide - 17],
                                               seed=15)
    assert pages[2].shape[1] == wide
    got, ref, ulp = _both(Q, lambda o: capi.paged_attention_decode(o, Q, *pages, lens, Hkv, scale, **kw))
    _close(got, ref, ulp)
    assert (got[2] == 0).all()


# infinities and NaNs: V of a key whose weight is 0 (alone, and among 20 pages
# of such keys, so that whole pieces are), V of one that counts (the last one
# too), K, q; scores far enough apart that weights underflow.  Whole sequences, and ones
# cut into as many or at most 3 pieces a row: there a piece that met one is
# computed key by key and merged with the others' products
@pytest.mark.parametrize("d", [64, 256])
@pytest.mark.parametrize("fmt,qt", [(F16, "f16"), (BF16, "bf16"), (Q8, "f16")])
@pytest.mark.parametrize("splits", [0, 1, 3])
@pytest.mark.parametrize("what", ["v_unused", "v_far", "v_inf", "v_last", "k_nan", "k_inf", "q_nan", "spread"])
def test_decode_specials(dev, d, fmt, qt, splits, what):
    from vm_c_amd import capi

    def edit(w, K, V, Q):
        row = int(np.asarray([1, 16, 0, 17, 31, 33]).sum()) + 40  # token 40 of the 1500-token sequence
        if what == "v_unused":
            K[row, 0, :] = -30 * Q[6, 0, :].sign()
            V[row, 0, 3] = float("inf")
        elif what == "v_far":
            K[row + 280:row + 600, 0, :] = -30 * Q[6, 0, :].sign()
            V[row + 400, 0, 3] = float("inf")
        elif what == "v_last":
            V[row - 40 + 1499, 0, 3] = float("inf")
        elif what == "v_inf":
            V[row, 0, 3] = float("inf")
        elif what == "k_nan":
            K[row, 0, 3] = float("nan")
        elif what == "k_inf":
            K[row, 0, 3] = float("inf")
        elif what == "q_nan":
            Q[6, 1, 3] = float("nan")
        else:
            Q.mul_(8.0)

    w, Q, pages, lens, Hkv, scale, kw = _setup(dev, d, (4, 2), fmt, qt, False, seed=13, edit=edit)
    got, ref, ulp = _both(Q, lambda o: capi.paged_attention_decode(o, Q, *pages, lens, Hkv, scale, max_splits=splits,
                                                                   **kw))
    # scores of order 100: their fp32 sums differ by up to 2^-24 * 2^7 * a few, and so do the weights, relatively
    _close(got, ref, ulp, atol=2e-4 if what == "spread" else 2e-5)
