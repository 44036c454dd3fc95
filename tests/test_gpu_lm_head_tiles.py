"""The wide-batch LM head kernel (more than 64 rows of a packed weight, more
than 128 of a plain one) at the edges of its tiles, in passes of 128 rows and of
256: one and several passes, vocabularies that end inside a tile, a key slot or
a 32-row block, more units than workgroups (the request streams run on into the
next unit) and the shortest k (one chunk of 64 ids).  Each case says which of
the two it is meant for, and the kernel that ran is looked up."""
import re

import numpy as np
import pytest

from llima_amd import workloads as wl
from .test_gpu_parity import _lm_head_check, _np, _say, _score_check, _t, torch_i32

pytestmark = pytest.mark.gpu


def _tile_rows(call):
    """The hidden rows per pass of the wide-batch kernels that call launches."""
    import torch
    from torch.profiler import ProfilerActivity, profile
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        call()
        torch.cuda.synchronize()
    return {int(m.group(1)) for e in prof.key_averages() if (m := re.search(r"lmh_tiles<(\d+)", e.key))}


# (rows per pass, B, H, V, softcap, packed): 257 tiles x 1 pass, 129 x 2 and
# 86 x 3 are more units than the 256 workgroups.
CASES = [(128, 65, 256, 255, 0.0, True), (128, 128, 512, 257, 30.0, True),
         (128, 100, 256, 65793, 0.0, True), (128, 129, 64, 256, 0.0, False),
         (128, 256, 128, 300, 30.0, False), (128, 257, 320, 2053, 0.0, False),
         (256, 300, 256, 33000, 0.0, True), (256, 520, 64, 22000, 0.0, False),
         (128, 129, 256, 2049, 0.0, True), (256, 200, 256, 33001, 30.0, False),
         (256, 257, 320, 32772, 0.0, False), (256, 129, 512, 32801, 30.0, True),
         (256, 513, 256, 11008, 0.0, False)]


@pytest.mark.parametrize("rows,B,H,V,cap,packed", CASES)
def test_tiles_against_float64_and_narrow_passes(gpu, oracle, rows, B, H, V, cap, packed):
    """Logits within the fp32 sum's bound of the float64 product, ids exact for
    them; the same bits as passes of at most 64 rows over the packed weight
    give; bf16 output and scoring over the same logits."""
    import torch
    import llima_amd
    _say("lm head tiles", rows, B, H, V, cap, packed)
    rng = np.random.default_rng(B + 3 * H + V)
    x = wl.f32_to_bf16_bits(rng.normal(0, 1, (B, H)).astype(np.float32))
    w = wl.f32_to_bf16_bits(rng.normal(0, 3.0 / np.sqrt(H), (V, H)).astype(np.float32))
    xt, pt = _t(x, gpu), _t(w, gpu)
    wt = llima_amd.lm_head_pack(pt) if packed else pt
    assert _tile_rows(lambda: llima_amd.lm_head_argmax(xt, wt, softcap=cap)) == {rows}
    for ld in ("bf16", "f32"):
        ids, vals, lg = llima_amd.lm_head_argmax(xt, wt, softcap=cap, return_logits=True,
                                                 logit_dtype=ld)
        _lm_head_check(_np(ids), _np(vals), _np(lg), x, w, cap, bf16=ld == "bf16")
        i2, v2 = llima_amd.lm_head_argmax(xt, wt, softcap=cap, logit_dtype=ld)
        assert torch.equal(i2, ids) and torch.equal(v2, vals)
        targets = rng.integers(0, V, B).astype(np.int32)
        targets[::2] = _np(ids)[::2]
        lp, g = llima_amd.lm_head_score(xt, wt, torch_i32(targets, gpu), softcap=cap,
                                        logit_dtype=ld)
        _score_check(_np(lp), _np(g), _np(lg), targets, oracle)
        if ld == "bf16":
            i3, _, l3 = llima_amd.lm_head_argmax(xt, wt, softcap=cap, return_logits=True,
                                                 logits_out="bf16")
            assert torch.equal(l3.float(), lg) and torch.equal(i3, ids)
        if H % 256 == 0:
            pk = wt if packed else llima_amd.lm_head_pack(pt)
            for r in range(0, B, 64):
                _, _, part = llima_amd.lm_head_argmax(xt[r:r + 64], pk, softcap=cap,
                                                      return_logits=True, logit_dtype=ld)
                assert torch.equal(part, lg[r:r + 64])


@pytest.mark.parametrize("rows_per_pass,B,V", [(128, 140, 1100), (256, 140, 33001), (256, 300, 17000)])
@pytest.mark.parametrize("packed", [False, True])
def test_tiles_ties_nan_and_infinities(gpu, oracle, packed, rows_per_pass, B, V):
    """Equal vocab rows at both halves of a slot, across slots and across tiles:
    the first index wins; a NaN row gives id 0 and NaN; rows of -inf and NaN
    logits; the scores are the oracle's for the written logits."""
    import llima_amd
    _say("lm head tiles ties", packed, rows_per_pass, B, V)
    rng = np.random.default_rng(11)
    H = 256
    xf = np.abs(rng.normal(0, 1, (B, H))).astype(np.float32)
    wf = rng.normal(0, 0.02, (V, H)).astype(np.float32)
    best = np.full(H, 0.5, np.float32)
    xf[3, 7] = np.nan
    xf[4, 0] = np.inf                                          # +-inf logits by the weight's sign
    wf[:, 0] = np.where(np.arange(V) % 3 == 0, -1.0, 1.0)
    best[0] = 1.0
    for v in (70, 66, 69, 300, V - 1):                         # lane halves, slots and tiles
        wf[v] = best
    x, w = wl.f32_to_bf16_bits(xf), wl.f32_to_bf16_bits(wf)
    xt, wt = _t(x, gpu), _t(w, gpu)
    wt = llima_amd.lm_head_pack(wt) if packed else wt
    assert _tile_rows(lambda: llima_amd.lm_head_argmax(xt, wt)) == {rows_per_pass}
    ids, vals, lg = llima_amd.lm_head_argmax(xt, wt, return_logits=True, logit_dtype="f32")
    ids, vals, lg = _np(ids), _np(vals), _np(lg)
    rows = np.array([b for b in range(B) if b not in (3, 4)])
    assert (ids[rows] == 66).all()
    assert ids[3] == 0 and np.isnan(vals[3])
    assert np.isinf(vals[4]) and ids[4] == int(np.flatnonzero(lg[4] == np.inf)[0])
    targets = rng.integers(0, V, B).astype(np.int32)
    targets[::2] = 66
    lp, g = llima_amd.lm_head_score(xt, wt, torch_i32(targets, gpu), logit_dtype="f32")
    _score_check(_np(lp), _np(g), lg, targets, oracle)
    xf[4] = -1.0                                               # every logit -inf
    wf[:, 0] = np.inf
    x, w = wl.f32_to_bf16_bits(xf), wl.f32_to_bf16_bits(wf)
    wt = _t(w, gpu)
    wt = llima_amd.lm_head_pack(wt) if packed else wt
    ids, vals, lg = llima_amd.lm_head_argmax(_t(x, gpu), wt, return_logits=True, logit_dtype="f32")
    assert int(ids[4]) == 0 and float(vals[4]) == -np.inf and bool((lg[4] == -np.inf).all())


@pytest.mark.parametrize("rows,V", [(128, 520), (256, 33000), (256, 33001)])
@pytest.mark.parametrize("bf16", [False, True])
def test_tiles_logits_output_not_16_byte_aligned(gpu, bf16, rows, V):
    """The C entry point writes the same logits at an address that is aligned to
    its values alone, and nothing beside them."""
    import torch
    import llima_amd
    from llima_amd import _lib
    _say("lm head tiles unaligned logits", bf16, rows, V)
    B, H = 130, 256
    g = torch.Generator(device=gpu).manual_seed(5)
    x = torch.randn(B, H, device=gpu, generator=g).to(torch.bfloat16)
    w = llima_amd.lm_head_pack(torch.randn(V, H, device=gpu, generator=g).to(torch.bfloat16))
    ids, _, lg = llima_amd.lm_head_argmax(x, w, return_logits=True,
                                          logits_out="bf16" if bf16 else "f32")
    assert _tile_rows(lambda: llima_amd.lm_head_argmax(x, w)) == {rows}
    buf = torch.full((B * V + 2,), 7.0, dtype=lg.dtype, device=gpu)
    out_ids = torch.empty(B, dtype=torch.int32, device=gpu)
    L = _lib.lib()
    ws = torch.empty(L.llima_lm_head_argmax_packed_workspace_bytes(B, H, V), dtype=torch.uint8,
                     device=gpu)
    ld = _lib.LLIMA_BF16 | (_lib.LLIMA_LOGITS_OUT_BF16 if bf16 else 0)
    rc = L.llima_lm_head_argmax_packed(x.data_ptr(), w.data.data_ptr(), B, H, V, 0.0, ld,
                                       out_ids.data_ptr(), None, buf[1:].data_ptr(), ws.data_ptr(),
                                       ws.numel(), torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    assert torch.equal(buf[1:-1].reshape(B, V), lg) and torch.equal(out_ids, ids)
    assert float(buf[0]) == 7.0 and float(buf[-1]) == 7.0
