"""GPU parity of the EAGLE3 draft-tree functions against the oracle: the heap
top-k (utils.hpp:216-281) -- indices and their order bit for bit, ties
included -- and the tree build (language_model_eagle3.cpp:808-1164) level by
level: input ids, parent rows, draft masks, then the final tokens, tree mask,
position ids and retrieve indices.  The log-softmax scores feed only index
decisions, so those are compared exactly; the oracle runs with the same
correctly rounded exp/log as the kernels (its C-library variant is checked
against this one on the CPU)."""
import numpy as np
import pytest

from llima_amd import workloads as wl

pytestmark = pytest.mark.gpu


def _say(*a):
    print("[gpu-case]", *a, flush=True)


def _t(a, dev):
    import torch
    if a.dtype == np.uint16:
        return torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).to(dev).view(torch.bfloat16)
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def _np(t):
    return t.cpu().numpy()


def _rows(kind, rows, cols, rng):
    if kind == "normal":
        return rng.normal(0, 3, (rows, cols)).astype(np.float32)
    if kind == "ties":                                   # a handful of distinct values
        return rng.integers(-6, 7, size=(rows, cols)).astype(np.float32)
    if kind == "ascending":                              # every value enters the heap
        return np.tile(np.arange(cols, dtype=np.float32), (rows, 1))
    if kind == "specials":
        x = rng.normal(0, 2, (rows, cols)).astype(np.float32)
        hit = rng.random((rows, cols)) < 0.01
        x[hit] = rng.choice(np.array([np.nan, -np.inf, np.inf, 0.0, -0.0], np.float32), hit.sum())
        x[0, 1] = np.nan                                 # a NaN among the first k: replay everything
        return x
    raise ValueError(kind)


CASES = [("normal", 5, 32000), ("ties", 5, 32000), ("normal", 1, 1000), ("ties", 15, 80),
         ("ties", 32, 5000), ("normal", 5, 128256), ("ties", 5, 70001), ("ascending", 5, 20000),
         ("specials", 5, 40000), ("specials", 3, 300), ("normal", 7, 7), ("ties", 16, 262144)]


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("kind,k,cols", CASES)
def test_topk_heap_order(gpu, oracle, dtype, kind, k, cols):
    import llima_amd
    _say("topk", kind, k, cols, dtype)
    rng = np.random.default_rng(k * 1000 + cols)
    x = _rows(kind, 4, cols, rng)
    if dtype == "bf16":
        x = wl.f32_to_bf16_bits(x)
    idx, val = llima_amd.topk(_t(x, gpu), k)
    eidx, evals = oracle.topk(x, k)
    assert (_np(idx) == eidx).all(), (_np(idx)[:2], eidx[:2])
    g = _np(val)
    assert ((g.view(np.uint32) == evals.view(np.uint32)) | (np.isnan(g) & np.isnan(evals))).all()


def test_topk_strided_rows(gpu, oracle):
    import llima_amd
    _say("topk strided")
    rng = np.random.default_rng(2)
    x = rng.integers(-5, 6, size=(3, 5003)).astype(np.float32)
    xt = _t(x, gpu)[:, 1:5000]
    idx, _ = llima_amd.topk(xt, 5)
    assert (_np(idx) == oracle.topk(np.ascontiguousarray(x[:, 1:5000]), 5)[0]).all()


def _run_tree(gpu, oracle, root, levels, d2t, K, depth, total, sample, pad=0):
    import llima_amd
    tree = llima_amd.Eagle3DraftTree(_t(d2t, gpu), topk=K, depth=depth)
    e = oracle.eagle3_tree(root, levels, d2t, K, depth, total, sample, cr=True)
    ids = tree.begin(_t(root, gpu))
    assert (_np(ids) == e["inputs"][0]).all()
    for lv in range(1, depth):
        rows = levels[lv - 1]
        if pad:                                          # a slice of wider rows
            rows = np.concatenate([rows, np.full((K, pad), rows.max(), rows.dtype)], axis=1)
        ids, prow, mask = tree.grow(_t(rows, gpu)[:, :levels.shape[2]])
        assert (_np(ids) == e["inputs"][lv]).all(), lv
        assert (_np(prow) == e["parent_rows"][lv - 1]).all(), lv
        assert (_np(mask) == e["masks"][lv - 1][:, :K * (lv + 1)]).all(), lv
    # the node scores themselves (log-softmax plus the parent's score), to 1e-5
    # relative: the kernels and this oracle round exp/log the same way, so they
    # agree far closer than that
    ns = _np(tree.node_scores())
    assert ns.shape == e["node_scores"].shape
    assert np.allclose(ns, e["node_scores"], rtol=1e-5, atol=1e-6, equal_nan=True)
    out = tree.finish(total, sample)
    assert (_np(out["tokens"]) == e["tokens"]).all()
    assert (_np(out["tree_mask"]) == e["tree_mask"]).all()
    assert (_np(out["position_ids"]) == e["position_ids"]).all()
    assert _np(out["retrieve"]).tolist() == e["retrieve"].tolist()
    return e


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("seed", range(3))
def test_eagle3_tree_llama3_draft(gpu, oracle, dtype, seed):
    """The reference's EAGLE3 shape: K = 5, depth 4, 15 draft tokens, a 32000-id
    draft vocabulary mapped to the 128256-id target vocabulary."""
    _say("eagle3 tree", dtype, seed)
    rng = np.random.default_rng(500 + seed)
    K, depth, total, Vd = 5, 4, 15, 32000
    root = rng.normal(0, 3, Vd).astype(np.float32)
    levels = rng.normal(0, 3, (depth - 1, K, Vd)).astype(np.float32)
    if dtype == "bf16":
        root, levels = wl.f32_to_bf16_bits(root), wl.f32_to_bf16_bits(levels)
    d2t = (np.sort(rng.choice(128256, Vd, replace=False)) - np.arange(Vd)).astype(np.int32)
    _run_tree(gpu, oracle, root, levels, d2t, K, depth, total, sample=int(rng.integers(0, 128256)))


def test_eagle3_tree_ties_and_shapes(gpu, oracle):
    """Integer-valued logits (ties in the heaps and in the cumulative scores),
    identical rows, and other (K, depth, total) shapes."""
    rng = np.random.default_rng(77)
    for K, depth, total, Vd in [(5, 4, 15, 32000), (2, 2, 3, 64), (8, 5, 32, 9000), (1, 3, 2, 100),
                                (5, 1, 4, 500), (32, 2, 32, 4096)]:
        _say("eagle3 tree ties", K, depth, total, Vd)
        root = rng.integers(-3, 4, Vd).astype(np.float32)
        levels = rng.integers(-3, 4, (max(depth - 1, 1), K, Vd)).astype(np.float32)[:depth - 1]
        if depth > 1 and K > 1:
            levels[0, 1] = levels[0, 0]                  # identical rows
        d2t = rng.integers(0, 1000, Vd).astype(np.int32)
        _run_tree(gpu, oracle, wl.f32_to_bf16_bits(root), wl.f32_to_bf16_bits(levels)
                  if depth > 1 else np.zeros((0, K, Vd), np.uint16), d2t, K, depth, total, 3)


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("kind", ["normal", "integers", "ascending", "descending", "nan_first",
                                  "nan_later", "inf", "zeros"])
def test_eagle3_split_rows_heap_order(gpu, oracle, dtype, kind):
    """Rows split into parts of 4096 values: the root row's ids are the
    oracle's heap top-k for every k of the register heap, at the edges of a
    part, with ties, with more candidates than a part stores (ascending rows)
    and with NaN among the first k values or after them."""
    import torch
    import llima_amd
    rng = np.random.default_rng(41)
    for k, cols in [(1, 1), (2, 4095), (5, 4096), (5, 4097), (8, 12289), (9, 32001), (13, 8192),
                    (16, 40007), (5, 262145)]:
        _say("eagle3 split rows", dtype, kind, k, cols)
        x = rng.normal(0, 3, cols).astype(np.float32)
        if kind == "integers":
            x = rng.integers(-3, 4, cols).astype(np.float32)
        elif kind in ("ascending", "descending"):
            x = np.sort(x)[::1 if kind == "ascending" else -1].copy()
        elif kind == "nan_first":
            x[min(k - 1, 2)] = np.nan
        elif kind == "nan_later":
            x[k::7] = np.nan
        elif kind == "inf":
            x[::3], x[1::3] = np.inf, -np.inf
        elif kind == "zeros":
            x = np.where(rng.random(cols) < 0.5, 0.0, -0.0).astype(np.float32)
        xb = wl.f32_to_bf16_bits(x) if dtype == "bf16" else x
        tree = llima_amd.Eagle3DraftTree(torch.zeros(cols, dtype=torch.int32, device=gpu), topk=k,
                                         depth=1)
        pad = torch.cat([torch.zeros(1, dtype=_t(xb, gpu).dtype, device=gpu), _t(xb, gpu)])
        expect = oracle.topk(xb[None], k)[0][0]
        assert (_np(tree.begin(_t(xb, gpu))) == expect).all()
        assert (_np(tree.begin(pad[1:])) == expect).all()          # not 16-byte aligned


@pytest.mark.parametrize("K,depth,total,Vd", [(3, 6, 32, 64000), (9, 3, 32, 8191), (10, 4, 20, 12288),
                                              (16, 2, 32, 4097), (17, 2, 20, 5000), (4, 2, 9, 262145)])
def test_eagle3_tree_split_rows_shapes(gpu, oracle, K, depth, total, Vd):
    """Whole trees around the limits of the split rows (k 16, 64 parts)."""
    _say("eagle3 split tree", K, depth, total, Vd)
    rng = np.random.default_rng(K * Vd)
    root = wl.f32_to_bf16_bits(rng.normal(0, 3, Vd).astype(np.float32))
    levels = wl.f32_to_bf16_bits(rng.normal(0, 3, (depth - 1, K, Vd)).astype(np.float32))
    d2t = rng.integers(0, 1000, Vd).astype(np.int32)
    _run_tree(gpu, oracle, root, levels, d2t, K, depth, total, 3)


def test_eagle3_tree_state_sizes(gpu, oracle):
    """A state of llima_eagle3_tree_bytes (no room for split rows' candidates),
    one byte short of room, exactly large enough, and one that is only 4-byte
    aligned give the same tree, and nothing is written past their end."""
    import torch
    from llima_amd._lib import LLIMA_BF16, check, lib
    L = lib()
    rng = np.random.default_rng(9)
    K, depth, total, Vd = 5, 3, 12, 9001
    root = wl.f32_to_bf16_bits(rng.normal(0, 3, Vd).astype(np.float32))
    levels = wl.f32_to_bf16_bits(rng.normal(0, 3, (depth - 1, K, Vd)).astype(np.float32))
    d2t = rng.integers(0, 1000, Vd).astype(np.int32)
    e = oracle.eagle3_tree(root, levels, d2t, K, depth, total, 3, cr=True)
    xr, xl, d2 = _t(root, gpu), _t(levels, gpu), _t(d2t, gpu)
    small, split = L.llima_eagle3_tree_bytes(K, depth), L.llima_eagle3_tree_split_bytes(K, depth, Vd)
    N, sp = total + 1, torch.cuda.current_stream(gpu).cuda_stream
    for nb, off in ((small, 0), (split - 1, 0), (split, 0), (split, 4)):
        _say("eagle3 tree state", nb, off)
        buf = torch.full((split + 64,), 0xAB, dtype=torch.uint8, device=gpu)
        state = buf[off:].data_ptr()
        i32 = lambda *s: torch.empty(s, dtype=torch.int32, device=gpu)
        ids, prow, tok, pos, ret, dims = i32(K), i32(K), i32(N), i32(N), i32(N, N), i32(2)
        mask = torch.empty(K * K * depth, device=gpu)
        tmask = torch.empty(N, N, device=gpu)
        check(L.llima_eagle3_tree_begin(xr.data_ptr(), LLIMA_BF16, Vd, d2.data_ptr(), K, depth, state,
                                        nb, ids.data_ptr(), sp), "begin")
        assert (_np(ids) == e["inputs"][0]).all()
        for lv in range(1, depth):
            check(L.llima_eagle3_tree_grow(xl[lv - 1].data_ptr(), LLIMA_BF16, Vd, Vd, d2.data_ptr(), K,
                                           depth, lv, state, nb, ids.data_ptr(), prow.data_ptr(),
                                           mask.data_ptr(), sp), "grow")
            assert (_np(ids) == e["inputs"][lv]).all() and (_np(prow) == e["parent_rows"][lv - 1]).all()
        check(L.llima_eagle3_tree_finish(state, nb, K, depth, total, 3, tok.data_ptr(), tmask.data_ptr(),
                                         pos.data_ptr(), ret.data_ptr(), dims.data_ptr(), sp), "finish")
        assert (_np(tok) == e["tokens"]).all() and (_np(tmask) == e["tree_mask"]).all()
        # rows are not split in the smaller states: the candidate slots stay as they were
        end = off + (split if nb == split and off == 0 else small)
        assert bool((buf[end:] == 0xAB).all())


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_eagle3_split_rows_nan_heaps(gpu, oracle, dtype):
    """NaNs at any places of the first k values, which fix parts of the heap,
    with ties and more NaNs behind them: the candidates of the parts hold every
    value that the reference's float compares let in."""
    import torch
    import llima_amd
    rng = np.random.default_rng(12)
    for k, cols in [(2, 4097), (3, 9000), (5, 32000), (7, 4096), (8, 12289), (11, 9000), (16, 8193)]:
        tree = llima_amd.Eagle3DraftTree(torch.zeros(cols, dtype=torch.int32, device=gpu), topk=k,
                                         depth=1)
        masks = [1 << i for i in range(k)] + [int(m) for m in rng.integers(1, 1 << k, 12)] + [(1 << k) - 1]
        for m in masks:
            _say("eagle3 nan heap", dtype, k, cols, bin(m))
            x = (rng.normal(0, 3, cols) if m & 1 else rng.integers(-9, 10, cols)).astype(np.float32)
            if m % 3 == 0:
                x = np.sort(x)                             # more candidates than a part stores
            x[:k][[(m >> i) & 1 == 1 for i in range(k)]] = np.nan
            x[k::11] = np.nan
            xb = wl.f32_to_bf16_bits(x) if dtype == "bf16" else x
            assert (_np(tree.begin(_t(xb, gpu))) == oracle.topk(xb[None], k)[0][0]).all()


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("K,Vd,pad", [(5, 9001, 0), (5, 12288, 7), (10, 8200, 8), (16, 4160, 3), (16, 9000, 0)])
def test_eagle3_split_rows_mixed_levels(gpu, oracle, dtype, K, Vd, pad):
    """Levels whose rows differ in kind: one ascending (more candidates than a
    part stores), one with NaNs among its first k, one of infinities, one of
    ties, one flat, the rest normal, each replayed by a wavefront of its own;
    with rows wider apart than Vd and not 16-byte aligned."""
    _say("eagle3 mixed levels", dtype, K, Vd, pad)
    rng = np.random.default_rng(K * Vd + pad)
    depth, total = 3, 20
    root = rng.normal(0, 3, Vd).astype(np.float32)
    levels = rng.normal(0, 3, (depth - 1, K, Vd)).astype(np.float32)
    for lv in range(depth - 1):
        at = rng.permutation(K)[:5]
        levels[lv, at[0]] = np.sort(levels[lv, at[0]])
        levels[lv, at[1], rng.integers(0, K, 2)] = np.nan
        levels[lv, at[2], ::5] = -np.inf
        levels[lv, at[2], Vd // 2] = np.inf
        levels[lv, at[3]] = rng.integers(-3, 4, Vd)
        levels[lv, at[4]] = 0.5
    if dtype == "bf16":
        root, levels = wl.f32_to_bf16_bits(root), wl.f32_to_bf16_bits(levels)
    d2t = rng.integers(0, 1000, Vd).astype(np.int32)
    _run_tree(gpu, oracle, root, levels, d2t, K, depth, total, 3, pad=pad)
