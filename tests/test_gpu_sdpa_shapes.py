"""GPU parity tests of the attention launch shapes and head dims.

bi_sdpa picks a launch shape from the grid (include/bi_testing.h): for
bf16/f16 the prefill "rows" shape (several 16-column tiles per workgroup), the
prefill "shared" shape (one column tile per wave, every key block loaded once
for all waves), one tile, or one tile with the output dims split over 2/4/8
workgroups; for fp32 how many query heads share a workgroup's loads. The reference has a single
launch shape (_attention.py:241-250) and rejects any route switch on query
length (reference ROADMAP.md:91-94), so every shape must give the same bits:

  * every shape, forced through bi_sdpa_with_shape, gives identical bits on the
    same input, for every built (D, V) pair, element type and mask mode;
  * the prefill rows and shared shapes, selected by bi_sdpa itself at the
    shapes they are built for, give each row the bits of that row computed
    alone at query length 1 over its visible keys (a one-tile shape), are
    accurate against the float64 oracle (reference
    tests/test_invariance.py:408-432), and give each other's bits;
  * keys no query row can see (an unwritten cache tail) never reach the
    output, whatever they hold (reference _attention.py:92-98).
"""

import ctypes
import math

import numpy as np
import pytest
import torch

import mlx_batch_invariant as bi
from mlx_batch_invariant import _attention, _lib
from oracle import sdpa as osdpa

from helpers import bits, f64, ndiff, rn

pytestmark = pytest.mark.gpu

LOW = [("float16", torch.float16), ("bfloat16", torch.bfloat16)]
TOL = {"float32": 2e-6, "float16": 5e-3, "bfloat16": 3e-2}
PAIRS = list(_attention.HEAD_DIMS)


def _mask_mode(spec, q, k):
    """(mode, mask, strides, causal_offset) for a mask spec: None, "end"
    (bi mask="causal": row s sees keys i <= N - qL + s), "start" (torch
    is_causal: i <= s) or an additive / boolean tensor."""
    B, H, qL, _ = q.shape
    N = k.shape[2]
    if spec is None:
        return _lib.MASK_NONE, None, (0, 0, 0), 0
    if isinstance(spec, str):
        return _lib.MASK_CAUSAL, None, (0, 0, 0), (N - qL if spec == "end" else 0)
    m, ms, mode = _attention._mask_args(spec, B, H, qL, N, q.dtype)
    return mode, m, ms, 0


def run(q, k, v, spec=None, shape=None, sinks=None):
    mode, m, ms, off = _mask_mode(spec, q, k)
    return _attention._sdpa_eager(q, k, v, 1.0 / math.sqrt(q.shape[-1]), mode, m, ms, off, sinks,
                                  shape)


def shapes_for(dtype, D, V, G):
    """Launch shapes built for the head dims (fp32: those dividing G heads)."""
    L = _lib.lib()
    code = _lib.DTYPE_CODES[dtype]
    out = []
    for s in range(_lib.SDPA_NUM_SHAPES):
        c, w = ctypes.c_int(), ctypes.c_int()
        if L.bi_sdpa_shape_info(D, V, code, s, c, w) != _lib.OK:
            continue
        if dtype == torch.float32 and G % c.value:
            continue
        out.append(s)
    return out


def _masks(B, qL, N, dtype, device, seed):
    g = torch.Generator().manual_seed(seed)
    add = (torch.randn(B, 1, qL, N, generator=g)).to(dtype)
    add[torch.rand(B, 1, qL, N, generator=g) < 0.1] = -float("inf")
    keep = torch.rand(1, 1, qL, N, generator=g) > 0.2
    keep[..., N - max(1, N // 10):] = False  # a padding tail
    return add.to(device), keep.to(device)


@pytest.mark.parametrize("D,V", PAIRS)
def test_every_shape_gives_the_same_bits(cuda, D, V):
    """One input through every launch shape, for each element type and mask
    mode: the bits must not move (the attention analogue of the GEMM's
    test_all_geometries_agree)."""
    B, H, Hkv, qL, N = 2, 16, 2, 40, 300
    for dname, dtype in LOW + [("float32", torch.float32)]:
        q = rn((B, H, qL, D), dtype, 101, device=cuda)
        k = rn((B, Hkv, N, D), dtype, 102, device=cuda)
        v = rn((B, Hkv, N, V), dtype, 103, device=cuda)
        sinks = rn((H,), dtype, 104, device=cuda)
        add, keep = _masks(B, qL, N, dtype, cuda, 105)
        shapes = shapes_for(dtype, D, V, H // Hkv)
        assert len(shapes) >= (2 if dtype == torch.float32 else 3), shapes
        for label, spec, sk in (("none", None, None), ("end", "end", None),
                                ("start", "start", None), ("additive", add, None),
                                ("bool", keep, None), ("sinks", None, sinks)):
            ref = None
            for s in shapes:
                if s == _lib.SDPA_SHARED and label in ("additive", "bool"):
                    # Built without array masks: bi_sdpa never picks it for one.
                    continue
                y = run(q, k, v, spec, shape=s, sinks=sk)
                got = bits(y)
                if ref is None:
                    ref = got
                    assert torch.isfinite(y).all() and bool((y != 0).any())
                else:
                    d = int((got != ref).sum())
                    assert d == 0, "%s D=%d V=%d %s shape %d: %d differ" % (
                        dname, D, V, label, s, d)


def test_short_contexts_through_the_loader_wave_shapes(cuda):
    """Decode at D = V = 128 without an array mask takes the dim-split shapes
    with loader waves, whose chains can hold no block at all (N < 97) or
    different block counts. Contexts of 1 to 129 keys, causal and not, with
    and without sinks: the picked shape gives the bits of the rows and
    one-tile shapes, and a single key returns its value row exactly."""
    H, Hkv, D = 32, 8, 128
    for dname, dtype in LOW:
        for B in (1, 8):
            for N in (1, 5, 32, 33, 97, 100, 129):
                q = rn((B, H, 1, D), dtype, 301 + N, device=cuda)
                k = rn((B, Hkv, N, D), dtype, 302 + N, device=cuda)
                v = rn((B, Hkv, N, D), dtype, 303 + N, device=cuda)
                sinks = rn((H,), dtype, 304, device=cuda)
                shape = _attention.launch_shape(q, k, v)
                assert shape in (_lib.SDPA_SPLIT2, _lib.SDPA_SPLIT4, _lib.SDPA_SPLIT8), (B, N, shape)
                for spec, sk in ((None, None), ("end", None), (None, sinks)):
                    y = run(q, k, v, spec, sinks=sk)
                    case = "%s B=%d N=%d %s sinks=%s shape %d" % (dname, B, N, spec, sk is not None, shape)
                    for forced in (_lib.SDPA_TILE, _lib.SDPA_ROWS):
                        d = int((bits(run(q, k, v, spec, shape=forced, sinks=sk)) != bits(y)).sum())
                        assert d == 0, "%s: forced %d: %d differ" % (case, forced, d)
                    if N == 1 and sk is None:
                        want = v.repeat_interleave(H // Hkv, dim=1)
                        assert np.array_equal(bits(y), bits(want.contiguous())), case


def test_long_contexts_through_the_loader_wave_shapes(cuda):
    """The dim-split shapes with loader waves run their chains as a pipeline
    (a step scores block j while it finishes block j - 1, four slots per wave
    at dim split 4 and 8; one block per step at dim split 2). Over 8192 keys
    (65 steps per chain) and 4099 keys (chains of unequal length, a ragged
    last block), each of them forced gives the one-tile shape's bits,
    without a mask, end-aligned causal and with sinks."""
    H, Hkv, D = 32, 8, 128
    for dname, dtype in LOW:
        for N in (8192, 4099):
            q = rn((2, H, 1, D), dtype, 401 + N, device=cuda)
            k = rn((2, Hkv, N, D), dtype, 402 + N, device=cuda)
            v = rn((2, Hkv, N, D), dtype, 403 + N, device=cuda)
            sinks = rn((H,), dtype, 404, device=cuda)
            for spec, sk in ((None, None), ("end", None), (None, sinks)):
                ref = bits(run(q, k, v, spec, shape=_lib.SDPA_TILE, sinks=sk))
                for forced in (_lib.SDPA_SPLIT2, _lib.SDPA_SPLIT4, _lib.SDPA_SPLIT8):
                    d = int((bits(run(q, k, v, spec, shape=forced, sinks=sk)) != ref).sum())
                    assert d == 0, "%s N=%d %s sinks=%s shape %d: %d differ" % (
                        dname, N, spec, sk is not None, forced, d)


def _oracle_rows(q, k, v, spec, rows, b, dname):
    """float64 and reference-order fp32 results for query rows `rows` of batch
    entry b (every head), each row as a one-row problem."""
    B, H, qL, D = q.shape
    N = k.shape[2]
    qh, kh, vh = f64(q[b:b + 1]), f64(k[b:b + 1]), f64(v[b:b + 1])
    want, fixed = [], []
    for s in rows:
        qs = qh[:, :, s:s + 1]
        mask, off = None, None
        if isinstance(spec, str):
            off = s + (N - qL if spec == "end" else 0)
        elif spec is not None:
            m = spec
            if m.dtype == torch.bool:
                m = torch.where(m, 0.0, -float("inf"))
            m = f64(m)
            mask = m[(0 if m.shape[0] == 1 else b):][:1, :, (s if m.shape[2] > 1 else 0):][:, :, :1]
        want.append(osdpa.sdpa_f64(qs, kh, vh, mask=mask, causal_offset=off))
        fixed.append(osdpa.sdpa_fixed32(qs, kh, vh, mask=mask, causal_offset=off,
                                        out_dtype=dname))
    return np.concatenate(want, axis=2), np.concatenate(fixed, axis=2)


def _alone(q, k, v, spec, b, s):
    """Row s of batch entry b computed alone at query length 1 over the keys it
    can see: causal rows as an unmasked call over their visible prefix, masked
    rows with their own mask row."""
    qL, N = q.shape[2], k.shape[2]
    qs = q[b:b + 1, :, s:s + 1].contiguous()
    if isinstance(spec, str):
        nvis = min(N, s + (N - qL if spec == "end" else 0) + 1)
        return run(qs, k[b:b + 1, :, :nvis], v[b:b + 1, :, :nvis])
    m = spec[(0 if spec.shape[0] == 1 else b):][:1, :, (s if spec.shape[2] > 1 else 0):][:, :, :1]
    return run(qs, k[b:b + 1], v[b:b + 1], m)


ROWS_CASES = [(4, 64), (1, 513), (2, 513), (1, 2048), (2, 2048)]


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("dname,dtype", LOW)
def test_prefill_rows_shape_is_invariant_and_accurate(cuda, dname, dtype, D):
    """The prefill shapes at 32/8 heads: bi_sdpa selects "rows" or (D = 128
    without an array mask, on the larger grids) "shared" for these problems;
    rows 0, middle and last are bitwise equal to the same row computed alone at
    query length 1 (which takes a one-tile shape), and every head of those rows
    is within the reference's float64 bound and no worse than 4x the
    reference-order fp32 restatement (tests:408-432). Where "shared" is built
    (D <= 128, no array mask), it and "rows", forced, give the whole output the
    same bits. Masks: end-aligned causal (mask="causal"), start-aligned causal
    (torch is_causal), additive per row, boolean per row."""
    H, Hkv = 32, 8
    picked = set()
    for B, qL in ROWS_CASES:
        for N in (qL, 4200):
            seed = 1000 * B + qL + N + D
            q = rn((B, H, qL, D), dtype, seed, device=cuda)
            k = rn((B, Hkv, N, D), dtype, seed + 1, device=cuda)
            v = rn((B, Hkv, N, D), dtype, seed + 2, device=cuda)
            add, keep = _masks(B, qL, N, dtype, cuda, seed + 3)
            rows = sorted({0, qL // 2, qL - 1})
            b = B - 1
            for label, spec in (("end", "end"), ("start", "start"), ("additive", add),
                                ("bool", keep)):
                mode = _mask_mode(spec, q, k)[0]
                shape = _attention.launch_shape(q, k, v, mode)
                assert shape in (_lib.SDPA_ROWS, _lib.SDPA_SHARED), (B, qL, D, label, shape)
                picked.add(shape)
                y = run(q, k, v, spec)
                case = "%s D=%d B=%d qL=%d N=%d %s shape %d" % (dname, D, B, qL, N, label, shape)
                assert torch.isfinite(y).all(), case
                if D <= 128 and mode != _lib.MASK_ARRAY:
                    for forced in (_lib.SDPA_ROWS, _lib.SDPA_SHARED):
                        yf = run(q, k, v, spec, shape=forced)
                        d = int((bits(yf) != bits(y)).sum())
                        assert d == 0, "%s: forced shape %d: %d differ" % (case, forced, d)
                for s in rows:
                    alone = _alone(q, k, v, spec, b, s)
                    assert np.array_equal(bits(alone[0, :, 0]), bits(y[b, :, s])), (case, s)
                ours = f64(y[b:b + 1, :, rows])
                want, fixed = _oracle_rows(q, k, v, spec, rows, b, dname)
                scale = max(np.abs(want).max(), 1e-30)
                err = np.abs(ours - want).max() / scale
                err_fixed = np.abs(fixed - want).max() / scale
                assert err < TOL[dname], "%s: %.3e" % (case, err)
                assert err < 4 * err_fixed + 1e-7, "%s: %.3e vs %.3e" % (case, err, err_fixed)
    # bi_sdpa's own choice covers the rows shape everywhere, and the shared
    # shape at D = 128.
    assert _lib.SDPA_ROWS in picked
    assert (_lib.SDPA_SHARED in picked) == (D == 128), picked


@pytest.mark.parametrize("dname,dtype", LOW + [("float32", torch.float32)])
def test_base_moves_in_later_blocks_for_some_columns(cuda, dname, dtype):
    """Scores that rise along the keys for some (row, head) columns and stay
    flat for others: head dim 0 carries k_i[0] = i / 2 and q[0] = a slope of
    0, 0.5, 1 or 1.5 by (row + head) mod 4, so a chain's lazily moved base
    (reference _attention.py:99-114, the online softmax) moves again in later
    blocks for some columns of a wave or workgroup (every block of a chain at
    the steeper slopes, every other block at 0.5) and never after the first
    for the flat ones. A block whose base moves for some columns takes the
    full step for the whole wave, where the others keep m and f = 1. Every
    launch shape gives the same bits, without a mask and end-aligned causal,
    and rows 0, 31 and 63 are no worse than 4x the reference-order fp32
    restatement against float64, and within the float64 bound (bf16, f16;
    fp32 within 2e-5: on these scores the restatement itself exceeds the
    random-input bound of 2e-6)."""
    B, H, Hkv, qL, N, D = 1, 8, 2, 64, 640, 128
    q = rn((B, H, qL, D), torch.float32, 121, std=0.3)
    k = rn((B, Hkv, N, D), torch.float32, 122, std=0.3)
    v = rn((B, Hkv, N, D), dtype, 123, device=cuda)
    slope = ((torch.arange(qL).view(1, 1, qL) + torch.arange(H).view(1, H, 1)) % 4) * 0.5
    q[..., 0] = slope.to(torch.float32)
    k[..., 0] = torch.arange(N, dtype=torch.float32).view(1, 1, N) / 2
    q, k = q.to(dtype).to(cuda), k.to(dtype).to(cuda)
    shapes = shapes_for(dtype, D, D, H // Hkv)
    assert len(shapes) >= (2 if dtype == torch.float32 else 5), shapes
    rows = [0, 31, 63]
    for label, spec in (("none", None), ("end", "end")):
        ref = None
        for sh in shapes:
            y = run(q, k, v, spec, shape=sh)
            case = "%s %s shape %d" % (dname, label, sh)
            assert torch.isfinite(y).all(), case
            if ref is None:
                ref = bits(y)
                ours = f64(y[0:1, :, rows])
                want, fixed = _oracle_rows(q, k, v, spec, rows, 0, dname)
                scale = max(np.abs(want).max(), 1e-30)
                err = np.abs(ours - want).max() / scale
                err_fixed = np.abs(fixed - want).max() / scale
                # fp32: scores in the hundreds, rescaled block after block,
                # take the reference-order restatement past the random-input
                # bound too; the restatement ratio is the check there.
                tol = 2e-5 if dtype == torch.float32 else TOL[dname]
                assert err < tol, "%s: %.3e (restatement %.3e)" % (case, err, err_fixed)
                assert err < 4 * err_fixed + 1e-7, "%s: %.3e vs %.3e" % (case, err, err_fixed)
            else:
                d = int((bits(y) != ref).sum())
                assert d == 0, "%s: %d differ" % (case, d)


def test_key_value_views_spanning_more_than_4_gib(cuda):
    """Key and value views whose rows are 1 MiB apart (the first 128 elements
    of each row of a wider cache), so that from a block's first row to the
    last visible row spans more than 4 GiB: the kernels' per-block buffer
    resources cap their byte count at 2^31 - 1 (a block's own rows lie within
    32 rows). Every bf16 launch shape gives, at decode and at a causal prefill
    chunk, the bits of the same call on compact copies."""
    dtype = torch.bfloat16
    B, H, Hkv, N, D, RS = 1, 8, 1, 4352, 128, 1 << 19
    assert (N - 1) * RS * 2 > 1 << 32
    kc = rn((B, Hkv, N, D), dtype, 131, device=cuda)
    vc = rn((B, Hkv, N, D), dtype, 132, device=cuda)
    kw = torch.zeros(N, RS, dtype=dtype, device=cuda)
    vw = torch.zeros(N, RS, dtype=dtype, device=cuda)
    kw[:, :D] = kc[0, 0]
    vw[:, :D] = vc[0, 0]
    kv, vv = kw[:, :D][None, None], vw[:, :D][None, None]
    assert kv.shape == (B, Hkv, N, D) and kv.stride()[2:] == (RS, 1)
    try:
        for qL, spec in ((1, None), (64, "end")):
            q = rn((B, H, qL, D), dtype, 133 + qL, device=cuda)
            for sh in [None] + shapes_for(dtype, D, D, H // Hkv):
                case = (qL, spec, sh)
                got, want = run(q, kv, vv, spec, shape=sh), run(q, kc, vc, spec, shape=sh)
                assert torch.isfinite(got).all(), case
                assert np.array_equal(bits(got), bits(want)), case
    finally:
        del kw, vw, kv, vv
        torch.cuda.empty_cache()


@pytest.mark.parametrize("dname,dtype", LOW + [("float32", torch.float32)])
def test_unwritten_cache_tail_never_reaches_the_output(cuda, dname, dtype):
    """Keys past every row's causal horizon hold NaN (an unwritten cache tail):
    the output is finite and bitwise equal to the same call with a zero tail,
    for start-aligned causal (torch is_causal over a longer cache) and for a
    cache view k[:, :, :N] whose storage continues with NaN rows (mask="causal",
    aligned to the end of the view), at decode and prefill shapes: the one
    bi_sdpa picks, and the two prefill shapes forced (bf16/f16)."""
    H, Hkv, D, NP = 32, 8, 128, 1200
    for B, qL in ((1, 1), (3, 5), (1, 300), (2, 700)):
        q = rn((B, H, qL, D), dtype, 111, device=cuda)
        k = rn((B, Hkv, NP, D), dtype, 112, device=cuda)
        v = rn((B, Hkv, NP, D), dtype, 113, device=cuda)
        shapes = [None]
        if dtype != torch.float32 and qL > 16:
            shapes += [_lib.SDPA_ROWS, _lib.SDPA_SHARED]
        for shape in shapes:
            case = (dname, B, qL, shape)
            # Start-aligned: row s sees keys 0..s; keys from qL on are never read.
            kn, vn, kz, vz = k.clone(), v.clone(), k.clone(), v.clone()
            kn[:, :, qL:] = float("nan")
            vn[:, :, qL:] = float("nan")
            kz[:, :, qL:] = 0
            vz[:, :, qL:] = 0
            got, want = run(q, kn, vn, "start", shape), run(q, kz, vz, "start", shape)
            assert torch.isfinite(got).all(), case
            assert np.array_equal(bits(got), bits(want)), case
            # End-aligned over a view of the first N rows; storage past N is NaN.
            N = NP - 77
            kn, vn, kz, vz = k.clone(), v.clone(), k.clone(), v.clone()
            kn[:, :, N:] = float("nan")
            vn[:, :, N:] = float("nan")
            kz[:, :, N:] = 0
            vz[:, :, N:] = 0
            got = run(q, kn[:, :, :N], vn[:, :, :N], "end", shape)
            want = run(q, kz[:, :, :N], vz[:, :, :N], "end", shape)
            assert torch.isfinite(got).all(), case
            assert np.array_equal(bits(got), bits(want)), case


@pytest.mark.parametrize("dname,dtype", LOW)
def test_nan_value_hidden_from_some_rows_by_the_causal_mask(cuda, dname, dtype):
    """A NaN value row at key j of a start-aligned causal prefill (qL = N):
    rows s >= j see it and are all NaN in every launch shape; a row s < j
    cannot see it, and is either bitwise its result with a finite value there
    or all NaN, by launch shape and by which rows share its workgroup and
    32-key block (its zero probability multiplies the value: 0 * NaN = NaN).
    So bit parity across shapes holds for finite values of the keys some row
    of the call can see (include/bi.h); the reference skips such a key per
    row (_attention.py:92-98)."""
    B, H, Hkv, D, L, j = 1, 8, 2, 128, 96, 40
    q = rn((B, H, L, D), dtype, 131, device=cuda)
    k = rn((B, Hkv, L, D), dtype, 132, device=cuda)
    v = rn((B, Hkv, L, D), dtype, 133, device=cuda)
    vn = v.clone()
    vn[:, :, j] = float("nan")
    leaked = {}
    for shape in shapes_for(dtype, D, D, H // Hkv):
        want = bits(run(q, k, v, "start", shape)).reshape(B, H, L, D)
        out = run(q, k, vn, "start", shape)
        got = bits(out).reshape(B, H, L, D)
        nan_rows = torch.isnan(out).all(-1).cpu().numpy()
        assert nan_rows[:, :, j:].all(), (dname, shape)
        same = (got == want).all(-1)
        assert (nan_rows | same)[:, :, :j].all(), (dname, shape)
        leaked[shape] = int(nan_rows[:, :, :j].sum())
    # Every matrix-core shape ran (how many rows before j turn NaN is the
    # shape's business; the finite ones are exact).
    assert len(leaked) >= 5, leaked


@pytest.mark.parametrize("D,V", PAIRS)
def test_head_dims_accuracy_and_query_length_invariance(cuda, D, V):
    """Every built (D, V) pair (the reference takes any multiples of 32,
    _attention.py:224-227): accurate against float64 within the reference's
    bounds, and a query row keeps its bits for query lengths 1..17."""
    H, Hkv, N = 8, 2, 777
    for dname, dtype in LOW + [("float32", torch.float32)]:
        k = rn((1, Hkv, N, D), dtype, 121, device=cuda)
        v = rn((1, Hkv, N, V), dtype, 122, device=cuda)
        qf = rn((1, H, 17, D), dtype, 123, device=cuda)
        base = None
        for qL in (1, 2, 9, 16, 17):
            q = qf[:, :, 17 - qL:].contiguous()
            y = run(q, k, v, "end")
            got = bits(y[:, :, -1])
            if base is None:
                base = got
            else:
                assert np.array_equal(got, base), (dname, D, V, qL)
        want = osdpa.sdpa_f64(f64(qf), f64(k), f64(v), causal_offset=N - 17)
        fixed = osdpa.sdpa_fixed32(f64(qf), f64(k), f64(v), causal_offset=N - 17,
                                   out_dtype=dname)
        err = np.abs(f64(y) - want).max() / np.abs(want).max()
        err_fixed = np.abs(fixed - want).max() / np.abs(want).max()
        assert err < TOL[dname], (dname, D, V, err)
        assert err < 4 * err_fixed + 1e-7, (dname, D, V, err, err_fixed)


def test_large_sinks_stay_accurate(cuda):
    """A sink far above every score (up to 12 in natural-log units, where e^-12
    is below f16's smallest normal) must not push the keys' probabilities out
    of the half-precision planes that carry them into the value products: the
    sink enters the fixed-order merge as its own partial, so f16 and bf16 stay
    within the reference's bounds and within 4x the reference-order fp32
    restatement rounded once."""
    H, Hkv, N, D = 8, 2, 500, 128
    for dname, dtype in LOW + [("float32", torch.float32)]:
        q = rn((1, H, 3, D), dtype, 131, std=0.3, device=cuda)
        k = rn((1, Hkv, N, D), dtype, 132, std=0.3, device=cuda)
        v = rn((1, Hkv, N, D), dtype, 133, device=cuda)
        for level in (4.0, 8.0, 12.0):
            sinks = torch.full((H,), level, dtype=dtype, device=cuda)
            y = run(q, k, v, None, sinks=sinks)
            want = osdpa.sdpa_f64(f64(q), f64(k), f64(v), sinks=f64(sinks))
            fixed = osdpa.sdpa_fixed32(f64(q), f64(k), f64(v), sinks=f64(sinks),
                                       out_dtype=dname)
            err = np.abs(f64(y) - want).max() / np.abs(want).max()
            err_fixed = np.abs(fixed - want).max() / np.abs(want).max()
            assert err < TOL[dname], (dname, level, err)
            assert err < 4 * err_fixed + 1e-7, (dname, level, err, err_fixed)


def test_fp32_head_grouping_prefill(cuda):
    """fp32 groups two query heads per workgroup for prefill (more than 16 query
    rows) and four for decode; with causal and additive masks each row keeps
    the bits of the same row computed alone at query length 1."""
    H, Hkv, qL, N, D = 32, 8, 64, 900, 128
    dtype = torch.float32
    q = rn((1, H, qL, D), dtype, 141, device=cuda)
    k = rn((1, Hkv, N, D), dtype, 142, device=cuda)
    v = rn((1, Hkv, N, D), dtype, 143, device=cuda)
    add, keep = _masks(1, qL, N, dtype, cuda, 144)
    assert _attention.launch_shape(q, k, v) == 1  # two heads per workgroup
    for spec in ("end", "start", add, keep):
        y = run(q, k, v, spec)
        for s in (0, 17, qL - 1):
            alone = _alone(q, k, v, spec, 0, s)
            assert np.array_equal(bits(alone[0, :, 0]), bits(y[0, :, s])), s


@pytest.mark.parametrize("D,V", [(128, 128), (64, 64), (256, 256), (576, 512)])
@pytest.mark.parametrize("N", [2047, 2049, 4096, 6200])
def test_segments_give_the_same_bits_in_one_workgroup_or_each_in_its_own(cuda, D, V, N):
    """bf16 / f16: every launch shape that computes its scores and every one that
    reads them from the scores kernel ("split") gives the same bits at contexts
    around 2048 keys and multiples of it: without a mask, causal with sinks, and
    with an additive mask that hides the first 2048 keys or the last 2048 from
    some rows; rows against float64."""
    H, Hkv, qL, B = 8, 2, 5, 2
    for dname, dtype in (("float16", torch.float16), ("bfloat16", torch.bfloat16)):
        q = rn((B, H, qL, D), dtype, 71, device=cuda)
        k = rn((B, Hkv, N, D), dtype, 72, device=cuda)
        v = rn((B, Hkv, N, V), dtype, 73, device=cuda)
        sinks = rn((H,), dtype, 74, std=3.0, device=cuda)
        add = rn((B, 1, qL, N), dtype, 75, device=cuda)
        add[:, :, 0, :2048] = -float("inf")
        add[:, :, 1, -(N % 2048 or 2048):] = -float("inf")
        for mode, mask, ms, sk in ((0, None, (0, 0, 0), None), (1, None, (0, 0, 0), sinks),
                                   (2, add, (qL * N, 0, N), None)):
            outs = {}
            for shape in range(_lib.SDPA_NUM_SHAPES):
                for split in (False, True):
                    try:
                        outs[shape, split] = _attention._sdpa_eager(
                            q, k, v, D ** -0.5, mode, mask, ms, N - qL, sk, shape=shape, split=split)
                    except (ValueError, NotImplementedError):
                        # "shared" takes D = V <= 128 without an array mask, and has no split form.
                        assert shape == _lib.SDPA_SHARED
            base = outs[_lib.SDPA_TILE, False]
            for key, y in outs.items():
                assert ndiff(y, base) == 0, "%s N=%d mode %d shape %d split %s" % (
                    dname, N, mode, key[0], key[1])
            picked = _attention._sdpa_eager(q, k, v, D ** -0.5, mode, mask, ms, N - qL, sk)
            assert ndiff(picked, base) == 0
            bias = None if mask is None else f64(mask)
            if mode == 1:
                vis = np.arange(N)[None, :] <= np.arange(qL)[:, None] + N - qL
                bias = np.where(vis, 0.0, -np.inf)[None, None]
            kk, vv = (np.repeat(f64(t), H // Hkv, axis=1) for t in (k, v))
            s = np.einsum("bhqd,bhnd->bhqn", f64(q), kk) * D ** -0.5
            s = s if bias is None else s + bias
            top = s.max(-1, keepdims=True)
            if sk is not None:
                top = np.maximum(top, f64(sk)[None, :, None, None])
            top = np.maximum(top, -1e30)  # a row whose keys are all hidden is 0
            p = np.exp(s - top)
            den = p.sum(-1, keepdims=True)
            if sk is not None:
                den = den + np.exp(f64(sk)[None, :, None, None] - top)
            want = np.einsum("bhqn,bhnd->bhqd", p / np.maximum(den, 1e-300), vv)
            # p and the output round once each to the element type (relative
            # 2^-9 bf16, 2^-12 f16, per product of the sum): 2-norm within 2.5 of it.
            err = np.linalg.norm(f64(base) - want) / np.linalg.norm(want)
            assert err < 2.5 * 2.0 ** (-9 if dname == "bfloat16" else -12), (dname, N, mode, err)


def _underflowing(B, H, Hkv, qL, N, D, dtype, device, low_block, rest):
    """A problem whose output is a negative product below the fp32 range: key 0
    scores 120 (base 2) above the first key of block `low_block`, and that one
    10 above the second, whose values are -2^-24; all other values are 0 and
    the other keys score `rest`. Every output is -2^-154."""
    q = torch.zeros(B, H, qL, D, dtype=dtype, device=device)
    k = torch.zeros(B, Hkv, N, D, dtype=dtype, device=device)
    v = torch.zeros(B, Hkv, N, D, dtype=dtype, device=device)
    ln2 = math.log(2.0)
    j = 32 * low_block
    q[..., 0] = 1.0
    k[..., 0] = rest * ln2
    k[:, :, 0, 0] = 120 * ln2
    k[:, :, j, 0] = 0
    k[:, :, j + 1, 0] = -10 * ln2
    v[:, :, j + 1] = -2.0 ** -24
    keep = torch.zeros(1, 1, 1, N, dtype=torch.bool, device=device)
    keep[..., [0, j, j + 1]] = True
    return q, k, v, keep


@pytest.mark.parametrize("dname,dtype", LOW)
def test_underflow_gives_the_same_zero_whatever_the_context(cuda, dname, dtype):
    """A negative result below the fp32 range is a zero of the same sign in every
    launch shape, for contexts of any length (the rest hidden by the mask, or
    by the causal bound) and with the scores from either kernel."""
    B, H, Hkv, qL, D = 1, 8, 2, 5, 128
    zero = {}
    for low_block in (3, 2, 67):  # the last chain, an earlier one, far along the keys
        for N in (2048, 2112, 4300, 8192):
            if 32 * low_block >= N:
                continue
            q, k, v, keep = _underflowing(B, H, Hkv, qL, N, D, dtype, cuda, low_block, 0)
            for split in (False, True):
                for shape in range(_lib.SDPA_NUM_SHAPES):
                    if shape == _lib.SDPA_SHARED:
                        continue  # no array mask
                    mode, m, ms, off = _mask_mode(keep, q, k)
                    y = _attention._sdpa_eager(q, k, v, 1.0, mode, m, ms, off, None, shape=shape,
                                               split=split)
                    assert bool((y == 0).all()), (dname, low_block, N, shape, split)
                    zero.setdefault(low_block, set()).update(bits(y).ravel().tolist())
                    assert len(zero[low_block]) == 1, (dname, low_block, N, shape, split)
    # Without a mask: the other keys score far below both (by 400), causal rows
    # of the shared shape among them.
    for N in (2048, 4300):
        q, k, v, _ = _underflowing(B, H, Hkv, 64, N, D, dtype, cuda, 3, -400)
        for spec in (None, "start"):
            for shape in range(_lib.SDPA_NUM_SHAPES):
                mode, m, ms, off = _mask_mode(spec, q, k)
                if spec:
                    off = 2000  # rows 0..63 see keys up to 2000..2063
                y = _attention._sdpa_eager(q, k, v, 1.0, mode, m, ms, off, None, shape=shape)
                assert bool((y == 0).all()), (dname, N, spec, shape)
                zero.setdefault("far", set()).update(bits(y).ravel().tolist())
                assert len(zero["far"]) == 1, (dname, N, spec, shape)


def _ws_bytes(B, H, Hkv, qL, N):
    c = H // Hkv * qL
    return B * Hkv * -(-c // 16) * -(-N // 32) * 128 * min(c, 16)


@pytest.mark.parametrize("D,V", PAIRS)
def test_scores_kernel_gives_the_same_bits(cuda, D, V):
    """The scores route (raw scores by a kernel of their own, the rest reading
    them) gives the one-kernel shapes' bits: key counts below, at and past a
    block, a chain's round and a group of blocks; fewer columns than a tile,
    a last tile cut short, an odd number of tiles; more query rows than keys;
    additive and boolean masks (-inf, the type's lowest value, an infinite
    score), sinks, a negative scale, bases that move in every block, and NaNs
    in the keys and values no row sees."""
    L = _lib.lib()
    cases = [(1, 8, 2, 1, 1), (2, 8, 2, 1, 31), (1, 4, 4, 3, 33), (1, 8, 2, 5, 129),
             (1, 6, 2, 11, 257), (2, 8, 1, 5, 1000), (1, 2, 2, 40, 1100), (1, 8, 2, 9, 4),
             (1, 8, 8, 1, 2100)]
    for dname, dtype in LOW:
        low = torch.finfo(dtype).min
        for n, (B, H, Hkv, qL, N) in enumerate(cases):
            q = rn((B, H, qL, D), dtype, 500 + n, device=cuda)
            cache_k = rn((B, Hkv, N + 40, D), dtype, 520 + n, device=cuda)
            cache_v = rn((B, Hkv, N + 40, V), dtype, 540 + n, device=cuda)
            cache_k[:, :, N:] = float("nan")
            cache_v[:, :, N:] = float("nan")
            k, v = cache_k[:, :, :N], cache_v[:, :, :N]
            sinks = rn((H,), dtype, 560, device=cuda)
            add, keep = _masks(B, qL, N, dtype, cuda, 580 + n)
            add[:, :, :, ::7] = low
            if N > 3:
                add[0, 0, -1, 2] = float("inf")
            rising = k.clone()
            rising[..., 0] = torch.arange(N, device=cuda, dtype=torch.float32).to(dtype) / 2
            hidden_k, hidden_v = cache_k.clone(), cache_v.clone()
            hidden_k[:, :, max(1, N - 20):] = float("nan")
            hidden_v[:, :, max(1, N - 20):] = float("nan")
            seen = torch.zeros(1, 1, 1, N, dtype=torch.bool, device=cuda)
            seen[..., :max(1, N - 20)] = True
            for label, kk, vv, spec, sk, scale in (
                    ("none", k, v, None, None, D ** -0.5), ("end", k, v, "end", sinks, D ** -0.5),
                    ("start", k, v, "start", None, -0.3), ("additive", k, v, add, sinks, D ** -0.5),
                    ("bool", k, v, keep, None, D ** -0.5), ("rising", rising, v, "end", None, 0.2),
                    ("hidden", hidden_k[:, :, :N], hidden_v[:, :, :N], seen, None, D ** -0.5)):
                mode, m, ms, off = _mask_mode(spec, q, kk)
                ref = bits(_attention._sdpa_eager(q, kk, vv, scale, mode, m, ms, off, sk,
                                                  shape=_lib.SDPA_TILE))
                for shape in (_lib.SDPA_TILE, _lib.SDPA_SPLIT2, _lib.SDPA_SPLIT4, _lib.SDPA_SPLIT8):
                    y = _attention._sdpa_eager(q, kk, vv, scale, mode, m, ms, off, sk, shape=shape,
                                               split=True)
                    case = "%s D=%d V=%d %s %s shape %d" % (dname, D, V, cases[n], label, shape)
                    if label in ("none", "hidden"):
                        assert torch.isfinite(y).all(), case
                    d = int((bits(y) != ref).sum())
                    assert d == 0, "%s: %d differ" % (case, d)
    assert L.bi_sdpa_workspace(1, 8, 2, 1, 1, D, V, _lib.BF16, 0) == 0


def _scores_problem(cuda, dtype=torch.bfloat16, B=1, qL=1, N=8192, seed=600):
    q = rn((B, 32, qL, 128), dtype, seed, device=cuda)
    k = rn((B, 8, N, 128), dtype, seed + 1, device=cuda)
    v = rn((B, 8, N, 128), dtype, seed + 2, device=cuda)
    need = _lib.lib().bi_sdpa_workspace(B, 32, 8, qL, N, 128, 128, _lib.DTYPE_CODES[dtype], 0)
    return q, k, v, need


def test_workspace_of_any_size_gives_the_same_bits(cuda):
    """bi_sdpa_ws without a workspace, with one byte too few and with exactly
    bi_sdpa_workspace's gives bi_sdpa's bits; exactly that many bytes are
    written, and a misaligned buffer is refused."""
    L = _lib.lib()
    for dname, dtype in LOW:
        q, k, v, need = _scores_problem(cuda, dtype)
        assert need == _ws_bytes(1, 32, 8, 1, 8192)
        want = run(q, k, v, None, shape=_lib.SDPA_TILE)
        buf = torch.full((need + 4096,), 171, dtype=torch.uint8, device=cuda)
        strides = _lib.i64_array((32 * 128, 128, 128) + 2 * (8 * 8192 * 128, 8192 * 128, 128))

        def call(ptr, size):
            out = torch.full_like(want, float("nan"))
            rc = L.bi_sdpa_ws(q.data_ptr(), k.data_ptr(), v.data_ptr(), None, None, None,
                              out.data_ptr(), 1, 32, 8, 1, 8192, 128, 128, strides,
                              1.0 / math.sqrt(128), _lib.MASK_NONE, 0, _lib.DTYPE_CODES[dtype], ptr, size,
                              torch.cuda.current_stream().cuda_stream)
            return rc, out

        for ptr, size in ((None, 0), (None, need), (buf.data_ptr(), need - 1)):
            rc, out = call(ptr, size)
            assert rc == _lib.OK and ndiff(out, want) == 0, (dname, size)
            assert bool((buf == 171).all())
        rc, out = call(buf.data_ptr(), need)
        assert rc == _lib.OK and ndiff(out, want) == 0, dname
        assert bool((buf[need:] == 171).all()) and not bool((buf[:need] == 171).all())
        assert call(buf.data_ptr() + 8, need)[0] == _lib.EINVAL


def test_workspace_route_in_a_graph_and_on_two_streams(cuda):
    """The route with a workspace, captured and replayed with other attention
    calls and allocations between the replays, and run on two streams at once
    with different inputs: every result has the eager call's bits."""
    q, k, v, need = _scores_problem(cuda)
    assert need > 0
    eager = bi.scaled_dot_product_attention(q, k, v).clone()
    assert ndiff(eager, run(q, k, v, None, shape=_lib.SDPA_TILE)) == 0
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        bi.scaled_dot_product_attention(q, k, v)
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = bi.scaled_dot_product_attention(q, k, v)
    q2, k2, v2, _ = _scores_problem(cuda, seed=620)
    eager2 = bi.scaled_dot_product_attention(q2, k2, v2).clone()
    for rep in range(4):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert ndiff(y, eager) == 0, rep
        junk = torch.full((need,), 255, dtype=torch.uint8, device=cuda)
        assert ndiff(bi.scaled_dot_product_attention(q2, k2, v2), eager2) == 0, rep
        del junk
        torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    for st in streams:
        st.wait_stream(torch.cuda.current_stream())
    outs = [[], []]
    for rep in range(8):
        for i, (st, a) in enumerate(zip(streams, ((q, k, v), (q2, k2, v2)))):
            with torch.cuda.stream(st):
                outs[i].append(bi.scaled_dot_product_attention(*a))
    torch.cuda.synchronize()
    for i, want in enumerate((eager, eager2)):
        for rep, got in enumerate(outs[i]):
            assert ndiff(got, want) == 0, (i, rep)


def test_picked_route_is_invariant_along_the_batch_and_query_rows(cuda):
    """Problems that take the scores route and problems that do not, as
    bi_sdpa_workspace says, give a row the same bits: batch 1 and 16, query
    rows 1 and 64 of a causal chunk, with and without an array mask."""
    L = _lib.lib()
    for dname, dtype in LOW:
        for D, N in ((128, 6000), (64, 9000), (256, 2500)):
            q = rn((16, 16, 64, D), dtype, 700, device=cuda)
            k = rn((16, 4, N, D), dtype, 701, device=cuda)
            v = rn((16, 4, N, D), dtype, 702, device=cuda)
            code = _lib.DTYPE_CODES[dtype]
            assert L.bi_sdpa_workspace(1, 16, 4, 1, N, D, D, code, 0) > 0
            assert L.bi_sdpa_workspace(16, 16, 4, 64, N, D, D, code, 1) == 0
            full = bi.scaled_dot_product_attention(q, k, v, mask="causal")
            one = bi.scaled_dot_product_attention(q[3:4, :, 63:], k[3:4], v[3:4])
            assert ndiff(one[0, :, 0], full[3, :, 63].contiguous()) == 0, (dname, D)
            zeros = torch.zeros(1, 1, 1, N, dtype=dtype, device=cuda)
            one = bi.scaled_dot_product_attention(q[3:4, :, 63:], k[3:4], v[3:4], mask=zeros)
            assert ndiff(one[0, :, 0], full[3, :, 63].contiguous()) == 0, (dname, D)
