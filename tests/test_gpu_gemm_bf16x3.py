"""The matmul on the bf16 matrix cores (csrc/kernels/tcmi_gemm_bf16x3.h) where it can go
wrong: tiles, slices and loads that end inside a product, both transposed forms, batches, the K
split, operands the split into bf16 parts does not cover (infinities, NaN, values near the
largest and the smallest float32), and its error beside the fp32 kernel's."""
import ctypes
import pathlib

import numpy as np
import pytest

from oracle import bounds
from test_zz_no_alloc import ARG_BYTES, pack

pytestmark = pytest.mark.gpu

PKG = pathlib.Path(__file__).resolve().parent.parent / "tensor-compiler-webgpu_amd"

# (M, K, N): one past and one short of the 128 x 256, 64 x 128 and 64 x 64 tiles, K ending 1, 3
# and 31 short of a slice of 32 and a group of 4, rows of odd length (unaligned 128-bit loads).
RAGGED = [(2049, 1027, 1025), (1087, 1025, 2047), (1023, 1058, 2050), (1000, 515, 1777), (4095, 97, 1021)]


def test_forward_and_both_transposed_products_within_budget(tmp_path, tool):
    import tcmi_bridge
    print("gpu step: gpu-configs, ragged products forward and gradient", flush=True)
    tool("gpu-configs", {"c4": [{"act": "tanh", "M": M, "K": K, "N": N, "rows": 24, "cols": 24} for M, K, N in RAGGED],
                         "unfused": True}, out=str(tmp_path), timeout=600)
    b = tcmi_bridge.Bundle(tmp_path)
    assert len(b.cases) == 2 * len(RAGGED)
    for c in b.cases:
        assert c["canaryFused"] and c["canaryUnfused"] and c["perf"]["canary"], c["name"]
        assert c["perf"]["same"] == c["perf"]["total"], (c["name"], c["perf"])
        for s in c["samples"]:
            ins = {k: b.arr(v) for k, v in s["inputs"].items()}
            ids = [x["id"] for x in s["compare"]]
            ref = bounds.streaming_reference(s["graph"], ins, ids)
            j = bounds.judge_outputs([ref[i][0] for i in ids], [ref[i][1] for i in ids], [b.arr(x["fused"]) for x in s["compare"]])
            assert j["pass"], (c["name"], s["slice"], j["first"], j["unjudged"])


def operand(nodes, name, x, view):
    """Appends the operand's nodes, reading `x` in place through `view`: 't' its last two axes exchanged,
    'h' its axes [B, H, rows, cols] from [B, rows, H, cols], ('m', B, H) its [B·T, H·d] from [B, H, T, d].
    Returns its node and the array the input holds."""
    def add(op, ins, attrs, shape):
        nodes.append({"op": op, "inputs": ins, "attrs": attrs, "shape": list(shape)})
        return len(nodes) - 1

    if view is None:
        return add("input", [], {"name": name, "shape": list(x.shape)}, x.shape), x
    perm = list(range(x.ndim - 2)) + [x.ndim - 1, x.ndim - 2] if view == "t" else [0, 2, 1, 3]
    if view in ("t", "h"):
        source, shape = x.transpose(perm), x.shape
    else:
        _, B, H = view
        T, d = x.shape[0] // B, x.shape[1] // H
        source, shape = x.reshape(B, T, H, d).transpose(perm), (B, T, H, d)
    at = add("transpose", [add("input", [], {"name": name, "shape": list(source.shape)}, source.shape)], {"perm": perm}, shape)
    return at if shape == x.shape else add("reshape", [at], {"shape": list(x.shape)}, x.shape), np.ascontiguousarray(source)


def product(tool, x, w, views=(None, None)):
    """x [.., M, K] times w [.., K, N], the operands behind `views`, by the lowering's kernels, in this process; and their text."""
    import tcmi_ctypes
    u32, u64 = tcmi_ctypes.u32, tcmi_ctypes.u64
    shape = list(x.shape[:-1]) + [w.shape[-1]]
    nodes = []
    (a, x), (b, w) = operand(nodes, "x", x, views[0]), operand(nodes, "w", w, views[1])
    nodes.append({"op": "matmul", "inputs": [a, b], "attrs": {}, "shape": shape})
    res = tool("lower", {"graph": {"nodes": nodes}, "sources": True, "perf": True, "keep": [len(nodes) - 1]})["launches"]
    assert len(res) == 1, "an operand is not read in place"
    launch = res[0]
    read = {i: v for i, v in zip([i for i, n in enumerate(nodes) if n["op"] == "input"], (x, w))}
    x, w = (read[i] for i in launch["inputs"])
    t = tcmi_ctypes.load()
    t.init()
    t.set_include_dir(str(PKG / "csrc" / "kernels").encode())
    t.set_cache_dir(str(PKG / "_build" / "kcache").encode())
    mod = u64()
    text = '#include "tcmi_device.h"\n' + "\n".join(k["source"] for k in launch["kernels"])
    t.module_compile(text.encode(), None, ctypes.byref(mod))
    owned = []

    def alloc(nbytes):
        h = u64()
        t.malloc((nbytes + 15) // 16 * 16, ctypes.byref(h))
        owned.append(h.value)
        return h.value

    try:
        y = np.empty(shape, dtype=np.float32)
        hx, hw, hy, ws = alloc(x.nbytes), alloc(w.nbytes), alloc(y.nbytes), alloc(max(16, launch["workspace"]))
        for h, v in ((hx, x), (hw, w)):
            t.h2d(h, 0, v.ctypes.data, v.nbytes)
        a = pack([hx, hw], hy, ws, launch["params"])
        for k in launch["kernels"]:
            f = u64()
            t.module_function(mod.value, k["name"].encode(), ctypes.byref(f))
            t.launch(f.value, (u32 * 3)(*k["grid"]), (u32 * 3)(*k["block"]), k["lds"], a.ctypes.data, ARG_BYTES)
        t.sync()
        t.d2h(y.ctypes.data, hy, 0, y.nbytes)
        return y, text
    finally:
        for h in owned:
            t.free(h)
        t.module_unload(mod)


@pytest.mark.parametrize("batch,M,K,N", [(1, 1024, 512, 832), (1, 4097, 96, 1024), (1, 256, 8192, 512), (3, 520, 530, 900), (1, 1024, 4096, 2048)])
def test_sums_are_no_less_exact_than_fp32_ones(tool, batch, M, K, N):
    """Every element within gamma(K) of float64's, and their 2-norm error within what an fp32 sum of K terms makes: K
    roundings of 2^-24 / sqrt(3) of the partial sum, whose square grows as k / K (K / 2 in all), and the result's own."""
    print(f"gpu step: product {batch}x{M}x{K}x{N}", flush=True)
    rng = np.random.default_rng(M + K + N)
    lead = (batch,) if batch > 1 else ()
    x = rng.standard_normal(lead + (M, K)).astype(np.float32)
    w = rng.standard_normal(lead + (K, N)).astype(np.float32)
    y, text = product(tool, x, w)
    assert "gemm_bf16x3" in text
    exact = x.astype(np.float64) @ w.astype(np.float64)
    u = 2.0 ** -24
    assert np.all(np.abs(y - exact) <= K * u / (1 - K * u) * (np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64)))
    rel = np.linalg.norm(y - exact) / np.linalg.norm(exact)
    assert rel <= u * np.sqrt(K / 2 / 3 + 1), rel


def test_selection_returns_the_values_bit_for_bit(tool):
    """A product with the identity's first columns: the three parts sum back to the value. Values over
    60 binades, zeros of both signs."""
    print("gpu step: selection 1024x544x832", flush=True)
    rng = np.random.default_rng(5)
    x = (rng.standard_normal((1024, 544)) * 2.0 ** rng.integers(-30, 30, (1024, 544))).astype(np.float32)
    x[::7, ::5] = 0.0
    y, text = product(tool, x, np.eye(544, 832, dtype=np.float32))
    assert "gemm_bf16x3" in text
    want = np.zeros((1024, 832), dtype=np.float32)
    want[:, :544] = x
    assert np.array_equal(y, want)


@pytest.mark.parametrize("what", ["infinite", "nan", "near the largest", "overflowing", "tiny", "subnormal results", "wide"])
def test_values_the_parts_do_not_cover_take_the_fp32_sums(tool, what):
    """One such row (and one column) among ordinary ones: IEEE results where they are not finite, fp32's accuracy
    where they are."""
    print(f"gpu step: 1024x512x832, {what}", flush=True)
    rng = np.random.default_rng(9)
    x = rng.standard_normal((1024, 512)).astype(np.float32)
    w = rng.standard_normal((512, 832)).astype(np.float32)
    if what == "infinite":
        x[130, 7], w[9, 300] = np.inf, -np.inf
    elif what == "nan":
        x[130, 7] = np.nan
    elif what == "near the largest":
        x[130, :] = 0.0
        x[130, 7] = np.float32(3.4028235e38)      # rounds to infinity in bf16
        w[7, :] = np.where(np.abs(w[7, :]) < 0.9, w[7, :], 0.5)
    elif what == "overflowing":
        x[130, 7], w[7, :] = 1e30, 1e30
    elif what == "tiny":
        x[130, :] = (rng.standard_normal(512) * 1e-35).astype(np.float32)
        x[500, :] = (rng.standard_normal(512) * 1e-32).astype(np.float32)
    elif what == "subnormal results":
        x[130, :] = (rng.standard_normal(512) * 1e-38).astype(np.float32)
    elif what == "wide":
        x[130, :] = (rng.standard_normal(512) * 1e-34).astype(np.float32)
        w[:, 300] = (rng.standard_normal(512) * 1e34).astype(np.float32)
    y, text = product(tool, x, w)
    assert "gemm_bf16x3" in text
    with np.errstate(invalid="ignore", over="ignore"):
        exact = x.astype(np.float64) @ w.astype(np.float64)
        want = exact.astype(np.float32)
    finite = np.isfinite(want)
    assert np.array_equal(np.isnan(y), np.isnan(want))
    assert np.array_equal(y[~finite & ~np.isnan(want)], want[~finite & ~np.isnan(want)])
    # Finite sums: 512 fp32 roundings of each product and partial sum; a subnormal may be flushed to 0.
    budget = 512 * 2.0 ** -24 * (np.abs(np.nan_to_num(x, posinf=0, neginf=0)).astype(np.float64)
                                 @ np.abs(np.nan_to_num(w, posinf=0, neginf=0)).astype(np.float64)) + 2.0 ** -126
    assert np.all(np.abs(y[finite] - exact[finite]) <= budget[finite])
    if what in ("tiny", "wide"):   # 1e-35 by itself has no third part in bf16: 2-norm errors as an ordinary row's
        for r in (130, 500) if what == "tiny" else (130,):
            assert np.linalg.norm(y[r] - exact[r]) <= 1e-6 * np.linalg.norm(exact[r]), r


@pytest.mark.parametrize("what,value,scale", [
    ("no part in bf16", 2.0 ** -135, 2.0 ** 40), ("the least subnormal", 2.0 ** -149, 2.0 ** 90),
    ("leading parts that cancel", 0.0, 2.0 ** 30)])
def test_operands_below_the_range_of_bf16_keep_their_bits(tool, what, value, scale):
    """An operand below 2^-134 is 0 in bf16, and a sum whose leading parts cancel is left with bits below bf16's range: a
    sum of 0 if they are lost, an ordinary value in fp32, exact here (few bits)."""
    print(f"gpu step: 1024x512x832, {what}", flush=True)
    rng = np.random.default_rng(3)
    x = rng.standard_normal((1024, 512)).astype(np.float32)
    w = rng.standard_normal((512, 832)).astype(np.float32)
    w[:, 300] = scale
    if value:
        x[130, :] = value
    else:
        x[130, :] = 0.0
        x[130, 7], x[130, 300] = 2.0 ** -118 * (1 + 2.0 ** -20), -2.0 ** -118
    y, text = product(tool, x, w)
    assert "gemm_bf16x3" in text
    assert y[130, 300] == (512 * value * scale if value else 2.0 ** -138 * scale)


def test_subnormal_parts_keep_their_bits(tool):
    """Operands whose third (below: second) part is subnormal as a bf16 by itself: exact, as every partial sum is a float32."""
    print("gpu step: 1024x512x832, subnormal third parts", flush=True)
    x = np.full((1024, 512), 2.0 ** -110 * (1 + 2.0 ** -9 + 2.0 ** -18), dtype=np.float32)
    y, text = product(tool, x, np.ones((512, 832), dtype=np.float32))
    assert "gemm_bf16x3" in text
    assert np.all(y == np.float32(512 * 2.0 ** -110 * (1 + 2.0 ** -9 + 2.0 ** -18)))
    # The second part, beside larger operands.
    x[:, :256], x[:, 256:] = 2.0 ** -118 * (1 + 2.0 ** -9), 2.0 ** -108
    y, _ = product(tool, x, np.ones((512, 832), dtype=np.float32))
    assert np.all(y == np.float32(256 * (2.0 ** -118 + 2.0 ** -127 + 2.0 ** -108)))


def test_products_left_out_add_to_no_more_than_a_rounding(tool):
    """Operands of one value whose left-out products are the largest there are, all of one sign: 2^-24 of the sum. The
    accumulator's roundings, 6 in 32 k, add at most 6 · (1 + .. + 16) / 16 = 51 of the result's."""
    print("gpu step: 1024x512x832, the largest left-out products", flush=True)
    c = np.float32(1 + 2.0 ** -8 - 2.0 ** -17)
    y, text = product(tool, np.full((1024, 512), c), np.full((512, 832), c))
    assert "gemm_bf16x3" in text
    exact = 512 * float(c) ** 2
    assert np.all(np.abs(y.astype(np.float64) - exact) <= (1 + 51) * 2.0 ** -24 * 1.001 * exact)


# Tiles (wavefronts along n, 16-wide tiles of one along m and n), views and what else sets an instantiation apart.
FALLBACKS = [
    ("128 x 256, transposed x", "<2, 4, 4, 4, false, false, false, 1, 0, false", (), 4096, 512, 4096, ("t", None)),
    ("128 x 256, transposed w", "<2, 4, 4, 4, true, true, false, 0, 1, false", (), 1024, 256, 8192, (None, "t")),
    ("64 x 128, both transposed", "<2, 4, 2, 2, false, true, false, 1, 1, false", (), 8192, 512, 256, ("t", "t")),
    ("64 x 128, K split", "<2, 4, 2, 2, false, false, false, 1, 0, true", (), 256, 8192, 512, ("t", None)),
    ("64 x 64, odd rows", "<2, 2, 2, 2, true, false, true, 2, 2, false", (), 1023, 513, 2049, (None, None)),
    ("64 x 64, odd rows transposed", "<2, 2, 2, 2, false, true, true, 2, 2, false", (), 1023, 513, 2049, ("t", "t")),
    ("64 x 64, batches", "<2, 2, 2, 2, true, false, true, 2, 0, false", (3,), 520, 530, 900, (None, None)),
    ("64 x 128, heads", "<2, 4, 2, 2, true, false, false, 0, 0, false", (4, 2), 512, 128, 512, ("h", "h")),
    ("64 x 128, mapped rows", "<2, 4, 2, 2, true, false, false, 0, 0, false", (), 2048, 512, 1024, (("m", 16, 4), None)),
]


@pytest.mark.parametrize("name,tile,lead,M,K,N,views", FALLBACKS, ids=[f[0] for f in FALLBACKS])
def test_every_instantiation_falls_back(tool, name, tile, lead, M, K, N, views):
    """One infinity in each operand, a NaN, a value that bf16 rounds to infinity, and a subnormal row in the last tile
    against a large column there: IEEE results where they are not finite, fp32's accuracy where they are."""
    print(f"gpu step: fallback, {name}", flush=True)
    rng = np.random.default_rng(M + N)
    x = rng.standard_normal(lead + (M, K)).astype(np.float32)
    w = rng.standard_normal(lead + (K, N)).astype(np.float32)
    w[..., K - 2, :] = np.where(np.abs(w[..., K - 2, :]) < 0.9, w[..., K - 2, :], 0.5)
    x[..., M // 2, :], x[..., M // 2, K - 2] = 0.0, 3.4028235e38
    x[..., 1, 7], w[..., 9, 3], x[..., M // 4, K - 1] = np.inf, -np.inf, np.nan
    x[..., M - 1, :] = (rng.integers(1, 1 << 10, lead + (K,)) * 2.0 ** -149).astype(np.float32)
    w[..., :, N - 1] *= np.float32(1e27)
    y, text = product(tool, x, w, views)
    assert "gemm_bf16x3" + tile in text
    with np.errstate(invalid="ignore", over="ignore"):
        exact = x.astype(np.float64) @ w.astype(np.float64)
        want = exact.astype(np.float32)
    finite = np.isfinite(want)
    assert np.array_equal(np.isnan(y), np.isnan(want))
    assert np.array_equal(y[~finite & ~np.isnan(want)], want[~finite & ~np.isnan(want)])
    xs, ws = (np.abs(np.nan_to_num(v, nan=0.0, posinf=0.0, neginf=0.0)).astype(np.float64) for v in (x, w))
    budget = K * 2.0 ** -24 * (xs @ ws) + 2.0 ** -126     # K roundings of products and partial sums; a subnormal may be flushed
    assert np.all(np.abs(y[finite] - exact[finite]) <= budget[finite])
