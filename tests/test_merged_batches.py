"""Merged batches (js/src/mi355x/codegen.js mergedKernel): independent elementwise or rowwise launches
that read the same operands, computed by one kernel that loads each operand once. On the CPU, the
batch checker compares what the merged text stores for each member, value by value, with what the
member's own kernel stores; on the GPU, the perf lowering that runs them equals the plain one (a
launch per node) bit for bit, at sizes with remainders (the full sizes are test_gpu_c2.py's and
test_gpu_configs.py's)."""
import numpy as np
import pytest

CHAINS = [(0, 8192, 1024), (3, 8192, 1024), (11, 4097, 515), (13, 4097, 515), (0, 4097, 515), (13, 2049, 1024), (3, 64, 1024)]
ROWS = [("softmax", 16384, 4096), ("logSoftmax", 16384, 4096), ("softmax", 8191, 258), ("logSoftmax", 4099, 2049), ("softmax", 8193, 61),
        ("softmax", 64, 258), ("softmax", 300, 3000), ("logSoftmax", 513, 2048)]


def graphs(tool):
    g = tool("config-graphs", {"c2": [{"seed": s, "R": R, "C": C} for s, R, C in CHAINS],
                               "c3": [{"fn": f, "R": R, "C": C} for f, R, C in ROWS]})
    return [dict(name=f"chain-{x['seed']}-{x['R']}x{x['C']}", **x["gradient"]) for x in g["c2"]] + \
        [dict(name=f"{x['fn']}-{x['R']}x{x['C']}", **x["gradient"]) for x in g["c3"]]


def test_merged_kernels_store_each_members_own_values(tool):
    res = {r["name"]: r for r in tool("batch-check", {"graphs": graphs(tool), "models": [{"model": "transformer", "B": 64, "attention": True}],
                                                      "plant": True})}
    assert all(r["check"]["ok"] for r in res.values()), [r for r in res.values() if not r["check"]["ok"]]
    assert res["chain-0-8192x1024"]["merged"][0]["count"] == 4 and res["chain-13-4097x515"]["merged"][0]["count"] == 2
    assert res["logSoftmax-16384x4096"]["merged"][0]["count"] == 2 and res["logSoftmax-4099x2049"]["merged"][0]["count"] == 2
    assert res["softmax-8193x61"]["merged"] and res["transformer-64-attention"]["merged"]
    # A grid that does not fill the chip keeps its members side by side.
    assert not res["chain-3-64x1024"]["merged"] and not res["softmax-64x258"]["merged"]
    # Two members exchanged in the launch list: each output would be the other's value.
    for name in ("chain-0-8192x1024", "chain-3-8192x1024", "chain-0-4097x515", "logSoftmax-16384x4096", "softmax-8193x61"):
        assert not res[name]["body"]["ok"] and "member" in res[name]["body"]["why"], (name, res[name]["body"])


def copies(c, n):
    """n independent copies of a graph, each over inputs of its own."""
    nodes, keep = [], []
    for i in range(n):
        at = len(nodes)
        for x in c["graph"]["nodes"]:
            attrs = dict(x["attrs"], name=f"{x['attrs']['name']}{i}") if x["op"] == "input" else x["attrs"]
            nodes.append(dict(x, inputs=[at + k for k in x["inputs"]], attrs=attrs))
        keep += [at + k for k in c["keep"]]
    return {"graph": {"nodes": nodes}, "keep": keep}


def test_wide_rows_that_do_not_merge_share_dispatches_as_other_launches_do(tool):
    """Rows that a workgroup reduces (2048 elements or more): few rows' launches in a ragged batch, launches of one text side
    by side, a pair that reads one operand merged whatever else is ready beside it."""
    few = [("softmax", 64, 4096), ("logSoftmax", 64, 4096), ("softmax", 256, 4096), ("logSoftmax", 512, 2048), ("softmax", 300, 3000)]
    many = [("softmax", 64, 2048, 6, 1), ("softmax", 256, 2048, 3, 2), ("softmax", 16384, 4096, 6, 2), ("logSoftmax", 512, 2048, 4, 2)]
    g = tool("config-graphs", {"c3": [{"fn": f, "R": R, "C": C} for f, R, C in few] + [{"fn": f, "R": R, "C": C} for f, R, C, _, _ in many]
                               + [{"fn": "softmax", "R": 16384, "C": 4096}]})["c3"]
    req = [dict(x["gradient"], name=f"one {x['fn']} {x['R']}x{x['C']}") for x in g[:len(few)]]
    req += [dict(copies(x["forward"], m[3]), name=f"{m[3]} {x['fn']} {x['R']}x{x['C']}") for x, m in zip(g[len(few):], many)]
    pair = g[-1]["gradient"], copies(g[-1]["forward"], 1)
    n = len(pair[0]["graph"]["nodes"])
    req.append({"name": "pair and another", "keep": pair[0]["keep"] + [n + k for k in pair[1]["keep"]], "graph": {"nodes": pair[0]["graph"]["nodes"]
                + [dict(x, inputs=[n + k for k in x["inputs"]]) for x in pair[1]["graph"]["nodes"]]}})
    res = tool("batch-check", {"graphs": req})
    assert all(r["check"]["ok"] for r in res), [r for r in res if not r["check"]["ok"]]
    dispatches = {r["name"]: r["launches"] - r["check"]["saved"] for r in res}
    assert [dispatches[x["name"]] for x in req] == [1] * len(few) + [m[4] for m in many] + [2], dispatches
    assert [r["merged"] for r in res[:-1]] == [[]] * (len(res) - 1) and res[-1]["merged"][0]["count"] == 2


def test_rowwise_members_merge_where_it_was_measured_faster(tool):
    """Below 128 MiB: members whose wavefronts hold one row each, three or more of them over a multiple of 8 workgroups,
    stay side by side; few wide rows stay a ragged batch; the others merge, as all do from 128 MiB."""
    ln = [(2176, 960, 0), (4096, 768, 0), (8192, 256, 3), (3000, 512, 3), (8192, 960, 3), (512, 2048, 0), (513, 2048, 3)]
    sm = [(6144, 512, 2), (512, 2048, 0), (513, 2048, 2), (1024, 4096, 2)]
    g = tool("config-graphs", {"ln": [{"R": R, "C": C} for R, C, _ in ln], "c3": [{"fn": "softmax", "R": R, "C": C} for R, C, _ in sm]})
    res = tool("batch-check", {"graphs": [dict(x["gradient"], name=f"{x.get('fn', 'layernorm')} {x['R']}x{x['C']}") for x in g["ln"] + g["c3"]]})
    assert all(r["check"]["ok"] for r in res), [r for r in res if not r["check"]["ok"]]
    rows = [[m["count"] for m in r["merged"] if m["kernel"].startswith("tcmi_grow")] for r in res]
    assert rows == [[n] if n else [] for _, _, n in ln + sm], [(r["name"], x) for r, x in zip(res, rows)]


def test_merged_batches_count_an_operand_once(tool):
    """The bytes of a lowering as it runs (the benchmark's step_bytes): config 2's 16 programs, of which merged batches load
    shared operands once, and the logSoftmax gradient, which reads x and dy and writes y and dx."""
    g = tool("config-graphs", {"c2": [{"seed": s, "R": 8192, "C": 1024} for s in range(8)], "c3": [{"fn": "logSoftmax", "R": 16384, "C": 4096}]})
    res = tool("batch-check", {"graphs": [dict(x[k], name=f"chain-{x['seed']}-{k}") for x in g["c2"] for k in ("forward", "gradient")]
                               + [dict(g["c3"][0]["gradient"], name="rows")]})
    assert res[-1]["bytes"] == 4 * 4 * 16384 * 4096
    tensor = 4 * 8192 * 1024
    merged = [r for r in res[:-1] if r["merged"]]
    # What one by one launches of the same lowering read and write, as the records of the launches add up to.
    apart = {r["name"]: r["apart"] for r in res}
    assert merged and all(apart[r["name"]] - r["bytes"] >= tensor for r in merged)
    assert all(apart[r["name"]] == r["bytes"] for r in res[:-1] if not r["merged"])
    assert apart["chain-0-gradient"] - res[1]["bytes"] == 8 * tensor + 4 * 1024    # and the row vector once
    assert sum(r["bytes"] for r in res[:-1]) == 2449633280


def over_zeros():
    """exp(x) / 0 and exp(x) / -0, one operand read by both: inf and -inf."""
    shape = [8192, 1024]
    n = [("input", [], {"name": "x", "shape": shape}, shape), ("exp", [0], {}, shape)]
    for zero in (0.0, -0.0):
        at = len(n)
        n += [("const", [], {"shape": [], "value": zero}, []), ("broadcast", [at], {"shape": shape}, shape), ("div", [1, at + 1], {}, shape)]
    return {"nodes": [{"id": i, "op": op, "inputs": ins, "attrs": attrs, "shape": s} for i, (op, ins, attrs, s) in enumerate(n)]}


def test_constants_that_differ_in_their_sign_of_zero_stay_apart(tool):
    """Two members that differ in a constant, 0 and -0: each output is its own member's."""
    r = tool("batch-check", {"graphs": [{"name": "zeros", "graph": over_zeros(), "keep": [4, 7]}]})[0]
    assert r["merged"] and r["merged"][0]["count"] == 2
    assert r["check"]["ok"], r["check"]


def test_launches_that_differ_in_their_sign_of_zero_run_their_own_kernels(tool):
    """The same two nodes as launches of the plain lowering, which shares a kernel among nodes alike."""
    res = tool("lower", {"graph": over_zeros(), "fuse": {"keep": [4, 7]}, "sources": True})
    a, b = [x["kernels"][0] for x in res["launches"] if "op_div" in x["kernels"][0]["source"]]
    assert "f32_bits(0x00000000u)" in a["source"] and "f32_bits(0x80000000u)" not in a["source"]
    assert "f32_bits(0x80000000u)" in b["source"] and "f32_bits(0x00000000u)" not in b["source"]


@pytest.mark.gpu
def test_merged_chains_equal_the_plain_lowering(tmp_path, tool):
    import tcmi_bridge
    from test_gpu_c2 import check, judge_bundle
    print("gpu step: gpu-chains seeds 0, 3, 11, 13 at [4097,515]", flush=True)
    tool("gpu-chains", {"seeds": [0, 3, 11, 13], "R": 4097, "C": 515, "unfused": True, "perf": True}, out=str(tmp_path), timeout=300)
    b = tcmi_bridge.Bundle(tmp_path)
    check(judge_bundle(b))


@pytest.mark.gpu
def test_merged_rows_equal_the_plain_lowering(tmp_path, tool):
    import tcmi_bridge
    from oracle import bounds
    print("gpu step: gpu-configs softmax/logSoftmax, odd rows and lengths", flush=True)
    tool("gpu-configs", {"c3": [{"fn": f, "R": R, "C": C, "rows": 24} for f, R, C in ROWS if R != 16384], "unfused": False}, out=str(tmp_path), timeout=300)
    b = tcmi_bridge.Bundle(tmp_path)
    for c in b.cases:
        assert c["canaryFused"] and c["perf"]["canary"], c["name"]
        assert c["perf"]["same"] == c["perf"]["total"], (c["name"], c["perf"])
        s = c["sample"]
        ids = [x["id"] for x in s["compare"]]
        ref = bounds.streaming_reference(s["graph"], {k: b.arr(v) for k, v in s["inputs"].items()}, ids)
        j = bounds.judge_outputs([ref[i][0] for i in ids], [ref[i][1] for i in ids], [b.arr(x["fused"]) for x in s["compare"]])
        assert j["pass"], (c["name"], j["first"])
        assert all(p["nonfiniteFused"] == 0 for p in c["props"]), c["name"]
    assert np.array_equal(sorted({c["kind"] for c in b.cases}), ["forward", "gradient"])
