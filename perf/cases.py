"""Workloads a program gives this backend, each as one timed pass through its public entry points.

A graph is built by the package's builders, fused and lowered in a node child (the host
modules INTEGRATION.md describes); its launches are issued in this process through the C ABI
(tcmi_ctypes): node buffers from tcmi_malloc, modules from tcmi_module_compile, a program's
launches in one tcmi_launch_dag call, a training step in one tcmi_graph_step call, as the
Node host's Program and HipTrainer do it. Sizes are the benchmark's five configurations, the
tests' smaller ones, and ragged sizes between them:

  mlp        a training step of 64 -> 128 tanh -> 10 class probabilities, SGD (configuration 1)
  chain      8-16 elementwise ops over [R, C] with a row vector, forward or gradient (2)
  softmax    softmax or logSoftmax over rows, forward or gradient (3)
  layernorm  the transformer's LayerNorm by itself, forward or gradient
  dense      act(X.W + b), forward or all its gradients (4)
  attention  softmax(q.k^T / sqrt(dh) + causal mask).v
  forward    the transformer's logits and loss
  step       the transformer's training step, SGD (5)

Everything is fp32, the only type the backend has.
"""
import ctypes
import json
import math
import os
import pathlib
import subprocess
import sys

import numpy as np
import torch

ROOT = pathlib.Path(__file__).resolve().parent.parent
PKG = ROOT / "tensor-compiler-webgpu_amd"
if str(PKG) not in sys.path:
    sys.path.insert(0, str(PKG))
import tcmi_ctypes  # noqa: E402

MASK = -1e4          # the transformer's causal mask
EPS = 1e-5           # LayerNorm's
# Chain programs in which no rounded value decides a step (an element within its error of the
# step's edge may land on either side, whatever computes it): their outputs can be compared.
PROGRAMS = (0, 13, 21)
MAX_IN, MAX_P = 8, 48          # TcmiArgs: operand pointers and parameter words

# Builds, fuses and lowers a case's graph; prints what a caller needs to run it: one buffer
# per owner node, the dispatches in order with their operands' nodes, and the kernels' text.
LOWER_JS = r"""
const fs = require('fs'), path = require('path');
const src = (p) => require(path.join(process.argv[1], 'js', 'src', p));
const c = JSON.parse(fs.readFileSync(0, 'utf8'));
const be = src('mi355x/index.js');
const { Graph } = src('ir/graph.js');
const { fuse } = src('fusion/fuse.js');
const { grad } = src('autodiff.js');
const tf = src('builders/transformer.js');
const size = (s) => s.reduce((a, b) => a * b, 1);
let graph, lowered, keep, inputs = {}, program = null;
const plain = (v, names, options) => {
  const f = fuse(v.graph, Object.assign({ keep: v.keep }, options || {}));
  const at = v.keep.map((id) => f.index.get(id));
  graph = f.graph;
  lowered = be.lowerMI355X(graph, { perf: true, keep: at });
  keep = {};
  names.forEach((n, k) => { keep[n] = at[k]; });
  for (const n of graph.nodes) if (n.op === 'input') inputs[n.attrs.name] = n.id;
};
const step = (s, options) => {
  const fs_ = be.fusedStep(s, options);
  graph = fs_.graph;
  lowered = fs_.lowered;
  keep = Object.assign({ loss: fs_.loss, logits: fs_.logits }, fs_.outputs);
  inputs = Object.assign({ cotangent: graph.inputId(fs_.cotangent) }, fs_.inputs);
};
const model = () => Object.assign({}, tf.C5_CONFIG, { T: c.T, d: c.H * c.dh, H: c.H, dh: c.dh, L: c.L, ff: c.ff });
if (c.family === 'chain') {
  const w = src('builders/chains.js').chainWorkload(c.program, c.R, c.C);
  program = { nodes: w.forward.graph.toJSON().nodes, output: w.forward.keep[0] };
  plain(w[c.gradient ? 'gradient' : 'forward'], c.gradient ? ['y', 'dx0', 'dx1', 'dr'] : ['y']);
} else if (c.family === 'softmax') {
  const g = src('builders/configs.js').c3Graphs(c.fn, c.R, c.C);
  plain(g[c.gradient ? 'gradient' : 'forward'], c.gradient ? ['y', 'dx'] : ['y']);
} else if (c.family === 'layernorm') {
  const g = new Graph();
  const x = g.input('x', [c.R, c.C]), gain = g.input('gain', [c.C]), bias = g.input('bias', [c.C]);
  const y = src('builders/direct_cases.js').layerNormGraph(g, x, gain, bias);
  const G = grad(g, [y], [x, gain, bias]);
  if (c.gradient) plain({ graph: G.graph, keep: [y].concat(G.grads) }, ['y', 'dx', 'dgain', 'dbias']);
  else plain({ graph: g, keep: [y] }, ['y']);
} else if (c.family === 'dense') {
  const g = src('builders/configs.js').c4Graphs(c.act, c.M, c.K, c.N);
  plain(g[c.gradient ? 'gradient' : 'forward'], c.gradient ? ['y', 'dX', 'dW', 'dbias'] : ['y']);
} else if (c.family === 'attention') {
  const g = new Graph();
  const s4 = [c.B, c.H, c.T, c.dh];
  const q = g.input('q', s4), k = g.input('k', s4), v = g.input('v', s4);
  let s = g.mul(g.matmul(q, g.transpose(k, [0, 1, 3, 2])), g.const(1 / Math.sqrt(c.dh)));
  s = g.add(s, g.const(tf.causalMask(c.T, tf.C5_CONFIG.mask), [c.T, c.T]));
  plain({ graph: g, keep: [g.matmul(g.softmax(s, 3), v)] }, ['y'], { attention: true });
} else if (c.family === 'forward') {
  const f = be.fusedForward(tf.buildForward(c.V, c.B, model()));
  graph = f.graph;
  lowered = f.lowered;
  keep = { logits: f.logits, loss: f.loss };
  for (const n of graph.nodes) if (n.op === 'input') inputs[n.attrs.name] = n.id;
} else if (c.family === 'mlp') {
  const m = src('builders/mlp.js');
  step(m.buildMlpStep({ batch: c.batch, inputs: c.inputs, hidden: c.hidden, classes: c.classes, lr: c.lr, seed: 0 }));
} else if (c.family === 'step') {
  step(tf.buildStep(c.V, c.B, model(), { kind: 'sgd', lr: c.lr }), { attention: true });
} else throw new Error(`no family '${c.family}'`);
const alias = new Map(lowered.aliases || []);
const none = new Set((lowered.folded || []).concat(lowered.dead || []));
const buffers = {}, consts = {};
for (const n of graph.nodes) {
  if (alias.has(n.id) || none.has(n.id)) continue;
  buffers[n.id] = size(n.shape);
  if (n.op === 'const') consts[n.id] = n.attrs.value;
}
const batchAt = new Map((lowered.batches || []).map((b) => [b.start, b]));
const kernel = (k) => ({ name: k.name, grid: k.grid, block: k.block, lds: k.lds });
const dispatches = [], L = lowered.launches;
for (let i = 0; i < L.length;) {
  const b = batchAt.get(i), members = L.slice(i, i + (b ? b.count : 1));
  for (const k of b ? b.kernels : members[0].kernels) {
    dispatches.push(Object.assign(kernel(k), { stride: b ? b.wsStride : 0, params: b ? null : Array.from(members[0].params),
      members: members.map((l) => ({ inputs: l.inputs, node: l.node })) }));
  }
  i += members.length;
}
const shapes = {};
for (const k of Object.keys(keep)) shapes[k] = graph.nodes[keep[k]].shape;
fs.writeSync(1, JSON.stringify({ keep, shapes, inputs, buffers, consts, dispatches, program, workspace: lowered.workspace,
  alias: Array.from(alias), sources: Array.from(be.kernelSources(lowered)) }));
"""


# ---- the caller's side of the C ABI --------------------------------------------------------

class Device:
    """The library, and the functions of every kernel loaded so far (a kernel's name is a hash of its text)."""

    def __init__(self):
        self.t = tcmi_ctypes.load()
        self.t.set_include_dir(str(PKG / "csrc" / "kernels").encode())
        self.t.set_cache_dir(os.environ.get("TCMI_KCACHE", str(PKG / "_build" / "kcache")).encode())
        self.t.init()
        self.loaded = {}

    def functions(self, sources):
        missing = sorted((name, text) for name, text in sources if name not in self.loaded)
        if missing:
            module = tcmi_ctypes.u64()
            text = '#include "tcmi_device.h"\n' + "\n".join(x for _, x in missing)
            self.t.module_compile(text.encode(), b"", ctypes.byref(module))
            for name, _ in missing:
                f = tcmi_ctypes.u64()
                self.t.module_function(module, name.encode(), ctypes.byref(f))
                self.loaded[name] = f.value
        return self.loaded


_device = None


def device():
    global _device
    if _device is None:
        torch.cuda.init()
        _device = Device()
    return _device


class Buffer:
    """`n` floats from tcmi_malloc, freed with the last tensor that shows them."""

    def __init__(self, n):
        self.t = device().t
        h = tcmi_ctypes.u64()
        self.t.malloc(max(16, -(-n * 4 // 16) * 16), ctypes.byref(h))
        self.at, self.n = h.value, n

    def tensor(self, shape=None):
        self.__cuda_array_interface__ = {"shape": (self.n,), "typestr": "<f4", "data": (self.at, False), "version": 2}
        x = torch.as_tensor(self, device="cuda")
        return x if shape is None else x.reshape(shape)

    def __del__(self):
        self.t.free(self.at)


class Program:
    """A lowered graph's launches over one buffer per node, their argument blocks packed once."""

    def __init__(self, plan, buffers=None):
        d = device()
        self.t, self.plan = d.t, plan
        fns = d.functions(plan["sources"])
        if buffers is None:
            buffers = {int(k): Buffer(n) for k, n in plan["buffers"].items()}
            for k, v in plan["consts"].items():
                b = buffers[int(k)]
                b.tensor().copy_(torch.tensor(v, dtype=torch.float32).reshape(-1).expand(b.n))
        self.buffers = dict(buffers)
        for node, source in plan["alias"]:
            if source in self.buffers:          # a reshape of a value formed inside its readers has no buffer either
                self.buffers[node] = self.buffers[source]
        self.ws = Buffer(max(4, -(-plan["workspace"] // 4)))
        blocks, dims = [], []
        for k in plan["dispatches"]:
            block = b"".join(self.pointers(m, self.ws.at + i * k["stride"]) for i, m in enumerate(k["members"]))
            if k["params"] is not None:
                block += np.array((k["params"] + [0] * MAX_P)[:MAX_P], dtype=np.uint32).tobytes()
            blocks.append(block)
            dims += list(k["grid"]) + list(k["block"]) + [k["lds"]]
        n = len(blocks)
        data = b"".join(blocks)
        offsets = np.cumsum([0] + [len(b) for b in blocks]).tolist()
        self.call = (n, (tcmi_ctypes.u64 * n)(*(fns[k["name"]] for k in plan["dispatches"])), (tcmi_ctypes.u32 * (7 * n))(*dims),
                     (ctypes.c_uint8 * len(data)).from_buffer_copy(data), (tcmi_ctypes.u32 * (n + 1))(*offsets), 1,
                     (ctypes.c_uint8 * n)(), (tcmi_ctypes.i32 * n)(*([-1] * n)), (tcmi_ctypes.u32 * (n + 1))(), None)

    def pointers(self, member, ws):
        ins = [self.buffers[i].at for i in member["inputs"]]
        return np.array(ins + [0] * (MAX_IN - len(ins)) + [self.buffers[member["node"]].at, ws], dtype=np.uint64).tobytes()

    def write(self, name, x):
        node = self.plan["inputs"].get(name)
        if node is not None and node in self.buffers:
            self.buffers[node].tensor().copy_(x.reshape(-1))

    def outputs(self):
        return {k: self.buffers[i].tensor(self.plan["shapes"][k]) for k, i in self.plan["keep"].items()}

    def run(self):
        self.t.launch_dag(*self.call)

    def capture(self):
        g = tcmi_ctypes.u64()
        self.t.capture_begin()
        self.run()
        self.t.capture_end(ctypes.byref(g))
        return g.value


class Forward:
    """A program whose inputs are on the GPU: a pass is one native call."""

    def __init__(self, plan, values):
        self.program = Program(plan)
        for name, x in values.items():
            self.program.write(name, x)
        self.results = self.program.outputs()
        torch.cuda.synchronize()

    def step(self):
        self.program.run()
        return self.results


class Trainer:
    """A training step: the batch from host memory, the captured launches, the loss back, in one native call.
    Two programs over the same buffers, each parameter's input and output exchanged, take turns."""

    def __init__(self, plan, params, x, y):
        first = Program(plan)
        first.write("cotangent", torch.ones(1))
        buffers = dict(first.buffers)
        for name, p in params.items():
            first.write(name, p)
            a, b = plan["inputs"][name], plan["keep"][name]
            buffers[a], buffers[b] = first.buffers[b], first.buffers[a]
        torch.cuda.synchronize()
        second = Program(plan, {k: v for k, v in buffers.items() if k not in dict(plan["alias"])})
        self.x, self.y = np.ascontiguousarray(x, dtype=np.float32), np.ascontiguousarray(y, dtype=np.float32)
        self.loss = np.zeros(1, dtype=np.float32)
        self.turns = []
        for p in (first, second):
            dst = (tcmi_ctypes.u64 * 2)(*(p.buffers[plan["inputs"][k]].at for k in ("x", "y")))
            src = (ctypes.c_void_p * 2)(self.x.ctypes.data, self.y.ctypes.data)
            sizes = (tcmi_ctypes.u64 * 2)(self.x.nbytes, self.y.nbytes)
            results = p.outputs()
            loss = results.pop("loss")
            call = (2, dst, src, sizes, p.capture(), loss.data_ptr(), self.loss.ctypes.data, 4)
            self.turns.append((p, call, results))
        self.turn = 0
        self.t = first.t

    def step(self):
        _, call, results = self.turns[self.turn]
        self.turn ^= 1
        self.t.graph_step(*call)
        return {"loss": float(self.loss[0]), **results}

    def __del__(self):
        for _, call, _ in getattr(self, "turns", []):
            self.t.graph_destroy(call[4])


def lower(case):
    p = subprocess.run([os.environ.get("TCMI_NODE", "node"), "-e", LOWER_JS, str(PKG)], input=json.dumps(case).encode(),
                       stdout=subprocess.PIPE, check=True)
    return json.loads(p.stdout)


# ---- the cases -----------------------------------------------------------------------------

def listed():
    return [
        # A small model's training step, bound by latency: what a user's first program runs.
        {"name": "mlp-step", "family": "mlp", "batch": 128, "inputs": 64, "hidden": 128, "classes": 10, "lr": 0.1},
        # The smallest elementwise call, the size the tests run.
        {"name": "chain-small", "family": "chain", "program": 13, "R": 64, "C": 1024, "gradient": False},
        # An elementwise program and its gradients over large tensors.
        {"name": "chain-gradient", "family": "chain", "program": 0, "R": 8192, "C": 1024, "gradient": True},
        # Class probabilities over an ordinary batch, rows of a length no power of two.
        {"name": "softmax-1000", "family": "softmax", "fn": "softmax", "R": 8192, "C": 1000, "gradient": False},
        # A large vocabulary's log-probabilities and their gradient.
        {"name": "logsoftmax-gradient", "family": "softmax", "fn": "logSoftmax", "R": 16384, "C": 4096, "gradient": True},
        # A transformer layer's normalisation, both directions.
        {"name": "layernorm-gradient", "family": "layernorm", "R": 8192, "C": 256, "gradient": True},
        # A small dense layer, a middling batch.
        {"name": "dense-512", "family": "dense", "act": "relu", "M": 512, "K": 512, "N": 512, "gradient": False},
        # The largest single product.
        {"name": "dense-4096", "family": "dense", "act": "relu", "M": 4096, "K": 4096, "N": 4096, "gradient": False},
        # A wide layer's forward and backward products (both transposed forms) and its bias gradient.
        {"name": "dense-gradient", "family": "dense", "act": "tanh", "M": 8192, "K": 1024, "N": 4096, "gradient": True},
        # Sizes that divide nothing: every load per element, every tile ragged.
        {"name": "dense-ragged-gradient", "family": "dense", "act": "tanh", "M": 1000, "K": 777, "N": 515, "gradient": True},
        # One attention layer of the transformer below.
        {"name": "attention", "family": "attention", "B": 64, "H": 4, "T": 128, "dh": 64},
        # The character transformer's whole training step.
        {"name": "transformer-step", "family": "step", "V": 96, "B": 64, "T": 128, "H": 4, "dh": 64, "L": 4, "ff": 1024, "lr": 0.05},
    ]


def draw(rng):
    def spread(lo, hi):
        """A size between lo and hi, even over its logarithm; half of them whole multiples of 32."""
        n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        return max(32, n // 32 * 32) if n >= 32 and rng.random() < 0.5 else n

    family = rng.choice(["mlp", "chain", "chain", "softmax", "softmax", "layernorm", "dense", "dense", "dense", "dense",
                         "attention", "attention", "forward", "step"])
    if family == "mlp":
        return {"family": family, "batch": spread(16, 1024), "inputs": spread(16, 256), "hidden": spread(32, 512),
                "classes": spread(2, 100), "lr": 0.1}
    if family == "chain":
        return {"family": family, "program": rng.choice(PROGRAMS), "R": spread(64, 8192), "C": spread(64, 1024),
                "gradient": rng.random() < 0.5}
    if family == "softmax":
        return {"family": family, "fn": rng.choice(["softmax", "logSoftmax"]), "R": spread(64, 16384), "C": spread(32, 4096),
                "gradient": rng.random() < 0.5}
    if family == "layernorm":
        return {"family": family, "R": spread(64, 8192), "C": spread(64, 1024), "gradient": rng.random() < 0.5}
    if family == "dense":
        gradient = rng.random() < 0.5
        return {"family": family, "act": "tanh" if gradient else rng.choice(["relu", "tanh"]), "M": spread(64, 8192),
                "K": spread(64, 2048), "N": spread(64, 2048), "gradient": gradient}
    if family == "attention":
        return {"family": family, "B": rng.randint(1, 32), "H": rng.randint(1, 8), "T": spread(16, 256),
                "dh": rng.choice([16, 20, 32, 48, 64])}
    c = {"family": family, "V": spread(16, 128), "B": spread(1, 32), "T": rng.choice([32, 64, 100, 128]), "H": rng.choice([2, 4]),
         "dh": rng.choice([16, 32, 64]), "L": rng.randint(1, 2)}
    c["ff"] = 4 * c["H"] * c["dh"]
    return dict(c, lr=0.05) if family == "step" else c


def transformer_params(c):
    """Names, shapes and spread (None: gains of 1) of the transformer's parameters, in their order: the embeddings' of
    uniform [-1, 1], the layers' of uniform [-1, 1] / sqrt(fan in), and LayerNorm's biases a little off 0."""
    d, ff = c["H"] * c["dh"], c["ff"]
    e, a, b = 1 / math.sqrt(3), 1 / math.sqrt(3 * d), 1 / math.sqrt(3 * ff)
    spec = [("tok", (c["V"], d), e), ("pos", (c["T"], d), e)]
    for layer in range(c["L"]):
        for name, shape, std in (("ln1.g", (d,), None), ("ln1.b", (d,), 0.02), ("wq", (d, d), a), ("wk", (d, d), a),
                                 ("wv", (d, d), a), ("wo", (d, d), a), ("bo", (d,), a), ("ln2.g", (d,), None),
                                 ("ln2.b", (d,), 0.02), ("w1", (d, ff), a), ("b1", (ff,), a), ("w2", (ff, d), b), ("b2", (d,), b)):
            spec.append((f"b{layer}.{name}", shape, std))
    return spec + [("lnf.g", (d,), None), ("lnf.b", (d,), 0.02), ("head", (d, c["V"]), a), ("headb", (c["V"],), a)]


def values(c, seed):
    """A case's inputs by name, in fp32: on the GPU, or for a training step's batch (x, y) what the host uploads."""
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, std=1.0):
        return torch.randn(*shape, generator=gen, device="cuda") * std

    def picked(n, among):
        return torch.nn.functional.one_hot(torch.randint(0, among, (n,), generator=gen, device="cuda"), among).float()

    f = c["family"]
    if f == "chain":
        v = {"x0": normal(c["R"], c["C"]), "x1": normal(c["R"], c["C"]), "r": normal(c["C"])}
        return dict(v, d0=normal(c["R"], c["C"])) if c["gradient"] else v
    if f == "softmax":
        # Logits of standard deviation 2; one row in a hundred far out, which only the max shift keeps finite.
        x = normal(c["R"], c["C"], std=2.0)
        x[torch.randperm(c["R"], generator=gen, device="cuda")[: round(c["R"] / 100)]] += 800
        return {"x": x, "d0": normal(c["R"], c["C"])} if c["gradient"] else {"x": x}
    if f == "layernorm":
        v = {"x": normal(c["R"], c["C"]), "gain": 1 + normal(c["C"], std=0.1), "bias": normal(c["C"], std=0.1)}
        return dict(v, d0=normal(c["R"], c["C"])) if c["gradient"] else v
    if f == "dense":
        s = 1 / math.sqrt(c["K"])
        v = {"X": normal(c["M"], c["K"], std=s), "W": normal(c["K"], c["N"], std=s), "bias": normal(c["N"], std=math.sqrt(0.1))}
        return dict(v, d0=normal(c["M"], c["N"])) if c["gradient"] else v
    if f == "attention":
        return {k: normal(c["B"], c["H"], c["T"], c["dh"]) for k in "qkv"}
    if f == "mlp":
        return {"W1": normal(c["inputs"], c["hidden"], std=1 / math.sqrt(c["inputs"])), "b1": torch.zeros(c["hidden"], device="cuda"),
                "W2": normal(c["hidden"], c["classes"], std=1 / math.sqrt(c["hidden"])), "b2": torch.zeros(c["classes"], device="cuda"),
                "x": torch.randint(0, 17, (c["batch"], c["inputs"]), generator=gen, device="cuda").float() / 16,
                "y": picked(c["batch"], c["classes"])}
    v = {name: torch.ones(shape, device="cuda") if std is None else normal(*shape, std=std) for name, shape, std in transformer_params(c)}
    return dict(v, x=picked(c["B"] * c["T"], c["V"]), y=picked(c["B"] * c["T"], c["V"]))


def prepare(case, seed):
    v = values(case, seed)
    plan = lower(case)
    if case["family"] in ("mlp", "step"):
        return Trainer(plan, {k: x for k, x in v.items() if k not in ("x", "y")}, v["x"].cpu().numpy(), v["y"].cpu().numpy())
    return Forward(plan, v)


def run(state):
    return state.step()


# ---- what a pass needs, and what it gives ----------------------------------------------------

def work(case):
    """Inputs read once and outputs written once, and the flops of the products."""
    c, f = case, case["family"]
    if f in ("chain", "softmax", "layernorm"):
        tensors = {"chain": (3, 6), "softmax": (2, 4), "layernorm": (2, 4)}[f][c["gradient"]]
        vectors = {"chain": (1, 2), "softmax": (0, 0), "layernorm": (2, 4)}[f][c["gradient"]]
        return {"bytes": 4 * (tensors * c["R"] * c["C"] + vectors * c["C"]), "flops": 0}
    if f == "dense":
        M, K, N = c["M"], c["K"], c["N"]
        if c["gradient"]:
            return {"bytes": 4 * (2 * M * K + 2 * K * N + 2 * N + 2 * M * N), "flops": 6 * M * K * N}
        return {"bytes": 4 * (M * K + K * N + N + M * N), "flops": 2 * M * K * N}
    if f == "attention":
        heads = c["B"] * c["H"]
        return {"bytes": 16 * heads * c["T"] * c["dh"], "flops": 4 * heads * c["T"] ** 2 * c["dh"]}
    if f == "mlp":
        params = c["inputs"] * c["hidden"] + c["hidden"] + c["hidden"] * c["classes"] + c["classes"]
        # The first layer's input has no gradient.
        return {"bytes": 4 * (2 * params + c["batch"] * (c["inputs"] + 2 * c["classes"])),
                "flops": 2 * c["batch"] * (2 * c["inputs"] * c["hidden"] + 3 * c["hidden"] * c["classes"])}
    rows, d = c["B"] * c["T"], c["H"] * c["dh"]
    params = sum(math.prod(shape) for _, shape, _ in transformer_params(c))
    layers = c["L"] * (2 * rows * (4 * d * d + 2 * d * c["ff"]) + 4 * c["B"] * c["T"] ** 2 * d)
    ends = 2 * rows * c["V"] * d
    if f == "forward":
        return {"bytes": 4 * (params + 3 * rows * c["V"]), "flops": layers + 2 * ends}
    return {"bytes": 4 * (2 * params + 3 * rows * c["V"]), "flops": 3 * layers + 5 * ends}


def tolerance(case):
    # 32-bit sums of up to 8192 terms: within 1.1e-6 of float64 (2-norm) over these ranges.
    return {"rel": 5e-6, "max": 2.5e-4}


def exact(case, seed):
    c, f = case, case["family"]
    v = {k: x.double() for k, x in values(case, seed).items()}

    def gradients(y, names):
        for n, g in zip(names, torch.autograd.grad(y, [v[n] for n in names], v["d0"], allow_unused=True)):
            out["d" + n] = torch.zeros_like(v[n]) if g is None else g
        return out

    if c.get("gradient"):
        for k in v:
            if k != "d0":
                v[k].requires_grad_()
    if f == "chain":
        y = chain_value(lower(case)["program"], v)
        out = {"y": y.detach()}
        return gradients(y, ["x0", "x1", "r"]) if c["gradient"] else out
    if f == "softmax":
        y = (torch.softmax if c["fn"] == "softmax" else torch.log_softmax)(v["x"], 1)
        out = {"y": y.detach()}
        return gradients(y, ["x"]) if c["gradient"] else out
    if f == "layernorm":
        y = torch.nn.functional.layer_norm(v["x"], (c["C"],), v["gain"], v["bias"], EPS)
        out = {"y": y.detach()}
        return gradients(y, ["x", "gain", "bias"]) if c["gradient"] else out
    if f == "dense":
        y = getattr(torch, c["act"])(v["X"] @ v["W"] + v["bias"])
        out = {"y": y.detach()}
        return gradients(y, ["X", "W", "bias"]) if c["gradient"] else out
    if f == "attention":
        return {"y": attend(v["q"], v["k"], v["v"])}
    if f == "forward":
        logits, loss = transformer(c, v)
        return {"logits": logits, "loss": loss}
    names = [k for k in v if k not in ("x", "y")]
    for k in names:
        v[k].requires_grad_()
    if f == "mlp":
        logits = torch.tanh(v["x"] @ v["W1"] + v["b1"]) @ v["W2"] + v["b2"]
        loss = -(v["y"] * torch.log_softmax(logits, 1)).sum() / c["batch"]
    else:
        logits, loss = transformer(c, v)
    grads = torch.autograd.grad(loss, [v[k] for k in names])
    return {"loss": loss.item(), "logits": logits.detach(), **{k: (v[k] - c["lr"] * g).detach() for k, g in zip(names, grads)}}


def chain_value(program, v):
    """An elementwise program's output in the inputs' precision."""
    ops = {"add": torch.add, "sub": torch.sub, "mul": torch.mul, "div": torch.div, "neg": torch.neg, "exp": torch.exp,
           "log": torch.log, "relu": torch.relu, "tanh": torch.tanh, "step": lambda x: (x > 0).to(x.dtype)}
    got = []
    for n in program["nodes"]:
        ins = [got[i] for i in n["inputs"]]
        if n["op"] == "input":
            got.append(v[n["attrs"]["name"]])
        elif n["op"] == "const":
            got.append(torch.tensor(n["attrs"]["value"], dtype=torch.float64, device="cuda").reshape(n["shape"]))
        elif n["op"] == "broadcast":
            got.append(ins[0].expand(n["shape"]))
        else:
            got.append(ops[n["op"]](*ins))
    return got[program["output"]]


def attend(q, k, v):
    T = q.shape[2]
    mask = torch.full((T, T), MASK, dtype=q.dtype, device=q.device).triu(1)
    s = q @ k.transpose(2, 3).contiguous() / math.sqrt(q.shape[3]) + mask
    return torch.softmax(s, 3) @ v


def transformer(c, v):
    d = c["H"] * c["dh"]

    def norm(x, name):
        return torch.nn.functional.layer_norm(x, (d,), v[name + ".g"], v[name + ".b"], EPS)

    def heads(x):
        return x.reshape(c["B"], c["T"], c["H"], c["dh"]).transpose(1, 2).contiguous()

    h = ((v["x"] @ v["tok"]).reshape(c["B"], c["T"], d) + v["pos"]).reshape(-1, d)
    for i in range(c["L"]):
        p = f"b{i}."
        a = norm(h, p + "ln1")
        o = attend(heads(a @ v[p + "wq"]), heads(a @ v[p + "wk"]), heads(a @ v[p + "wv"]))
        h = h + o.transpose(1, 2).reshape(-1, d) @ v[p + "wo"] + v[p + "bo"]
        m = norm(h, p + "ln2")
        h = h + torch.relu(m @ v[p + "w1"] + v[p + "b1"]) @ v[p + "w2"] + v[p + "b2"]
    logits = norm(h, "lnf") @ v["head"] + v["headb"]
    return logits, -(v["y"] * torch.log_softmax(logits, 1)).sum() / (c["B"] * c["T"])
