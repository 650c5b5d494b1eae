"""Performance cases of the simulator: what its users run, through the public Python API.

Four kinds of work, each over the range it is used at:

* ``circuit``: a compiled circuit is run from |0...0> on a resident state and
  read out (expectation values, the 16 most probable outcomes, measurement
  shots, or the whole state), in every execution mode and both precisions.
* ``batch``: a fixed set of ansatz circuits of uneven sizes, captured once and
  replayed (parameter sweeps).
* ``serve``: requests submitted to an engine that compiles, batches and answers
  them; their compilation is part of a pass, as it is for a served request.
* ``readout``: one readout of a state that is already in device memory.

``prepare`` makes what a program holds before the call: the circuit compiled,
the batch captured, the engine created with the requests' circuits built, the
state uploaded.  Values that derive from a complex64 state are returned in
single precision, the precision they are computed from.
"""
import math
import random

import numpy as np
import torch

import hyquas_amd as hq

TWO_PI = 2 * math.pi


# ---- the cases ----------------------------------------------------------------

def _circuit(name, family, qubits, layers, precision="c128", mode="mix", output="expect", mat=0):
    c = dict(kind="circuit", family=family, qubits=qubits, layers=layers, precision=precision, mode=mode,
             output=output, mat=mat)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # inner step of a variational optimiser on a small problem: latency and launches
        _circuit("ansatz_10q_c128_expect", "ansatz", 10, 6),
        # odd size in single precision, asked for its most probable outcomes
        _circuit("random_17q_c64_topk", "random", 17, 25, "c64", output="topk"),
        # the 20-qubit, 20-layer configuration, sampled as a device run would be
        _circuit("random_20q_c128_sample", "random", 20, 20, output="sample"),
        # the same configuration by the plain method (one pass per gate), all amplitudes returned
        _circuit("random_20q_c128_plain", "random", 20, 20, mode="serial", output="state"),
        # a mid-size run on specialised kernels
        _circuit("random_25q_c128_expect", "random", 25, 24),
        # the headline configuration: 30 qubits, 30 layers, complex128
        _circuit("random_30q_c128_expect", "random", 30, 30),
        # the precision form's circuit (24 layers, complex64) with matrix groups on the matrix cores
        _circuit("random_28q_c64_matrix", "random", 28, 12, "c64", mode="blas", mat=6),
        # the precision form's circuit on gate-group kernels
        _circuit("random_31q_c64_expect", "random", 31, 24, "c64"),
        # parameter sweep: ansatz circuits of 10..22 qubits, depth 4..40, replayed as one batch
        dict(name="batch_256_c64", kind="batch", circuits=256, nmin=10, nmax=22, spec=0, precision="c64"),
        # a burst of requests, 12..26 qubits, up to 60 layers, half asking for the top 16
        dict(name="serve_40_c64", kind="serve", requests=40, nmin=12, nmax=26, spec=1, precision="c64"),
        # 100 000 measurement shots of a state in device memory
        dict(name="sample_25q_c128", kind="readout", op="sample", qubits=25, precision="c128", shots=100000),
        # the readouts of one large single-precision state: <Z>, <ZZ>, norm, top 16
        dict(name="readout_28q_c64", kind="readout", op="all", qubits=28, precision="c64", shots=0),
    ]


def draw(rng):
    kind = rng.choices(["circuit", "readout", "serve", "batch"], [10, 5, 3, 2])[0]
    precision = rng.choice(["c128", "c64"])
    if kind == "circuit":
        mode = rng.choices(["mix", "serial", "blas"], [7, 1, 2])[0]
        if mode == "serial":
            n, layers, out = rng.randint(9, 24), rng.randint(6, 20), rng.choice(["expect", "state"])
            out = out if n <= 22 else "expect"
        elif mode == "blas":
            n, layers, out = rng.randint(13, 28), rng.randint(6, 14), "expect"
        else:
            n = rng.randint(8, 29 if precision == "c128" else 30)
            out = rng.choice(["expect", "topk", "sample"] if precision == "c128" else ["expect", "topk"])
            # outcomes of shallow circuits can be equally probable: their order would be rounding alone
            layers = rng.randint(16 if out == "topk" else 6, 40 if n <= 26 else 24)
        return _circuit(None, rng.choice(["random", "ansatz"]), n, layers, precision, mode, out,
                        rng.randint(4, 7) if mode == "blas" else 0)
    if kind == "readout":
        op = rng.choice(["expect", "topk", "norm", "zero", "inner", "sample", "all"])
        return dict(kind=kind, op=op, qubits=rng.randint(11, 27 if precision == "c128" else 28),
                    precision=precision, shots=int(10 ** rng.uniform(1, 5)) if op == "sample" else 0)
    if kind == "serve":
        return dict(kind=kind, requests=rng.randint(3, 36), nmin=12, nmax=rng.randint(16, 25),
                    spec=rng.randrange(1 << 30), precision=precision)
    return dict(kind=kind, circuits=int(2 ** rng.uniform(3, 7)), nmin=10, nmax=rng.randint(14, 22),
                spec=rng.randrange(1 << 30), precision=precision)


# ---- circuits: lists of (gate, qubits, angle) -----------------------------------------

def _random_layers(n, layers, seed):
    """Each layer: one of H, RX, RY, RZ, T on every qubit, then CNOTs on a random perfect matching."""
    r = np.random.default_rng(seed)
    gates = []
    for _ in range(layers):
        kind = r.integers(0, 5, n)
        angle = r.uniform(0, TWO_PI, n)
        for q in range(n):
            g = ("h", "rx", "ry", "rz", "t")[kind[q]]
            gates.append((g, (q,), float(angle[q]) if g[0] == "r" else None))
        p = [int(x) for x in r.permutation(n)]
        gates += [("cx", (p[i], p[i + 1]), None) for i in range(0, n - 1, 2)]
    return gates


def _ansatz_angles(n, layers, seed):
    return np.random.default_rng(seed).uniform(0, TWO_PI, (layers, n, 2))


def _ansatz_layers(n, layers, seed):
    """Each layer: RY and RZ on every qubit, then a CZ ladder."""
    a = _ansatz_angles(n, layers, seed)
    gates = []
    for d in range(layers):
        for q in range(n):
            gates.append(("ry", (q,), float(a[d, q, 0])))
            gates.append(("rz", (q,), float(a[d, q, 1])))
        gates += [("cz", (q, q + 1), None) for q in range(n - 1)]
    return gates


def _gates(family, n, layers, seed):
    return _random_layers(n, layers, seed) if family == "random" else _ansatz_layers(n, layers, seed)


def _build(n, gates):
    lines = ["OPENQASM 2.0;", 'include "qelib1.inc";', "qreg q[%d];" % n]
    for g, q, a in gates:
        lines.append("%s%s %s;" % (g, "" if a is None else "(%r)" % a, ",".join("q[%d]" % x for x in q)))
    return hq.Circuit.from_qasm("\n".join(lines) + "\n")


def _log_uniform_int(r, lo, hi):
    return int(round(math.exp(r.uniform(math.log(lo), math.log(hi)))))


def _batch_specs(case):
    r = random.Random(case["spec"])
    return [(_log_uniform_int(r, case["nmin"], case["nmax"]), r.randint(4, 40)) for _ in range(case["circuits"])]


def _serve_specs(case):
    r = random.Random(case["spec"])
    out = []
    for _ in range(case["requests"]):
        n = _log_uniform_int(r, case["nmin"], case["nmax"])
        # single-precision circuits of up to 13 qubits stay below 40 layers: deeper ones leave float's range
        depth = r.randint(8, 60 if n > 13 else 40)
        out.append((r.choice(["random", "ansatz"]), n, depth, r.random() < 0.5))
    return out


def _sub(seed, i):
    return [int(seed) & 0xffffffff, i]


def _precision(case):
    return hq.HQ_C128 if case["precision"] == "c128" else hq.HQ_C64


def _typed(case, x):
    return np.asarray(x, dtype=np.float64 if case["precision"] == "c128" else np.float32)


# ---- states of a readout --------------------------------------------------------------

def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _amplitudes(case, seed, which=0):
    """A normalised state of normally distributed amplitudes, as a random circuit leaves."""
    g = torch.Generator(device=_device()).manual_seed((int(seed) * 2 + which) & 0x7fffffff)
    real = torch.float64 if case["precision"] == "c128" else torch.float32
    x = torch.randn((1 << case["qubits"], 2), generator=g, dtype=real, device=_device())
    x /= math.sqrt(2.0 * (1 << case["qubits"]))
    return torch.view_as_complex(x)


# ---- one pass ------------------------------------------------------------------------

MODES = {"mix": hq.HQ_MODE_MIX, "serial": hq.HQ_MODE_SERIAL, "blas": hq.HQ_MODE_BLAS}


def prepare(case, seed):
    if case["kind"] == "circuit":
        c = _build(case["qubits"], _gates(case["family"], case["qubits"], case["layers"], _sub(seed, 0)))
        c.set_option("mode", MODES[case["mode"]])
        c.set_option("precision", _precision(case))
        if case["mat"]:
            c.set_option("blas_mat", case["mat"])
        c.compile()
        c.run(copy_back=False, destroy=False)
        return dict(case=case, circuit=c, seed=int(seed) & 0xffff)
    if case["kind"] == "batch":
        e = hq.Engine(_precision(case), 32 << 30)
        e.set_option("jit", 1)
        e.set_option("compile_threads", 8)
        cs = [_build(n, _ansatz_layers(n, d, _sub(seed, i))) for i, (n, d) in enumerate(_batch_specs(case))]
        return dict(case=case, engine=e, batch=e.batch(cs))
    if case["kind"] == "serve":
        e = hq.Engine(_precision(case), 64 << 30)
        e.set_option("compile_threads", 8)
        req = [(_build(n, _gates(f, n, d, _sub(seed, i))), topk) for i, (f, n, d, topk) in
               enumerate(_serve_specs(case))]
        return dict(case=case, engine=e, requests=req)
    s = hq.State(case["qubits"], _precision(case))
    s.upload(_amplitudes(case, seed).cpu().numpy())
    other = None
    if case["op"] == "inner":
        other = hq.State(case["qubits"], _precision(case))
        other.upload(_amplitudes(case, seed, 1).cpu().numpy())
    return dict(case=case, state=s, other=other, seed=int(seed) & 0xffff)


def _read(case, s, op, seed, shots, other=None):
    if op == "expect":
        z, zz = s.expect_z()
        return dict(z=_typed(case, z), zz=_typed(case, zz))
    if op == "topk":
        idx, prob = s.topk(16)
        return dict(idx=np.array(idx, dtype=np.int64), prob=_typed(case, prob))
    if op == "sample":
        return dict(shots=s.sample(shots, seed).astype(np.int64))
    if op == "state":
        return dict(state=s.download())
    if op == "norm":
        return dict(norm=_typed(case, [s.norm2()]))
    if op == "zero":
        return dict(zero=_typed(case, [s.measure_zero(q) for q in range(0, s.n, 3)]))
    if op == "inner":
        v = s.inner(other)
        return dict(inner=_typed(case, [v.real, v.imag]))
    out = _read(case, s, "expect", seed, 0)
    out.update(_read(case, s, "norm", seed, 0))
    out.update(_read(case, s, "topk", seed, 0))
    return out


def run(state):
    case = state["case"]
    if case["kind"] == "circuit":
        c = state["circuit"]
        c.run(copy_back=False, destroy=False)
        return _read(case, c.state_view(_precision(case)), case["output"], state["seed"], 4096)
    if case["kind"] == "batch":
        state["batch"].run()
        e3, _ = state["batch"].results()
        return dict(expect=_typed(case, e3))
    if case["kind"] == "serve":
        e = state["engine"]
        jobs = [e.submit(c, hq.HQ_OUT_EXPECT | (hq.HQ_OUT_TOPK if topk else 0)) for c, topk in state["requests"]]
        e.drain()
        e.poll()
        expect, idx, prob = [], [], []
        for j, (_, topk) in zip(jobs, state["requests"]):
            r = e.result(j, topk=topk)
            expect.append([r["norm"], r["z"], r["zz"]])
            if topk:
                idx.append(r["topk"][0])
                prob.append(r["topk"][1])
            e.release(j)
        return dict(expect=_typed(case, expect), idx=np.array(idx, dtype=np.int64), prob=_typed(case, prob))
    return _read(case, state["state"], case["op"], state["seed"], case["shots"], state["other"])


# ---- what a pass cannot do without -------------------------------------------------------

# real operations per amplitude: rotations and H are real 2x2 forms, RZ one
# complex product, T one on half the amplitudes, CZ a sign on a quarter
_OPS = {"h": 4, "rx": 6, "ry": 6, "rz": 6, "t": 3, "cx": 0, "cz": 0.5}


def _circuit_flops(family, n, layers):
    if family == "ansatz":
        per = n * (_OPS["ry"] + _OPS["rz"]) + (n - 1) * _OPS["cz"]
    else:
        per = n * sum(_OPS[g] for g in ("h", "rx", "ry", "rz", "t")) / 5
    return per * layers * 2.0 ** n


def work(case):
    amp = 16 if case["precision"] == "c128" else 8
    if case["kind"] == "circuit":
        # a run starts from |0...0>, so the state is written and, for its readout, read
        n = case["qubits"]
        return {"bytes": 2.0 * amp * 2.0 ** n, "flops": _circuit_flops(case["family"], n, case["layers"])}
    if case["kind"] == "batch":
        specs = _batch_specs(case)
        return {"bytes": float(sum(24 + 16 * n * d for n, d in specs)),
                "flops": sum(_circuit_flops("ansatz", n, d) for n, d in specs)}
    if case["kind"] == "serve":
        specs = _serve_specs(case)
        return {"bytes": float(sum(24 + 16 * n * d + (2 * amp * 2 ** n if topk else 0) for _, n, d, topk in specs)),
                "flops": sum(_circuit_flops(f, n, d) for f, n, d, _ in specs)}
    size = amp * 2.0 ** case["qubits"] * (2 if case["op"] == "inner" else 1)
    return {"bytes": size + 16.0 * case["shots"], "flops": (8.0 if case["op"] == "inner" else 3.0) * 2.0 ** case["qubits"]}


# ---- the same in 64 bits, with torch alone ---------------------------------------------------

def _apply(psi, gate):
    name, q, a = gate
    if name in ("cx", "cz"):
        lo, hi = min(q), max(q)
        v = psi.view(-1, 2, 1 << (hi - lo - 1), 2, 1 << lo)   # dims 1 and 3: the higher and the lower qubit
        if name == "cz":
            v[:, 1, :, 1] *= -1
            return
        if q[0] == hi:
            t = v[:, 1, :, 0].clone()
            v[:, 1, :, 0] = v[:, 1, :, 1]
            v[:, 1, :, 1] = t
        else:
            t = v[:, 0, :, 1].clone()
            v[:, 0, :, 1] = v[:, 1, :, 1]
            v[:, 1, :, 1] = t
        return
    v = psi.view(-1, 2, 1 << q[0])
    if name == "t":
        v[:, 1] *= complex(math.sqrt(0.5), math.sqrt(0.5))
        return
    if name == "rz":
        v[:, 0] *= complex(math.cos(a / 2), -math.sin(a / 2))
        v[:, 1] *= complex(math.cos(a / 2), math.sin(a / 2))
        return
    if name == "h":
        r = math.sqrt(0.5)
        m = (r, r, r, -r)
    else:
        c, s = math.cos(a / 2), math.sin(a / 2)
        m = (c, -s, s, c) if name == "ry" else (c, -1j * s, -1j * s, c)
    x, y = v[:, 0].clone(), v[:, 1].clone()
    v[:, 0] = m[0] * x + m[1] * y
    v[:, 1] = m[2] * x + m[3] * y


def _simulate(n, gates):
    psi = torch.zeros(1 << n, dtype=torch.complex128, device=_device())
    psi[0] = 1
    for g in gates:
        _apply(psi, g)
    return psi


def _probabilities(psi):
    x = torch.view_as_real(psi).double()
    return x[..., 0].square() + x[..., 1].square()


def _expect(p, n):
    z, zz = [], []
    for q in range(n):
        s = p.view(-1, 2, 1 << q).sum((0, 2))
        z.append(float(s[0] - s[1]))
        if q + 1 < n:
            s = p.view(-1, 2, 2, 1 << q).sum((0, 3))
            zz.append(float(s[0, 0] + s[1, 1] - s[0, 1] - s[1, 0]))
    return z, zz


def _exact_read(psi, n, op, other=None):
    p = _probabilities(psi)
    if op == "expect":
        z, zz = _expect(p, n)
        return dict(z=np.array(z), zz=np.array(zz))
    if op == "topk":
        return dict(idx=None, prob=torch.topk(p, 16).values.cpu().numpy())
    if op == "state":
        return dict(state=psi.cpu().numpy())
    if op == "norm":
        return dict(norm=np.array([float(p.sum())]))
    if op == "zero":
        return dict(zero=np.array([float(p.view(-1, 2, 1 << q)[:, 0].sum()) for q in range(0, n, 3)]))
    if op == "inner":
        v = complex((psi.to(torch.complex128).conj() * other.to(torch.complex128)).sum())
        return dict(inner=np.array([v.real, v.imag]))
    out = _exact_read(psi, n, "expect")
    out.update(_exact_read(psi, n, "norm"))
    out.update(_exact_read(psi, n, "topk"))
    return out


def _exact_batch(case, seed):
    """Circuits of one size advance together, deepest first, so that the active ones are a leading slice."""
    specs = _batch_specs(case)
    out = np.zeros((len(specs), 3))
    for n in sorted({s[0] for s in specs}):
        idx = sorted((i for i, s in enumerate(specs) if s[0] == n), key=lambda i: -specs[i][1])
        bits = torch.arange(1 << n, device=_device())
        sign = torch.ones(1 << n, dtype=torch.float64, device=_device())
        for q in range(n - 1):
            sign *= 1 - 2 * ((bits >> q) & (bits >> (q + 1)) & 1).double()
        step = max(1, (1 << 26) >> n)
        for at in range(0, len(idx), step):
            part = idx[at:at + step]
            depth = [specs[i][1] for i in part]
            ang = np.zeros((len(part), depth[0], n, 2))
            for k, i in enumerate(part):
                ang[k, :depth[k]] = _ansatz_angles(n, depth[k], _sub(seed, i))
            ang = torch.from_numpy(ang / 2).to(_device())
            cos, sin = ang.cos(), ang.sin()
            psi = torch.zeros((len(part), 1 << n), dtype=torch.complex128, device=_device())
            psi[:, 0] = 1
            for d in range(depth[0]):
                m = sum(1 for x in depth if x > d)
                for q in range(n):
                    v = psi[:m].view(m, -1, 2, 1 << q)
                    c, s = cos[:m, d, q, 0].view(m, 1, 1), sin[:m, d, q, 0].view(m, 1, 1)
                    f = torch.complex(cos[:m, d, q, 1], sin[:m, d, q, 1]).view(m, 1, 1)
                    x, y = v[:, :, 0].clone(), v[:, :, 1].clone()
                    v[:, :, 0] = (c * x - s * y) * f.conj()
                    v[:, :, 1] = (s * x + c * y) * f
                psi[:m] *= sign
            p = _probabilities(psi)
            for k, i in enumerate(part):
                z, zz = _expect(p[k].contiguous(), n)
                out[i] = float(p[k].sum()), sum(z), sum(zz)
    return dict(expect=out)


def exact(case, seed):
    if case["kind"] == "circuit":
        n = case["qubits"]
        if case["output"] == "sample" or n > 27 or (n > 25 and case["layers"] > 16):
            return None   # shots are whole numbers; larger circuits take minutes of torch passes
        return _exact_read(_simulate(n, _gates(case["family"], n, case["layers"], _sub(seed, 0))), n, case["output"])
    if case["kind"] == "batch":
        return _exact_batch(case, seed)
    if case["kind"] == "serve":
        expect, prob = [], []
        for i, (f, n, d, topk) in enumerate(_serve_specs(case)):
            p = _probabilities(_simulate(n, _gates(f, n, d, _sub(seed, i))))
            z, zz = _expect(p, n)
            expect.append([float(p.sum()), sum(z), sum(zz)])
            if topk:
                prob.append(torch.topk(p, 16).values.cpu().numpy())
        return dict(expect=np.array(expect), idx=None, prob=np.array(prob))
    if case["op"] == "sample":
        return None   # whole numbers
    other = _amplitudes(case, seed, 1) if case["op"] == "inner" else None
    return _exact_read(_amplitudes(case, seed), case["qubits"], case["op"], other)
