"""The work that users of the engine have it do, as measurable cases.

Kinds (a case's "kind"):
  circuit   a tape applied to a resident state: gate by gate (apply_tape), as
            tile passes (apply_tape_tiled) or as fused matrix-core blocks
            (apply_tape_fused); the state goes on from pass to pass
  expval    <H> of a Hamiltonian of random Pauli strings of weight 1..4
  readout   samples from given uniforms and a marginal distribution
  adjoint   a whole gradient: |0...0>, the forward pass, every expectation
            value and the adjoint Jacobian
  vjp       the forward pass and a vector-Jacobian product
  batch     energies and gradients of many layered circuits in one replay
  mlp       Adam steps of the surrogate network and a screening prediction

Inputs come from the seed alone; `exact` repeats the computation in torch at
64 bits from the definitions of the gates.
"""
import math
import random

import numpy as np
import torch

from lightning_unification_amd import capi
from lightning_unification_amd.circuits import Obs, Tape, pauli_word, tfim

# gates of the large random circuits, and those with one parameter and a
# generator, which the gradients take
MIX = ["Hadamard", "T", "RX", "RY", "RZ", "Rot", "CRX", "CRZ", "IsingXX", "IsingZZ", "SWAP", "Toffoli"]
GRAD_MIX = ["Hadamard", "T", "RX", "RY", "RZ", "CRX", "CRZ", "IsingXX", "IsingZZ", "SWAP", "CNOT"]
ARITY = {"Hadamard": 1, "T": 1, "RX": 1, "RY": 1, "RZ": 1, "Rot": 1, "CRX": 2, "CRZ": 2, "IsingXX": 2,
         "IsingZZ": 2, "SWAP": 2, "CNOT": 2, "Toffoli": 3}
NPARAMS = {"RX": 1, "RY": 1, "RZ": 1, "Rot": 3, "CRX": 1, "CRZ": 1, "IsingXX": 1, "IsingZZ": 1}


def listed():
    return [
        # the first thing anyone runs: a handful of qubits, a small ansatz and
        # its whole gradient; all latency
        {"name": "gradient_6q", "kind": "adjoint", "n": 6, "layers": 2, "obs": 6, "mix": False, "dtype": "c128"},
        # the plain workload: 20 qubits, 600 parameters, <Z> of every wire
        {"name": "gradient_20q", "kind": "adjoint", "n": 20, "layers": 10, "obs": 20, "mix": False,
         "dtype": "c128"},
        # a machine-learning layer's backward pass at single precision, mixed
        # gates, an odd qubit count
        {"name": "vjp_17q_c64", "kind": "vjp", "n": 17, "layers": 6, "mix": True, "dtype": "c64"},
        # single gates streaming over a large state, the headline's operation
        {"name": "gates_28q", "kind": "circuit", "mode": "gates", "n": 28, "layers": 1, "dtype": "c128"},
        # the same calls where a gate is all launch
        {"name": "gates_13q_c64", "kind": "circuit", "mode": "gates", "n": 13, "layers": 10, "dtype": "c64"},
        # a deep circuit on a large state by tile passes
        {"name": "tiled_28q", "kind": "circuit", "mode": "tiled", "n": 28, "layers": 12, "dtype": "c128"},
        # the precision form: five-qubit blocks on FP32 matrix cores with FP64
        # renormalisation
        {"name": "fused_28q_c64", "kind": "circuit", "mode": "fused", "n": 28, "layers": 6, "dtype": "c64"},
        # energy of a 100-term Hamiltonian on a large state
        {"name": "expval_28q", "kind": "expval", "n": 28, "terms": 100, "dtype": "c128"},
        # a million shots and an 8-wire marginal
        {"name": "readout_27q_c64", "kind": "readout", "n": 27, "shots": 1000000, "wires": 8, "dtype": "c64"},
        # uneven circuits in one replay
        {"name": "batch_512", "kind": "batch", "count": 512, "nmin": 8, "nmax": 20, "dmin": 4, "dmax": 12,
         "dtype": "c128"},
        # one accepted optimiser step: a single 16-qubit, 6-layer circuit
        {"name": "batch_single_16q", "kind": "batch", "count": 1, "nmin": 16, "nmax": 16, "dmin": 6, "dmax": 6,
         "dtype": "c128"},
        # the surrogate: Adam steps of 192-512-512-193 and 256 candidates
        {"name": "surrogate", "kind": "mlp", "d0": 192, "hidden": 512, "batch": 1024, "steps": 16,
         "candidates": 256},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["circuit", "circuit", "circuit", "expval", "readout", "adjoint", "adjoint", "vjp", "batch",
                       "batch", "mlp"])
    dtype = rng.choice(["c128", "c64"])
    if kind == "circuit":
        mode = rng.choice(["gates", "tiled", "fused"])
        if mode == "fused":
            dtype = "c64"
        n = rng.randint(9, 27)
        return {"kind": kind, "mode": mode, "n": n, "layers": rng.randint(1, 12 if n < 24 else 4), "dtype": dtype}
    if kind == "expval":
        return {"kind": kind, "n": rng.randint(6, 27), "terms": _log_int(rng, 5, 150), "dtype": dtype}
    if kind == "readout":
        n = rng.randint(6, 27)
        return {"kind": kind, "n": n, "shots": _log_int(rng, 100, 1000000), "wires": rng.randint(1, min(n, 12)),
                "dtype": dtype}
    if kind == "adjoint":
        n = rng.randint(4, 20)
        return {"kind": kind, "n": n, "layers": rng.randint(1, 8), "obs": rng.randint(1, n),
                "mix": rng.random() < 0.4, "dtype": dtype}
    if kind == "vjp":
        return {"kind": kind, "n": rng.randint(4, 21), "layers": rng.randint(1, 8), "mix": rng.random() < 0.5,
                "dtype": dtype}
    if kind == "batch":
        lo = rng.randint(5, 14)
        dlo = rng.randint(2, 6)
        hi = rng.randint(lo, 18)
        return {"kind": kind, "count": _log_int(rng, 1, 512), "nmin": lo, "nmax": hi, "dmin": dlo,
                "dmax": rng.randint(dlo, 12), "dtype": dtype}
    d0 = rng.randint(20, 256)
    return {"kind": "mlp", "d0": d0, "hidden": rng.choice([64, 96, 128, 200, 256, 384, 512]),
            "batch": _log_int(rng, 64, 1024), "steps": rng.randint(4, 16), "candidates": rng.randint(1, 256)}


# ---- inputs -------------------------------------------------------------------

def _np_dtype(case):
    return np.complex128 if case["dtype"] == "c128" else np.complex64


def _torch_dtype(case):
    return torch.complex128 if case["dtype"] == "c128" else torch.complex64


def _random_ops(n, layers, gates, rng):
    """Each layer walks the shuffled wires, so every wire is touched once.
    The circuit is the case's own, its angles are the seed's."""
    shape, ops = random.Random(n * 100 + layers), []
    for _ in range(layers):
        order = list(range(n))
        shape.shuffle(order)
        while order:
            g = shape.choice([x for x in gates if ARITY[x] <= len(order)])
            w, order = order[:ARITY[g]], order[ARITY[g]:]
            ops.append((g, w, [rng.uniform(0, 2 * math.pi) for _ in range(NPARAMS.get(g, 0))]))
    return ops


def _plain_ops(n, layers, rng):
    """RX, RY, RZ on every wire, then a CNOT ladder."""
    ops = []
    for _ in range(layers):
        for w in range(n):
            for g in ("RX", "RY", "RZ"):
                ops.append((g, [w], [rng.uniform(0, 2 * math.pi)]))
        for i in range(n - 1):
            ops.append(("CNOT", [i, i + 1], []))
    return ops


def _ops(case, seed):
    rng = random.Random(seed)
    if case["kind"] == "circuit":
        return _random_ops(case["n"], case["layers"], MIX, rng)
    if case["mix"]:
        return _random_ops(case["n"], case["layers"], GRAD_MIX, rng)
    return _plain_ops(case["n"], case["layers"], rng)


def _tape(ops):
    t = Tape()
    for g, w, p in ops:
        t.add(g, w, p)
    return t


def _words(case, seed):
    """(coefficient, letters, wires) of each Hamiltonian term."""
    rng = random.Random(seed + 1)
    out = []
    for _ in range(case["terms"]):
        k = rng.randint(1, min(4, case["n"]))
        out.append((rng.gauss(0, 1), "".join(rng.choice("XYZ") for _ in range(k)), rng.sample(range(case["n"]), k)))
    return out


def _random_state(n, seed, dtype):
    """Normal amplitudes, the statistics of a deep circuit's state."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    v = torch.randn(1 << n, 2, generator=g, device="cuda", dtype=torch.float32)
    v = v.to(torch.float64 if dtype == torch.complex128 else torch.float32)
    v /= torch.linalg.vector_norm(v.reshape(-1), dtype=torch.float64).to(v.dtype)
    return torch.view_as_complex(v)


class _DeviceArray:
    """Names the state's memory to torch and, held by the tensor, keeps the
    state alive as long as any tensor on that memory is."""

    def __init__(self, sv):
        self.sv = sv
        self.__cuda_array_interface__ = {"shape": (sv.size,), "typestr": sv.dtype.str, "version": 3,
                                         "data": (sv.device_ptr(), False)}


def _view(sv):
    """The state's amplitudes as a tensor on the state's own memory."""
    return torch.as_tensor(_DeviceArray(sv), device="cuda")


def _resident(case, seed):
    sv = capi.DeviceStateVector(case["n"], _np_dtype(case))
    view = _view(sv)
    sv.synchronize()
    view.copy_(_random_state(case["n"], seed, _torch_dtype(case)))
    torch.cuda.synchronize()
    return sv, view


def _uniforms(case, seed):
    return np.random.default_rng(seed + 2).random(case["shots"])


def _marginal_wires(case, seed):
    return sorted(random.Random(seed + 3).sample(range(case["n"]), case["wires"]))


def _cotangent(case, seed):
    r = np.random.default_rng(seed + 4)
    v = r.standard_normal(1 << case["n"]) + 1j * r.standard_normal(1 << case["n"])
    return v / np.linalg.norm(v)


def _batch_inputs(case, seed):
    # shapes are the plan a program keeps (the same for every seed of a case);
    # fields too; angles are the call's input
    shape = random.Random(case["count"] * 1000 + case["nmin"] * 100 + case["nmax"])
    ns = [shape.randint(case["nmin"], case["nmax"]) for _ in range(case["count"])]
    ds = [shape.randint(case["dmin"], case["dmax"]) for _ in range(case["count"])]
    hs = [shape.uniform(0.5, 1.5) for _ in range(case["count"])]
    np_ = sum(2 * n * d for n, d in zip(ns, ds))
    return ns, ds, hs, np.random.default_rng(seed).random(np_) * 2 * math.pi


def _mlp_inputs(case, seed):
    r = np.random.default_rng(seed)
    d0, h, d3 = case["d0"], case["hidden"], case["d0"] + 1
    rows = case["batch"] * 4
    x = (2 * r.random((rows, d0)) - 1).astype(np.float32)
    # smooth targets of the features, standardised
    t = np.sin(x @ r.standard_normal((d0, d3)) * (2.0 / math.sqrt(d0)))
    t = ((t - t.mean(axis=0)) / t.std(axis=0)).astype(np.float32)
    p = []
    for a, b in ((d0, h), (h, h), (h, d3)):
        p += [((2 * r.random(a * b) - 1) * math.sqrt(6.0 / a)).astype(np.float32), np.zeros(b, np.float32)]
    cand = (2 * r.random((case["candidates"], d0)) - 1).astype(np.float32)
    return x, t, np.concatenate(p), cand


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "circuit":
        s["tape"] = _tape(_ops(case, seed))
        s["sv"], s["view"] = _resident(case, seed)
    elif kind == "expval":
        words = _words(case, seed)
        s["ham"] = Obs.hamiltonian([c for c, _, _ in words], [pauli_word(a, w) for _, a, w in words])
        s["sv"], s["view"] = _resident(case, seed)
    elif kind == "readout":
        s["u"], s["wires"] = _uniforms(case, seed), _marginal_wires(case, seed)
        s["sv"], s["view"] = _resident(case, seed)
    elif kind in ("adjoint", "vjp"):
        s["tape"] = _tape(_ops(case, seed))
        s["tp"] = list(range(s["tape"].num_params()))
        s["sv"] = capi.DeviceStateVector(case["n"], _np_dtype(case))
        if kind == "adjoint":
            s["obs"] = [Obs.named("PauliZ", [w]) for w in range(case["obs"])]
        else:
            s["dy"] = _cotangent(case, seed)
    elif kind == "batch":
        ns, ds, hs, s["params"] = _batch_inputs(case, seed)
        s["plan"] = capi.BatchPlan(ns, ds, "YZ", "ring", [tfim(n, 1.0, h) for n, h in zip(ns, hs)],
                                   dtype=_np_dtype(case))
    else:
        x, t, p, s["cand"] = _mlp_inputs(case, seed)
        s["net"] = capi.Mlp((case["d0"], case["hidden"], case["hidden"], case["d0"] + 1), 1024, seed)
        s["net"].set_params(p)
        s["net"].load_data(x, t)
    return s


# ---- one pass -----------------------------------------------------------------

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "circuit":
        if case["mode"] == "gates":
            s["sv"].apply_tape(s["tape"])
        elif case["mode"] == "tiled":
            s["sv"].apply_tape_tiled(s["tape"])
        else:
            s["sv"].apply_tape_fused(s["tape"], 5, renorm=True)
        return s["view"]
    if kind == "expval":
        return {"energy": s["sv"].expval(s["ham"])}
    if kind == "readout":
        return {"idx": s["sv"].sample(s["u"]), "probs": s["sv"].probs(s["wires"])}
    if kind == "adjoint":
        s["sv"].reset()
        s["sv"].apply_tape(s["tape"])
        return {"expvals": np.array([s["sv"].expval(o) for o in s["obs"]]),
                "jac": s["sv"].adjoint_jacobian(s["tape"], s["obs"], s["tp"])}
    if kind == "vjp":
        s["sv"].reset()
        s["sv"].apply_tape(s["tape"])
        return {"vjp": s["sv"].vjp(s["tape"], s["dy"], s["tp"])}
    if kind == "batch":
        e, g = s["plan"].run(s["params"])
        return {"energies": e, "grads": g}
    loss = s["net"].train(case["steps"], case["batch"], 1e-3)
    return {"loss": loss, "params": s["net"].params(), "predicted": s["net"].predict(s["cand"])}


# ---- what a pass cannot do without ---------------------------------------------

_FLOPS = {"Hadamard": 8, "T": 3, "RX": 8, "RY": 8, "RZ": 6, "Rot": 14, "CRX": 4, "CRZ": 3, "IsingXX": 8,
          "IsingZZ": 6, "SWAP": 0, "CNOT": 0, "Toffoli": 0}  # per amplitude of the state


def work(case):
    kind = case["kind"]
    amp = 0 if "dtype" not in case else (16 if case["dtype"] == "c128" else 8)
    if kind == "batch":
        ns, ds, _, p = _batch_inputs(case, 0)
        # per wire and layer: two rotations forward, then undone on two states
        # with their gradients; states fit nowhere but in memory for one pass each
        flops = sum((1 << n) * n * d * (14 + 2 * 14 + 20) for n, d in zip(ns, ds))
        return {"bytes": 16 * len(p) + 8 * len(ns) + sum((1 << n) * amp * 4 for n in ns), "flops": flops}
    if kind == "mlp":
        d0, h, d3 = case["d0"], case["hidden"], case["d0"] + 1
        weights = d0 * h + h * h + h * d3
        step = {"bytes": 28 * weights + case["batch"] * (2 * d0 + 4 * d3),
                "flops": 2 * case["batch"] * (3 * weights - d0 * h)}
        return {"bytes": case["steps"] * step["bytes"] + case["candidates"] * 4 * (d0 + d3) + 4 * weights,
                "flops": case["steps"] * step["flops"] + 2 * case["candidates"] * weights}
    size = 1 << case["n"]
    if kind == "circuit":
        return {"bytes": 2 * size * amp, "flops": sum(_FLOPS[g] * size for g, _, _ in _ops(case, 1))}
    if kind == "expval":
        return {"bytes": size * amp, "flops": 8 * size * case["terms"]}
    if kind == "readout":
        return {"bytes": size * amp + 16 * case["shots"], "flops": 4 * size}
    ops = _ops(case, 1)
    forward = sum(_FLOPS[g] * size for g, _, _ in ops)
    states = 1 + (case["obs"] if kind == "adjoint" else 1)
    return {"bytes": (size * amp + (0 if kind == "adjoint" else 16 * size)) + 8 * len(ops),
            "flops": forward * (1 + states) + sum(4 * size * (states - 1) for _, _, p in ops if p)}


# ---- the same in 64 bits, from the definitions of the gates ---------------------

def _matrix(g, p):
    i = 1j
    c, s = (math.cos(p[0] / 2), math.sin(p[0] / 2)) if p else (0, 0)
    if g == "Hadamard":
        return np.array([[1, 1], [1, -1]]) / math.sqrt(2)
    if g == "T":
        return np.diag([1, np.exp(i * math.pi / 4)])
    if g == "RX":
        return np.array([[c, -i * s], [-i * s, c]])
    if g == "RY":
        return np.array([[c, -s], [s, c]], complex)
    if g == "RZ":
        return np.diag([c - i * s, c + i * s])
    if g == "Rot":
        return _matrix("RZ", [p[2]]) @ _matrix("RY", [p[1]]) @ _matrix("RZ", [p[0]])
    if g in ("CRX", "CRZ"):
        m = np.eye(4, dtype=complex)
        m[2:, 2:] = _matrix(g[1:], p)
        return m
    if g == "IsingXX":
        return np.eye(4) * c - i * s * np.eye(4)[::-1]
    if g == "IsingZZ":
        return np.diag([c - i * s, c + i * s, c + i * s, c - i * s])
    if g == "SWAP":
        return np.eye(4)[[0, 2, 1, 3]]
    if g == "CNOT":
        return np.eye(4)[[0, 1, 3, 2]]
    if g == "Toffoli":
        return np.eye(8)[[0, 1, 2, 3, 4, 5, 7, 6]]
    raise ValueError(g)


def _generator(g):
    """G of U = exp(-i theta/2 G)."""
    x, z = np.array([[0, 1], [1, 0]]), np.diag([1, -1])
    if g in ("RX", "CRX"):
        m = x
    elif g in ("RZ", "CRZ"):
        m = z
    elif g == "RY":
        m = np.array([[0, -1j], [1j, 0]])
    else:
        return np.kron(x, x) if g == "IsingXX" else np.kron(z, z)
    return np.kron(np.diag([0, 1]), m) if g[0] == "C" else m


def _apply(v, n, m, wires):
    """m on `wires` (the first is its index's highest bit) of states v[batch, 2^n]; a new tensor."""
    order = sorted(wires)
    shape, last = [v.shape[0]], 0
    for w in order:
        shape += [1 << (w - last), 2]
        last = w + 1
    a = v.reshape(shape + [1 << (n - last)])
    k = len(wires)

    def part(t, idx):
        sel = [slice(None)] * t.dim()
        for j, w in enumerate(wires):
            sel[2 + 2 * order.index(w)] = (idx >> (k - 1 - j)) & 1
        return t[tuple(sel)]

    out = torch.zeros_like(a)
    for r in range(1 << k):
        for c in range(1 << k):
            if m[r, c] != 0:
                part(out, r).add_(part(a, c), alpha=complex(m[r, c]))
    return out.reshape(v.shape)


def _zero_state(n, batch=1):
    v = torch.zeros(batch, 1 << n, dtype=torch.complex128, device="cuda")
    v[:, 0] = 1
    return v


def _signs(n, wire):
    i = torch.arange(1 << n, device="cuda")
    return (1 - 2 * ((i >> (n - 1 - wire)) & 1)).to(torch.float64)


def _exact_sweep(n, ops, lam, bras):
    """<bra_k| G lambda> of every parametrised op in tape order, (parameters, bras)."""
    both, got = torch.cat([lam, bras]), []
    for g, w, p in reversed(ops):
        if p:
            gl = _apply(both[:1], n, _generator(g), w)
            got.append(torch.stack([torch.vdot(b, gl[0]) for b in both[1:]]))
        both = _apply(both, n, np.conj(_matrix(g, p)).T, w)
    return torch.stack(got[::-1]) if got else torch.zeros(0, len(bras), dtype=torch.complex128)


def _exact_words(case, seed, psi):
    n, total, chunk = case["n"], 0.0, 1 << min(case["n"], 24)
    for coeff, letters, wires in _words(case, seed):
        x = sum(1 << (n - 1 - w) for a, w in zip(letters, wires) if a in "XY")
        z = [n - 1 - w for a, w in zip(letters, wires) if a in "YZ"]
        acc = 0.0
        for at in range(0, 1 << n, chunk):
            i = torch.arange(at, at + chunk, device="cuda")
            par = torch.zeros_like(i)
            for b in z:
                par ^= (i >> b) & 1
            acc += complex((psi[at:at + chunk].conj() * psi[i ^ x] * (1 - 2 * par)).sum())
        total += coeff * (acc * (-1j) ** letters.count("Y")).real
    return total


def _exact_batch(case, seed):
    ns, ds, hs, params = _batch_inputs(case, seed)
    starts = np.concatenate([[0], np.cumsum([2 * n * d for n, d in zip(ns, ds)])])
    energies, grads = np.zeros(len(ns)), np.zeros(len(params))
    groups = {}
    for j, key in enumerate(zip(ns, ds)):
        groups.setdefault(key, []).append(j)
    for (n, d), members in groups.items():
        for at in range(0, len(members), max(1, (1 << 25) >> n)):
            js = members[at:at + max(1, (1 << 25) >> n)]
            th = torch.tensor(np.stack([params[starts[j]:starts[j + 1]] for j in js]), device="cuda")
            th = th.reshape(len(js), d, n, 2)
            h = torch.tensor([hs[j] for j in js], dtype=torch.float64, device="cuda")
            # the ring of CNOTs as an index map: out[ring(i)] = in[i]
            i = torch.arange(1 << n, device="cuda")
            ring = i.clone()
            for w in range(n if n > 1 else 0):
                ring ^= ((ring >> (n - 1 - w)) & 1) << (n - 1 - (w + 1) % n)
            back = torch.empty_like(ring)
            back[ring] = i

            def rotate(v, w, layer, dagger):
                c = torch.cos(th[:, layer, w] / 2)
                s = torch.sin(th[:, layer, w] / 2) * (-1 if dagger else 1)
                a = v.reshape(len(js), -1, 1 << w, 2, 1 << (n - 1 - w))
                cy, sy = (t[:, 0].reshape(-1, 1, 1, 1) for t in (c, s))
                ph = (c[:, 1] - 1j * s[:, 1]).reshape(-1, 1, 1, 1)
                v0, v1 = a[..., 0, :], a[..., 1, :]
                if dagger:
                    v0, v1 = v0 * ph, v1 * ph.conj()
                    out = (cy * v0 - sy * v1, sy * v0 + cy * v1)
                else:
                    out = ((cy * v0 - sy * v1) * ph, (sy * v0 + cy * v1) * ph.conj())
                return torch.stack(out, dim=-2).reshape(v.shape)

            psi = _zero_state(n, len(js)).reshape(len(js), 1, -1)
            for layer in range(d):
                for w in range(n):
                    psi = rotate(psi, w, layer, False)
                psi = psi[..., back]
            zz = sum(_signs(n, w) * _signs(n, (w + 1) % n) for w in range(n))
            hp = -psi * zz
            for w in range(n):
                hp = hp - h.reshape(-1, 1, 1) * psi[..., i ^ (1 << (n - 1 - w))]
            e = (psi.conj() * hp).sum(-1).real.reshape(-1).cpu().numpy()
            both, g = torch.cat([psi, hp], dim=1), torch.zeros_like(th)
            for layer in reversed(range(d)):
                both = both[..., ring]
                for w in range(n):
                    a = both.reshape(len(js), 2, 1 << w, 2, 1 << (n - 1 - w))
                    l, k = a[:, 0], a[:, 1].conj()
                    g[:, layer, w, 1] = (k[:, :, 0] * l[:, :, 0] - k[:, :, 1] * l[:, :, 1]).sum((1, 2)).imag
                    s2, c2 = torch.sin(th[:, layer, w, 1]), torch.cos(th[:, layer, w, 1])
                    k0l1, k1l0 = (k[:, :, 0] * l[:, :, 1]).sum((1, 2)), (k[:, :, 1] * l[:, :, 0]).sum((1, 2))
                    # Y before the Z rotation is Y cos - X sin after it
                    g[:, layer, w, 0] = (c2 * (-1j * k0l1 + 1j * k1l0) - s2 * (k0l1 + k1l0)).imag
                    both = rotate(both, w, layer, True)
            for m, j in enumerate(js):
                energies[j] = e[m]
                grads[starts[j]:starts[j + 1]] = g[m].reshape(-1).cpu().numpy()
    return {"energies": energies, "grads": grads}


def _exact_mlp(case, seed):
    x, t, p, cand = (torch.tensor(a, dtype=torch.float64, device="cuda") for a in _mlp_inputs(case, seed))
    d0, h, d3, at, layers = case["d0"], case["hidden"], case["d0"] + 1, 0, []
    for a, b in ((d0, h), (h, h), (h, d3)):
        layers += [p[at:at + a * b].reshape(a, b).clone(), p[at + a * b:at + a * b + b].clone()]
        at += a * b + b
    for q in layers:
        q.requires_grad_(True)

    def net(v):
        v = torch.nn.functional.gelu(v @ layers[0] + layers[1])
        v = torch.nn.functional.gelu(v @ layers[2] + layers[3])
        return v @ layers[4] + layers[5]

    m1, m2 = [torch.zeros_like(q) for q in layers], [torch.zeros_like(q) for q in layers]
    loss_sum, cursor, b = 0.0, 0, case["batch"]
    for step in range(1, case["steps"] + 1):
        if cursor + b > len(x):
            cursor = 0
        loss = ((net(x[cursor:cursor + b]) - t[cursor:cursor + b]) ** 2).sum() / b
        cursor += b
        loss_sum += float(loss)
        for q, a, v, g in zip(layers, m1, m2, torch.autograd.grad(loss, layers)):
            a.mul_(0.9).add_(g, alpha=0.1)
            v.mul_(0.999).add_(g * g, alpha=0.001)
            with torch.no_grad():
                q -= 1e-3 * (a / (1 - 0.9 ** step)) / ((v / (1 - 0.999 ** step)).sqrt() + 1e-8)
    with torch.no_grad():
        return {"loss": loss_sum / case["steps"], "params": torch.cat([q.reshape(-1) for q in layers]),
                "predicted": net(cand)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return _exact_batch(case, seed)
    if kind == "mlp":
        return _exact_mlp(case, seed)
    n = case["n"]
    if kind in ("circuit", "expval", "readout"):
        psi = _random_state(n, seed, _torch_dtype(case)).to(torch.complex128)
        if kind == "expval":
            return {"energy": _exact_words(case, seed, psi)}
        if kind == "readout":
            p = psi.real ** 2 + psi.imag ** 2
            p, wires = p.reshape(1, -1), _marginal_wires(case, seed)
            # sum out the wires between the kept ones, the last first
            lo = n
            for w in reversed(wires):
                if lo - w - 1:
                    p = p.reshape(1 << (w + 1), 1 << (lo - w - 1), -1).sum(1)
                p = p.reshape(1 << (w + 1), -1)
                lo = w
                p = p.reshape(1 << w, -1)
            return {"idx": None, "probs": p.reshape(1 << lo, -1).sum(0)}
        psi = psi.reshape(1, -1)
        for g, w, p in _ops(case, seed):
            psi = _apply(psi, n, _matrix(g, p), w)
        if case["mode"] == "fused":
            psi = psi / torch.linalg.vector_norm(psi)
        return psi.reshape(-1)
    ops, psi = _ops(case, seed), _zero_state(n)
    for g, w, p in ops:
        psi = _apply(psi, n, _matrix(g, p), w)
    if kind == "vjp":
        dy = torch.tensor(_cotangent(case, seed), device="cuda").reshape(1, -1)
        return {"vjp": -0.5j * _exact_sweep(n, ops, psi, dy)[:, 0]}
    bras = torch.cat([psi * _signs(n, w) for w in range(case["obs"])])
    return {"expvals": (psi.conj() * bras).sum(1).real,
            "jac": _exact_sweep(n, ops, psi, bras).imag.transpose(0, 1).contiguous()}
