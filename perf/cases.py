"""Measured cases of the engine: what programs that use it have it do, through quantr_amd._capi.

Every case is one pass of a user's loop over a circuit whose structure is fixed (its `circuit`
seed, its sizes) and whose numbers are new: rotation angles, custom tables, registers and the
uniform draws come from the seed, as in a parameter sweep, a training loop or repeated
measurements. Results of complex64 states are handed on as 32-bit values, which is what such a
state holds.

Kinds of pass:
  qft      load a custom register, apply the quantum Fourier transform, measure, read the state
  evolve   |0...0>, apply the whole circuit, evaluate an observable, measure all qubits
  grad     expectation value and full adjoint gradient of a hardware-efficient ansatz
  batch    the same for many small circuits of uneven size in one launch, new angles each time
  observe  <psi|O|psi> of a state that is in hand
  shots    measure_all_without_cache: every shot's circuit simulated anew and measured
"""
import math

import numpy as np
import torch

from quantr_amd import _capi
from quantr_amd import workloads as W

PREC = {"c128": _capi.QR_C128, "c64": _capi.QR_C64}


def listed():
    return [
        # the reference's own test: a 10-qubit Fourier transform and 500 shots; pure latency
        {"name": "qft10_c128", "kind": "qft", "n": 10, "prec": "c128", "shots": 500},
        # Fourier transform of a large register, state read back by the program
        {"name": "qft17_c128", "kind": "qft", "n": 17, "prec": "c128", "shots": 1000},
        # an everyday small circuit simulated with 500 shots and its amplitudes looked at
        {"name": "evolve13_c128", "kind": "evolve", "family": "brickwork", "n": 13, "depth": 20, "prec": "c128",
         "custom": 0, "shots": 500, "circuit": 5},
        # a workstation-sized circuit with a user-defined 3-qubit gate and many shots
        {"name": "evolve25_c128_custom", "kind": "evolve", "family": "brickwork", "n": 25, "depth": 20,
         "prec": "c128", "custom": 3, "shots": 100000, "circuit": 3},
        # a variational ansatz in single precision at a size where the state leaves the caches
        {"name": "evolve28_c64", "kind": "evolve", "family": "hea", "n": 28, "depth": 6, "prec": "c64",
         "custom": 0, "shots": 0, "circuit": 0},
        # the headline circuit of bench.py: 30 qubits, depth 40, then an energy and 500 shots
        {"name": "evolve30_c128", "kind": "evolve", "family": "brickwork", "n": 30, "depth": 40, "prec": "c128",
         "custom": 0, "shots": 500, "circuit": 1234},
        # the gradient of bench.py: 20 qubits, 10 layers, 400 parameters
        {"name": "grad20_c128", "kind": "grad", "n": 20, "depth": 10, "prec": "c128"},
        # one training step of a small ansatz in single precision
        {"name": "grad13_c64", "kind": "grad", "n": 13, "depth": 6, "prec": "c64"},
        # serving: a mixed batch of ansatz gradients, as in bench.py's batch but up to 18 qubits
        {"name": "batch32_c64", "kind": "batch", "count": 32, "lo": 10, "hi": 18, "prec": "c64", "circuit": 512},
        # the energy of a large state under the Ising observable of bench.py
        {"name": "observe29_ising_c128", "kind": "observe", "n": 29, "prec": "c128", "terms": 0, "circuit": 0},
        # a mid-sized state under a Hamiltonian of many Pauli strings
        {"name": "observe22_strings_c128", "kind": "observe", "n": 22, "prec": "c128", "terms": 120, "circuit": 9},
        # bench.py's re-simulated shots: 12 qubits, a new custom table for every one of 500 shots
        {"name": "shots12_c128", "kind": "shots", "n": 12, "depth": 10, "prec": "c128", "shots": 500, "circuit": 5},
    ]


def draw(rng):
    kind = rng.choice(["qft", "evolve", "evolve", "evolve", "grad", "grad", "batch", "observe", "observe", "shots"])
    prec = rng.choice(["c128", "c128", "c64"])
    seed = rng.randrange(1, 100000)
    if kind == "qft":
        return {"kind": kind, "n": rng.randint(3, 19), "prec": "c128", "shots": int(10 ** rng.uniform(1.5, 4.5))}
    if kind == "evolve":
        family = rng.choice(["brickwork", "hea"])
        n = rng.randint(4, 29)
        if prec == "c64":
            family, n = ("hea", rng.randint(10, 30)) if family == "hea" else (family, rng.randint(4, 18))
        shots = 0 if prec == "c64" else int(10 ** rng.uniform(1.5, 5))
        custom = rng.choice([0, 0, 2, 3, 4]) if family == "brickwork" and n > 5 else 0
        return {"kind": kind, "family": family, "n": n, "depth": rng.randint(5, 40) if family == "brickwork" else
                rng.randint(2, 12), "prec": prec, "custom": custom, "shots": shots, "circuit": seed}
    if kind == "grad":
        return {"kind": kind, "n": rng.randint(5, 22), "depth": rng.randint(2, 12), "prec": prec}
    if kind == "batch":
        lo = rng.randint(6, 12)
        return {"kind": kind, "count": rng.randint(8, 64), "lo": lo, "hi": rng.randint(lo, 18), "prec": "c64",
                "circuit": seed}
    if kind == "observe":
        terms = rng.choice([0, int(2 ** rng.uniform(2, 8))])
        return {"kind": kind, "n": rng.randint(10, 24 if terms else 29), "prec": prec, "terms": terms, "circuit": seed}
    return {"kind": kind, "n": rng.randint(4, 14), "depth": rng.randint(4, 16), "prec": "c128",
            "shots": int(10 ** rng.uniform(1.7, 3)), "circuit": seed}


# ---- inputs ---------------------------------------------------------------------------------

def _angles(gates, seed):
    """The gate list with new angles U[0, 2 pi) in its rotations."""
    rng = W.SplitMix64(seed)
    return [(k, p, c, 2.0 * math.pi * rng.uniform() if k in ("Rx", "Ry", "Rz") else a, i) for k, p, c, a, i in gates]


def _unitary(k, seed):
    """A custom gate's table: images[j] is the image of local basis state j."""
    return np.ascontiguousarray(W.random_unitary(k, seed).T), np.ones(1 << k, dtype=np.uint8)


def _with_custom(gates, n, k, circuit, seed):
    """The gates with one k-qubit custom gate on seeded wires in the middle, and its table."""
    rng = W.SplitMix64(circuit + 1)
    wires = []
    while len(wires) < k:
        w = rng.below(n)
        if w not in wires:
            wires.append(w)
    cut = len(gates) // 2
    return gates[:cut] + [("Custom", wires[-1], tuple(wires[:-1]), 0.0, 0)] + gates[cut:], {cut: _unitary(k, seed)}


def _hea(n, depth, seed):
    """The ansatz near the identity, as variational circuits are initialised, so that its energy
    and gradients don't vanish with the size."""
    return W.hea(n, depth, seed=seed, angle_lo=-0.4, angle_hi=0.4)[0]


def _evolve_gates(case, seed):
    if case["family"] == "hea":
        return _hea(case["n"], case["depth"], seed), {}
    gates = _angles(W.brickwork(case["n"], depth=case["depth"], seed=case["circuit"]), seed)
    return _with_custom(gates, case["n"], case["custom"], case["circuit"], seed) if case["custom"] else (gates, {})


def _qft_gates(n):
    return [g for g in W.qft10(n, 0)[0] if g[0] != "X"]


def _register(n, seed):
    g = np.random.default_rng(seed)
    v = g.standard_normal(1 << n) + 1j * g.standard_normal(1 << n)
    return v / np.linalg.norm(v)


def _terms(case):
    """The Ising observable of the ansatz, or `terms` Pauli strings on one to four wires."""
    n = case["n"]
    if not case.get("terms"):
        return W.hea_observable(n)
    rng = W.SplitMix64(case["circuit"] + 77)
    out = []
    for _ in range(case["terms"]):
        k, wires = 1 + rng.below(4), []
        while len(wires) < k:
            w = rng.below(n)
            if w not in wires:
                wires.append(w)
        out.append((2.0 * rng.uniform() - 1.0, [(w, "XYZ"[rng.below(3)]) for w in wires]))
    return out


def _instances(case, seed):
    """(n, gates) of a batch: sizes from the circuit's seed, angles from the seed."""
    rng, new = W.SplitMix64(case["circuit"]), W.SplitMix64(seed)
    out = []
    for _ in range(case["count"]):
        n = case["lo"] + rng.below(case["hi"] - case["lo"] + 1)
        out.append((n, _hea(n, 2 + rng.below(7), new.next_u64())))
    return out


def _shot_programs(case, seed):
    """One program a shot: a brickwork whose 2-qubit custom gate has a table of its own."""
    n = case["n"]
    base = _angles(W.brickwork(n, depth=case["depth"], seed=case["circuit"]), seed)
    return [_with_custom(base, n, 2, case["circuit"], seed * 100003 + s) for s in range(case["shots"])]


def prepare(case, seed):
    kind, prec = case["kind"], PREC[case["prec"]]
    s = {"kind": kind, "prec": case["prec"]}
    if kind == "batch":
        items = [(n, W.to_program(g), _capi.Observable(W.hea_observable(n))) for n, g in _instances(case, seed)]
        s["batch"] = _capi.Batch(items, prec)
        s["programs"] = [p.c_struct() for _, p, _ in items]
        return s
    n = s["n"] = case["n"]
    if kind == "shots":
        s["programs"] = [W.to_program(g, c).c_struct() for g, c in _shot_programs(case, seed)]
        s["uniforms"] = np.array(W.uniforms(case["shots"], seed + 1))
        s["precision"] = prec
        return s
    if kind == "grad":
        s["program"] = W.to_program(_hea(n, case["depth"], seed)).c_struct()
        s["observable"] = _capi.Observable(W.hea_observable(n))
        s["grad"] = _capi.Grad(n, prec)
        return s
    s["state"] = _capi.State(n, prec)
    if kind == "observe":
        s["state"].apply(W.to_program(_hea(n, 2, seed)))
        s["state"].synchronize()
        s["observable"] = _capi.Observable(_terms(case))
        return s
    s["uniforms"] = np.array(W.uniforms(case["shots"], seed + 1))
    if kind == "qft":
        s["register"] = _register(n, seed)
        s["program"] = W.to_program(_qft_gates(n)).c_struct()
        return s
    gates, customs = _evolve_gates(case, seed)
    s["program"] = W.to_program(gates, customs).c_struct()
    s["observable"] = _capi.Observable(W.hea_observable(n))
    s["read"] = n <= 18
    return s


# ---- one pass -------------------------------------------------------------------------------

def _real(s, v):
    return np.float32(v) if s["prec"] == "c64" else v


def _reals(s, v):
    return v.astype(np.float32) if s["prec"] == "c64" else v


def _amplitudes(s):
    a = s["state"].amplitudes()
    return a.astype(np.complex64) if s["prec"] == "c64" else a


def run(s):
    kind = s["kind"]
    if kind == "batch":
        energies, grads, _ = s["batch"].run(s["programs"])
        return {"energies": _reals(s, energies), "grads": _reals(s, np.concatenate(grads))}
    if kind == "shots":
        return {"bins": _capi.sample_programs(s["n"], s["programs"], np.ones(len(s["programs"]), dtype=np.uint64),
                                              s["uniforms"], s["precision"]).view(np.int64)}
    if kind == "grad":
        energy = s["grad"].forward(s["program"], s["observable"])
        return {"energy": _real(s, energy), "grads": _reals(s, s["grad"].backward())}
    if kind == "observe":
        return {"energy": _real(s, s["state"].expectation(s["observable"]))}
    st = s["state"]
    if kind == "qft":
        st.set_amplitudes(s["register"])
        st.apply(s["program"])
        return {"bins": st.sample(s["uniforms"]).view(np.int64), "amplitudes": _amplitudes(s)}
    st.reset()
    st.apply(s["program"])
    out = {}
    if s["read"]:
        out["amplitudes"] = _amplitudes(s)
    else:
        out["energy"] = _real(s, st.expectation(s["observable"]))
    if len(s["uniforms"]):
        out["bins"] = st.sample(s["uniforms"]).view(np.int64)
    return out


# ---- what a pass cannot do without ----------------------------------------------------------

# real operations per amplitude of the state: a general 2x2 takes two complex products and a sum
# for each output, a real one half of that, a phase a product on half the amplitudes
FLOPS = {"H": 2, "Rx": 6, "Ry": 6, "Rz": 6, "S": 0, "T": 3, "CRk": 1.5, "Z": 0.5, "Y": 0, "X": 0, "CNot": 0,
         "Toffoli": 0, "Swap": 0}


def _flops(gates):
    return sum(FLOPS[g[0]] if g[0] != "Custom" else 8 << (len(g[2]) + 1) for g in gates)


def work(case):
    """The state is written once and read once; a gradient writes and reads two states and takes
    the gates three times (forward, and back on both)."""
    kind, width = case["kind"], 16 if case["prec"] == "c128" else 8
    if kind == "batch":
        items = _instances(case, 1)
        return {"bytes": sum(4 * width << n for n, _ in items), "flops": sum(_flops(g) * 3 * 2 ** n for n, g in items)}
    dim = 2 ** case["n"]
    if kind == "shots":
        gates = _with_custom(W.brickwork(case["n"], depth=case["depth"], seed=case["circuit"]), case["n"], 2,
                             case["circuit"], 1)[0]
        return {"bytes": 2 * width * dim * case["shots"], "flops": _flops(gates) * dim * case["shots"]}
    if kind == "grad":
        return {"bytes": 4 * width * dim, "flops": 3 * dim * _flops(_hea(case["n"], case["depth"], 1))}
    if kind == "observe":
        return {"bytes": width * dim, "flops": dim * (3 + 4 * len(_terms(case)))}
    if kind == "qft":
        return {"bytes": 2 * width * dim, "flops": dim * _flops(_qft_gates(case["n"]))}
    return {"bytes": 2 * width * dim, "flops": dim * _flops(_evolve_gates(case, 1)[0])}


# ---- the same in 64 bits with plain torch ---------------------------------------------------

S2 = math.sqrt(0.5)
PHASES = {"Z": -1.0, "S": 1j, "T": complex(S2, S2)}


def _parts(psi, n, wires):
    """psi seen with one axis of two for each of the wires: its slices by those wires' bits
    (wire 0 is the most significant index bit), as views."""
    order = sorted(wires)
    shape, at = [], 0
    for w in order:
        shape += [1 << (w - at), 2]
        at = w + 1
    v = psi.view(shape + [1 << (n - at)])

    def part(bits):
        index = []
        for w in order:
            index += [slice(None), bits[wires.index(w)]]
        return v[tuple(index)]

    return part


def _apply(psi, n, gate, table=None, invert=False):
    kind, target, controls, arg, arg_int = gate
    wires = list(controls) + [target]
    part = _parts(psi, n, wires)
    if kind == "Custom":
        k = len(wires)
        bits = [[(j >> (k - 1 - q)) & 1 for q in range(k)] for j in range(1 << k)]
        ins = [part(b).clone() for b in bits]
        for r, b in enumerate(bits):
            acc = ins[0] * complex(table[0][0][r])
            for j in range(1, 1 << k):
                acc += ins[j] * complex(table[0][j][r])
            part(b).copy_(acc)
        return
    if kind == "Swap":
        x, y = part([0, 1]), part([1, 0])
        keep = x.clone()
        x.copy_(y)
        y.copy_(keep)
        return
    ones = [1] * len(controls)
    x, y = part(ones + [0]), part(ones + [1])
    sign = -1.0 if invert else 1.0
    if kind in PHASES or kind in ("CRk", "Rz"):
        if kind == "Rz":
            x *= complex(math.cos(0.5 * arg), -sign * math.sin(0.5 * arg))
            y *= complex(math.cos(0.5 * arg), sign * math.sin(0.5 * arg))
        else:
            y *= PHASES[kind] if kind in PHASES else complex(math.cos(2 * math.pi / 2 ** arg_int),
                                                             math.sin(2 * math.pi / 2 ** arg_int))
        return
    keep = x.clone()
    if kind in ("X", "CNot", "Toffoli"):
        x.copy_(y)
        y.copy_(keep)
        return
    if kind == "H":
        m = (S2, S2, S2, -S2)
    elif kind == "Y":
        m = (0.0, -1j, 1j, 0.0)
    else:
        c, t = math.cos(0.5 * arg), sign * math.sin(0.5 * arg)
        m = (c, -t, t, c) if kind == "Ry" else (c, -1j * t, -1j * t, c)
    x.copy_(m[0] * x + m[1] * y)
    y.copy_(m[2] * keep + m[3] * y)


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _simulate(n, gates, customs=None, psi=None):
    if psi is None:
        psi = torch.zeros(1 << n, dtype=torch.complex128, device=_device())
        psi[0] = 1.0
    for i, g in enumerate(gates):
        _apply(psi, n, g, customs.get(i) if customs else None)
    return psi


def _pauli(psi, n, factors):
    out = psi.clone()
    for w, p in factors:
        _apply(out, n, (p, w, (), 0.0, 0))
    return out


def _energy(psi, n, terms):
    total = torch.zeros((), dtype=torch.float64, device=psi.device)
    for c, f in terms:
        total += c * torch.vdot(psi, _pauli(psi, n, f)).real
    return float(total)


def _gradient(n, gates, terms):
    """(energy, gradient) by undoing the gates on psi and O psi, one parameter after the other."""
    psi = _simulate(n, gates)
    lam = torch.zeros_like(psi)
    for c, f in terms:
        lam += c * _pauli(psi, n, f)
    energy = float(torch.vdot(psi, lam).real)
    grads = []
    for g in reversed(gates):
        if g[0] in ("Rx", "Ry", "Rz"):
            grads.append(torch.vdot(lam, _pauli(psi, n, [(g[1], g[0][1].upper())])).imag)
        for v in (psi, lam):
            _apply(v, n, g, invert=True)
    return energy, torch.stack(grads[::-1]).cpu()


def exact(case, seed):
    kind = case["kind"]
    if kind == "shots":
        return None
    if kind == "batch":
        got = [_gradient(n, g, W.hea_observable(n)) for n, g in _instances(case, seed)]
        return {"energies": np.array([e for e, _ in got]), "grads": torch.cat([g for _, g in got])}
    n = case["n"]
    if kind == "grad":
        energy, grads = _gradient(n, _hea(n, case["depth"], seed), W.hea_observable(n))
        return {"energy": energy, "grads": grads}
    if kind == "observe":
        terms = _terms(case)
        if len(terms) * 2 ** n > 4e10:
            return None
        return {"energy": _energy(_simulate(n, _hea(n, 2, seed)), n, terms)}
    if kind == "qft":
        psi = torch.from_numpy(_register(n, seed)).to(_device())
        return {"bins": None, "amplitudes": _simulate(n, _qft_gates(n), psi=psi).cpu()}
    gates, customs = _evolve_gates(case, seed)
    if len(gates) * 2 ** n > 3e11:
        return None
    psi = _simulate(n, gates, customs)
    out = {"amplitudes": psi.cpu()} if n <= 18 else {"energy": _energy(psi, n, W.hea_observable(n))}
    if case["shots"]:
        out["bins"] = None
    return out
