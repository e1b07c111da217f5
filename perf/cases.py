"""Performance cases of the engine, through the entry points its users call.

A case is a dict of plain values; its ``kind`` names what a user's program does:

  gates      gate tensors contracted into a register tensor one pair at a time
             (contract_pair, the drop-in of ContractIndices), the result read back
  product    two large tensors with shuffled axes contracted, and the result contracted
             with a third one down to a small open tensor
  inner      two large tensors contracted over nearly all of their axes
  energy     one QAOA energy on the drop-in path: text to value, one step per launch
  vector     the probabilities of every output string of a circuit, as one batch
  qaoa       energies of many angle sets of one graph: new angles from device memory,
             one launch, energies back
  amplitude  one amplitude of a random grid circuit (sliced, or in the sweep order)
  lightcone  one edge's expectation value of a 4-regular graph at depth 2

Sizes are those of the repository's benchmark and tests, or their neighbours.
"""
from __future__ import annotations

import functools
import math
import random

import numpy as np
import torch

import qtorch_amd as qa
from qtorch_amd import workloads as wl

FORMS = {"c128": qa.QT_PLAIN_C128, "4m": qa.QT_C64_4M, "3m": qa.QT_C64_3M, "bf16x3": qa.QT_C64_BF16X3,
         "4m_rescaled": qa.QT_C64_4M | qa.QT_RESCALE}


def listed():
    return [
        # the smallest calls: a gate superoperator at a time on a five-wire density
        # tensor, as every recorded order begins; launches and latency are all there is
        {"name": "gates_5wires_c128", "kind": "gates", "form": "c128", "dim_log2": 2, "rank": 5, "gates": 12},
        # a whole call of the reference's user: one energy, complex128, edge by edge
        {"name": "energy_3reg_n12_p1", "kind": "energy", "n": 12, "p": 1},
        # every output probability of an 8-qubit circuit, 256 measured networks at once
        {"name": "vector_qft8_c128", "kind": "vector", "form": "c128", "qubits": 8},
        # large products of tensors as they come out of earlier steps (axes in any
        # order), in the three arithmetics that are chosen in earnest
        {"name": "product_c128", "kind": "product", "form": "c128", "dim_log2": 1, "m": 11, "n": 11, "k": 12,
         "keep": 8, "open": 6},
        {"name": "product_4m", "kind": "product", "form": "4m", "dim_log2": 2, "m": 12, "n": 12, "k": 12,
         "keep": 8, "open": 6},
        {"name": "product_bf16x3", "kind": "product", "form": "bf16x3", "dim_log2": 1, "m": 10, "n": 13, "k": 11,
         "keep": 7, "open": 7},
        # the last steps of a large network: two large tensors, a few open indices
        {"name": "inner_4m", "kind": "inner", "form": "4m", "sum": 22, "free_a": 3, "free_b": 2},
        # whole amplitudes of the precision-stress circuits
        {"name": "amplitude_4x6_d14_c128", "kind": "amplitude", "form": "c128", "rows": 4, "cols": 6, "depth": 14,
         "order": "linegraph", "max_bits": 22},
        {"name": "amplitude_6x8_d14_4m", "kind": "amplitude", "form": "4m", "rows": 6, "cols": 8, "depth": 14,
         "order": "sweep", "max_bits": 29},
        # one large light cone of the uneven workload
        {"name": "lightcone_n20_4m", "kind": "lightcone", "form": "4m", "n": 20, "graph": 7020, "edge": 1},
        # an optimiser's step over many angle sets: generated code, energies only
        {"name": "qaoa_p1_131072_c128", "kind": "qaoa", "form": "c128", "n": 30, "p": 1, "sets": 131072,
         "compiled": True},
        # depth 2 does not fit generated code: the table executor
        {"name": "qaoa_p2_64_4m", "kind": "qaoa", "form": "4m", "n": 20, "p": 2, "sets": 64, "compiled": False},
    ]


def draw(rng):
    def log2_between(lo, hi):
        return int(round(2 ** rng.uniform(math.log2(lo), math.log2(hi))))

    kind = rng.choice(["gates", "gates", "product", "product", "product", "inner", "energy", "vector", "qaoa", "qaoa",
                       "amplitude", "amplitude", "lightcone", "lightcone"])
    if kind == "gates":
        dl = rng.choice([1, 2])
        return {"kind": kind, "form": rng.choice(["c128", "4m", "3m", "bf16x3"]), "dim_log2": dl,
                "rank": rng.randint(3, 12) if dl == 2 else rng.randint(5, 24), "gates": log2_between(3, 24)}
    if kind == "product":
        dl = rng.choice([1, 2])
        m, n = rng.randint(6, 12), rng.randint(6, 12)
        k = rng.randint(4, 23 - max(m, n))
        m, n, k = (x // dl * dl for x in (m, n, min(k, 13)))
        keep = rng.randint(2, min(m, 8)) // dl * dl
        return {"kind": kind, "form": rng.choice(["c128", "4m", "3m", "bf16x3", "4m_rescaled"]), "dim_log2": dl, "m": m,
                "n": n, "k": k, "keep": keep, "open": rng.randint(0, 7) // dl * dl}
    if kind == "inner":
        return {"kind": kind, "form": rng.choice(["c128", "4m", "3m"]), "sum": rng.randint(13, 22),
                "free_a": rng.randint(0, 3), "free_b": rng.randint(0, 3)}
    if kind == "energy":
        return {"kind": kind, "n": 2 * rng.randint(4, 12), "p": 1, "graph": rng.randint(1, 999)}
    if kind == "vector":
        return {"kind": kind, "form": rng.choice(["c128", "4m", "3m"]), "qubits": rng.randint(3, 8),
                "turns": rng.choice(["RX", "RY", "RX RZ", "RY RZ", "RX RY RZ"])}
    if kind == "qaoa":
        if rng.random() < 0.5:
            return {"kind": kind, "form": rng.choice(["c128", "4m"]), "n": 2 * rng.randint(5, 15), "p": 1,
                    "sets": log2_between(65, 131072), "compiled": True}
        return {"kind": kind, "form": rng.choice(["c128", "4m", "3m"]), "n": 2 * rng.randint(7, 12), "p": 2,
                "sets": log2_between(1, 64), "compiled": False}
    if kind == "amplitude":
        form = rng.choice(["c128", "4m", "3m", "bf16x3", "4m_rescaled"])
        r, c, d, order, bits = rng.choice([(4, 5, 8, "linegraph", 22), (6, 8, 8, "linegraph", 22),
                                           (4, 6, 14, "linegraph", 22), (4, 6, 14, "linegraph", 24),
                                           (4, 6, 14, "sweep", 28), (5, 6, 14, "sweep", 28), (3, 7, 11, "linegraph", 20),
                                           (5, 5, 14, "sweep", 28), (5, 6, 8, "linegraph", 19)])
        return {"kind": kind, "form": form, "rows": r, "cols": c, "depth": d, "order": order, "max_bits": bits,
                "circuit": rng.randint(600, 609)}
    while True:  # a light cone of a bounded plan
        case = {"kind": "lightcone", "form": rng.choice(["c128", "4m", "3m"]), "n": 2 * rng.randint(10, 40),
                "graph": rng.randint(7000, 7999), "edge": rng.randint(0, 39)}
        if work(case)["flops"] <= 8 * 2 ** 33:
            return case


# ---- inputs ------------------------------------------------------------------------


@functools.lru_cache(maxsize=1)
def _ctx():
    return qa.Context(0)


def _is_c128(case):
    return case["form"] == "c128"


def _values(n, k, case, seed, scale):
    """n complex normal values of standard deviation `scale`: the k-th tensor of a case."""
    g = torch.Generator(device="cuda").manual_seed(1000 * seed + k)
    real = torch.float64 if _is_c128(case) else torch.float32
    x = torch.randn(2 * n, dtype=real, device="cuda", generator=g) * (scale / math.sqrt(2.0))
    return torch.view_as_complex(x.view(-1, 2))


def _tensor(case, rank, dl, values):
    t = qa.Tensor(_ctx(), rank, dl, qa.QT_DTYPE_C128 if _is_c128(case) else qa.QT_DTYPE_C64)
    return t.upload(values.cpu().numpy())


def _gate_steps(case):
    """(axes of the register, pairs, free) of every gate: two neighbouring or distant
    wires, the register's other wires kept in order and the gate's outputs behind them."""
    rng = random.Random(case["rank"] * 100 + case["gates"])
    steps = []
    for _ in range(case["gates"]):
        ax = rng.sample(range(case["rank"]), 2)
        pairs = [(ax[0], 0), (ax[1], 1)]
        free = [(True, i) for i in range(case["rank"]) if i not in ax] + [(False, 2), (False, 3)]
        steps.append((pairs, free))
    return steps


OPEN_BITS = 12  # a register larger than this is projected before it is read back


def _gate_inputs(case, seed):
    dl, r = case["dim_log2"], case["rank"]
    reg = _values(1 << (dl * r), 0, case, seed, 1.0)
    gates = [_values(1 << (4 * dl), 1 + i, case, seed, 0.5 ** dl) for i in range(case["gates"])]
    bra_rank = max(0, r - OPEN_BITS // dl)
    bra = _values(1 << (dl * bra_rank), 1 + len(gates), case, seed, 2.0 ** (-dl * bra_rank / 2)) if bra_rank else None
    return reg, gates, bra_rank, bra


def _product_steps(case):
    """The two steps' axes, in units of one wire: A(m + k wires), B(k + n), D(n + m - keep + open),
    each with its wires shuffled."""
    dl = case["dim_log2"]
    m, n, k, keep, op = (case[x] // dl for x in ("m", "n", "k", "keep", "open"))
    rng = random.Random(m * 10000 + n * 100 + k)
    pa, pb, pd = list(range(m + k)), list(range(n + k)), list(range(n + m - keep + op))
    for p in (pa, pb, pd):
        rng.shuffle(p)
    pairs1 = [(pa[m + i], pb[n + i]) for i in range(k)]
    free1 = [(True, pa[i]) for i in range(m)] + [(False, pb[i]) for i in range(n)]
    pairs2 = [(keep + i, pd[i]) for i in range(m - keep + n)]
    free2 = [(True, i) for i in range(keep)] + [(False, pd[m - keep + n + i]) for i in range(op)]
    return (m + k, n + k, n + m - keep + op), (pairs1, free1), (pairs2, free2)


def _product_inputs(case, seed):
    dl = case["dim_log2"]
    ranks = _product_steps(case)[0]
    scales = (1.0, 2.0 ** (-case["k"] / 2), 2.0 ** (-(case["m"] - case["keep"] + case["n"]) / 2))
    return [_values(1 << (dl * r), i, case, seed, s) for i, (r, s) in enumerate(zip(ranks, scales))]


def _inner_step(case):
    s, fa, fb = case["sum"], case["free_a"], case["free_b"]
    rng = random.Random(s * 100 + fa * 10 + fb)
    pa, pb = list(range(s + fa)), list(range(s + fb))
    rng.shuffle(pa)
    rng.shuffle(pb)
    pairs = [(pa[fa + i], pb[fb + i]) for i in range(s)]
    return pairs, [(True, pa[i]) for i in range(fa)] + [(False, pb[i]) for i in range(fb)]


def _inner_inputs(case, seed):
    s = case["sum"]
    return [_values(1 << (s + case["free_a"]), 0, case, seed, 1.0),
            _values(1 << (s + case["free_b"]), 1, case, seed, 2.0 ** (-s / 2))]


def _graph(case):
    return wl.regular_graph(case["n"], 4 if case["kind"] == "lightcone" else 3, case.get("graph", 2024))


def _angles(case, seed, sets):
    """sets x 2p angles [betas..., gammas...] in the ranges an optimiser searches."""
    g = np.random.default_rng(seed)
    p = case.get("p", 2)
    return np.concatenate([g.uniform(0, math.pi / 2, (sets, p)), g.uniform(-math.pi, math.pi, (sets, p))], axis=1)


def _vector_circuit(case, seed):
    rng = random.Random(seed)
    n = case["qubits"]
    lines = wl.qft_qasm(n).strip().split("\n")
    axes = case.get("turns", "RX").split()
    turns = [f"{axis} {rng.uniform(0, 2 * math.pi):.9g} {i}" for axis in axes for i in range(n)]
    return "\n".join(lines[:1] + turns + lines[1:]) + "\n"


def _grid(case, seed):
    n = case["rows"] * case["cols"]
    circuit = wl.grid_random_circuit(case["rows"], case["cols"], case["depth"], seed=case.get("circuit", 2024))
    return circuit, wl.bitstring(n, seed)


def _sliced(case, seed):
    if case["kind"] == "amplitude":
        q, bits = _grid(case, seed)
        sweep = case["order"] == "sweep"
        return qa.SlicedNetwork(q, bits, dim_log2=1, order=qa.ORDER_SWEEP if sweep else qa.ORDER_LINEGRAPH,
                                seed=0 if sweep else 2, max_bits=case["max_bits"])
    q, m = qa.qaoa_edge_text(wl.dgf_text(_graph(case)), 2, False, case["edge"], list(_angles(case, seed, 1)[0]))
    return qa.SlicedNetwork(q, m, dim_log2=2, order=qa.ORDER_LINEGRAPH, max_bits=28)


def prepare(case, seed):
    kind = case["kind"]
    ctx = _ctx()
    if kind == "gates":
        reg, gates, bra_rank, bra = _gate_inputs(case, seed)
        dl, r = case["dim_log2"], case["rank"]
        return {"case": case, "reg": _tensor(case, r, dl, reg), "gates": [_tensor(case, 4, dl, g) for g in gates],
                "bra": _tensor(case, bra_rank, dl, bra) if bra_rank else None, "steps": _gate_steps(case)}
    if kind in ("product", "inner"):
        dl = case.get("dim_log2", 1)
        values = _product_inputs(case, seed) if kind == "product" else _inner_inputs(case, seed)
        steps = _product_steps(case)[1:] if kind == "product" else [_inner_step(case)]
        ranks = [(v.numel().bit_length() - 1) // dl for v in values]
        return {"case": case, "steps": steps, "tensors": [_tensor(case, r, dl, v) for r, v in zip(ranks, values)]}
    if kind == "energy":
        return {"case": case, "graph": wl.dgf_text(_graph(case)), "angles": list(_angles(case, seed, 1)[0])}
    if kind == "vector":
        n = case["qubits"]
        q = _vector_circuit(case, seed)
        strings = [wl.measure_text(format(i, f"0{n}b")[::-1]) for i in range(1 << n)]
        return {"case": case, "batch": qa.NetBatch(ctx, [q] * len(strings), strings, precision=FORMS[case["form"]])}
    if kind == "qaoa":
        b = qa.QaoaBatch(ctx, wl.dgf_text(_graph(case)), case["p"], ref_map=False, precision=FORMS[case["form"]])
        b.set_angles(_angles(case, 7, case["sets"]))  # where a search starts
        if case["compiled"]:
            b.compile(hermitian=True)
            b.sums_only(True)
        angles = torch.from_numpy(_angles(case, seed, case["sets"])).cuda()
        torch.cuda.synchronize()
        return {"case": case, "batch": b, "angles": angles}
    return {"case": case, "network": _sliced(case, seed)}


def run(state):
    case = state["case"]
    kind = case["kind"]
    ctx = _ctx()
    if kind in ("gates", "product", "inner"):
        form = FORMS[case["form"]]
        if kind == "gates":
            t = state["reg"]
            for g, (pairs, free) in zip(state["gates"], state["steps"]):
                t, _ = qa.contract_pair(ctx, t, g, pairs, free, form)
            if state["bra"] is not None:
                w, r = state["bra"].rank, case["rank"]
                t, _ = qa.contract_pair(ctx, t, state["bra"], [(i, i) for i in range(w)],
                                        [(True, i) for i in range(w, r)], form)
            return t.download()
        t = state["tensors"][0]
        for x, (pairs, free) in zip(state["tensors"][1:], state["steps"]):
            t, _ = qa.contract_pair(ctx, t, x, pairs, free, form)
        out = t.download()
        return np.ldexp(1.0, t.exponent()) * out if case["form"] == "4m_rescaled" else out
    if kind == "energy":
        return qa.qaoa_energy_plain(ctx, state["graph"], case["p"], False, state["angles"], seed=1)
    if kind == "vector":
        state["batch"].launch()
        return state["batch"].results()
    if kind == "qaoa":
        b = state["batch"]
        b.update_angles(device_ptr=state["angles"].data_ptr(), n_sets=case["sets"])
        b.launch()
        energies, zz = b.results()
        return energies if zz is None else (energies, zz)
    value, _ = state["network"].run(ctx, FORMS[case["form"]])
    return np.array([value])


def work(case):
    kind = case["kind"]
    elem = 16 if case.get("form") == "c128" else 8
    if kind == "gates":  # each gate reads and writes the register
        dl, r, g = case["dim_log2"], case["rank"], case["gates"]
        n = 1 << (dl * r)
        return {"bytes": elem * (2 * g * n + g * (1 << 4 * dl)), "flops": 8 * g * n * (1 << (2 * dl))}
    if kind == "product":
        m, n, k, keep, op = (case[x] for x in ("m", "n", "k", "keep", "open"))
        elems = 2 ** (m + k) + 2 ** (n + k) + 2 * 2 ** (m + n) + 2 ** (n + m - keep + op) + 2 ** (keep + op)
        return {"bytes": elem * elems, "flops": 8 * (2 ** (m + n + k) + 2 ** (m + n + op))}
    if kind == "inner":
        s, fa, fb = case["sum"], case["free_a"], case["free_b"]
        return {"bytes": elem * (2 ** (s + fa) + 2 ** (s + fb)), "flops": 8 * 2 ** (s + fa + fb)}
    if kind in ("energy", "qaoa"):
        # complex multiply-adds of the light cones' plans; generated code for depth 1 needs
        # 224 real multiply-adds of a light cone's (zeros, ones and mirror images left out)
        edges, sets = 3 * case["n"] // 2, case.get("sets", 1)
        if case.get("compiled"):
            return {"bytes": 8 * sets * (2 * case["p"] + 1), "flops": 2 * 224 * edges * sets}
        dgf = wl.dgf_text(_graph(case))
        macs = 0
        for e in range(edges):
            net = qa.Network(*qa.qaoa_edge_text(dgf, case["p"], False, e, list(_angles(case, 1, 1)[0])))
            net.order(qa.ORDER_GREEDY)
            macs += net.program_stats()["cmacs"]
            net.close()
        return {"bytes": 8 * sets * (2 * case["p"] + 1 + 2 * edges), "flops": 8 * macs * sets}
    if kind == "vector":
        n = case["qubits"]
        net = qa.Network(_vector_circuit(case, 1), wl.measure_text("0" * n))
        net.order(qa.ORDER_GREEDY)
        macs = net.program_stats()["cmacs"]
        net.close()
        return {"bytes": 16 << n, "flops": 8 * macs * 2 ** n}
    net = _sliced(case, 1)
    plan = net.plan()
    net.close()
    return {"bytes": 16, "flops": 8 * plan["cmacs_per_slice"] * plan["slices"]}


# ---- the same values in 64 bits, with plain torch ------------------------------------


def _gathered(x, dl, axes):
    """The flat values of x (axis 0 fastest) with its axes in the order given."""
    at = torch.arange(x.numel(), device=x.device)
    src = torch.zeros_like(at)
    for i, ax in enumerate(axes):
        src += ((at >> (dl * i)) & ((1 << dl) - 1)) << (dl * ax)
    return x[src]


def _pair64(a, b, dl, pairs, free):
    """The contraction of two flat tensors; A's free axes come before B's."""
    m = [ax for from_a, ax in free if from_a]
    n = [ax for from_a, ax in free if not from_a]
    assert free == [(True, ax) for ax in m] + [(False, ax) for ax in n]
    left = _gathered(a, dl, m + [x for x, _ in pairs]).view(-1, 1 << (dl * len(m)))
    right = _gathered(b, dl, [y for _, y in pairs] + n).view(1 << (dl * len(n)), -1)
    return (right @ left).reshape(-1)


def _text_float(x):
    """An angle printed with 6 digits and read as a float, as circuits are written."""
    return float(np.float32(float("%.6g" % x)))


def _one(psi, u, ax):
    """The 2 x 2 matrix u on axis ax of psi."""
    return torch.movedim(torch.tensordot(u, psi, dims=([1], [ax])), 0, ax)


def _matrix(name, t):
    c, s = math.cos(t / 2), math.sin(t / 2)
    m = {"RX": [[c, -1j * s], [-1j * s, c]], "RY": [[c, -s], [s, c]],
         "RZ": [[complex(c, -s), 0], [0, complex(c, s)]], "H": [[0.5 ** 0.5, 0.5 ** 0.5], [0.5 ** 0.5, -(0.5 ** 0.5)]]}
    return torch.tensor(m[name], dtype=torch.complex128, device="cuda")


def _state_vector(qasm):
    """|psi> with qubit q on axis q."""
    lines = qasm.strip().split("\n")
    n = int(lines[0])
    psi = torch.zeros([2] * n, dtype=torch.complex128, device="cuda")
    psi[(0,) * n] = 1.0
    for line in lines[1:]:
        t = line.split()
        if t[0] in ("CZ", "CPHASE"):
            phase = -1.0 if t[0] == "CZ" else complex(math.cos(float(t[1])), math.sin(float(t[1])))
            at = [slice(None)] * n
            at[int(t[-2])] = at[int(t[-1])] = 1
            psi[tuple(at)] *= phase
        elif t[0] == "SWAP":
            psi = psi.transpose(int(t[1]), int(t[2])).contiguous()
        else:
            angle = float(np.float32(t[1])) if len(t) == 3 else 0.0
            psi = _one(psi, _matrix(t[0], angle), int(t[-1])).contiguous()
    return psi


def _zz(edges, u, v, p, angles):
    """<Z_u Z_v> for every row of angles, on the vertices within p edges of u and v."""
    ball = [u, v]
    for _ in range(p):
        ball += sorted({b for a, b in edges + [(y, x) for x, y in edges] if a in ball and b not in ball})
    at = {x: i for i, x in enumerate(ball)}
    n, sets = len(ball), angles.shape[0]
    bits = torch.arange(1 << n, device="cuda")
    z = [1.0 - 2.0 * ((bits >> i) & 1).double() for i in range(n)]
    cost = sum(z[at[a]] * z[at[b]] for a, b in edges if a in at and b in at)
    psi = torch.full((sets, 1 << n), 2.0 ** (-n / 2), dtype=torch.complex128, device="cuda")
    for layer in range(p):
        turn = torch.tensor([_text_float(-x) for x in angles[:, p + layer]], device="cuda", dtype=torch.float64)
        mix = torch.tensor([_text_float(2 * x) for x in angles[:, layer]], device="cuda", dtype=torch.float64) / 2
        psi = psi * torch.exp(-0.5j * turn[:, None] * cost[None])
        c, s = torch.cos(mix)[:, None, None, None], -1j * torch.sin(mix)[:, None, None, None]
        for i in range(n):
            x = psi.view(sets, -1, 2, 1 << i)
            psi = (c * x + s * x.flip(2)).view(sets, -1)
    return (psi.abs() ** 2 * (z[0] * z[1])[None]).sum(1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "gates":
        dl = case["dim_log2"]
        reg, gates, bra_rank, bra = _gate_inputs(case, seed)
        t = reg.to(torch.complex128)
        for g, (pairs, free) in zip(gates, _gate_steps(case)):
            t = _pair64(t, g.to(torch.complex128), dl, pairs, free)
        if bra_rank:
            t = _pair64(t, bra.to(torch.complex128), dl, [(i, i) for i in range(bra_rank)],
                        [(True, i) for i in range(bra_rank, case["rank"])])
        return t.cpu().numpy()
    if kind in ("product", "inner"):
        dl = case.get("dim_log2", 1)
        values = _product_inputs(case, seed) if kind == "product" else _inner_inputs(case, seed)
        steps = _product_steps(case)[1:] if kind == "product" else [_inner_step(case)]
        t = values[0].to(torch.complex128)
        for x, (pairs, free) in zip(values[1:], steps):
            t = _pair64(t, x.to(torch.complex128), dl, pairs, free)
        return t.cpu().numpy()
    if kind in ("energy", "qaoa"):
        edges, p = _graph(case), case["p"]
        angles = _angles(case, seed, case.get("sets", 1))
        energy, zz = 0.0, []
        for u, v in edges:
            x = torch.cat([_zz(edges, u, v, p, part) for part in np.array_split(angles, -(-len(angles) // 16384))])
            energy = energy + 0.5 * (1.0 - x)
            zz.append(x)
        energy, zz = energy.cpu().numpy(), torch.stack(zz, 1).cpu().numpy()
        if kind == "energy":
            return float(energy[0]), zz[0]
        return energy if case["compiled"] else (energy, zz)
    if kind == "vector":
        psi = _state_vector(_vector_circuit(case, seed))
        n = case["qubits"]
        return (psi.permute(list(reversed(range(n)))).reshape(-1).abs() ** 2).to(torch.complex128).cpu().numpy()
    if kind == "amplitude":
        if case["rows"] * case["cols"] > 25:
            return None  # beyond a state vector
        q, bits = _grid(case, seed)
        return _state_vector(q)[tuple(int(b) for b in bits)].reshape(1).cpu().numpy()
    edges = _graph(case)
    u, v = edges[case["edge"]]
    try:
        return _zz(edges, u, v, 2, _angles(case, seed, 1)).to(torch.complex128).cpu().numpy()
    except torch.cuda.OutOfMemoryError:
        return None  # light cones of up to 26 vertices fit
