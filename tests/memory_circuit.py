"""Surface-code memory circuits for the tests."""

from __future__ import annotations

import numpy as np


def memory_text(d, rounds, p, circuit=42):
    """Rotated distance-d memory in the Z basis: d*d data qubits, one ancilla
    per face, depolarizing and flip noise at p, one T per round on a random
    data qubit, detectors between rounds, Z on the first data row as the
    observable."""
    rng = np.random.default_rng(circuit)
    faces = []  # (type, {corner: data qubit})
    for r in range(-1, d):
        for c in range(-1, d):
            at = {k: (r + dr, c + dc) for k, (dr, dc) in dict(NW=(0, 0), NE=(0, 1), SW=(1, 0), SE=(1, 1)).items()}
            at = {k: i * d + j for k, (i, j) in at.items() if 0 <= i < d and 0 <= j < d}
            typ = "X" if (r + c) % 2 == 0 else "Z"
            inner = 0 <= r < d - 1 and 0 <= c < d - 1
            edge = len(at) == 2 and ((typ == "X" and r in (-1, d - 1)) or (typ == "Z" and c in (-1, d - 1)))
            if inner or edge:
                faces.append((typ, at))
    n, m = d * d, len(faces)
    anc = list(range(n, n + m))
    xs = [a for a, (typ, _) in zip(anc, faces) if typ == "X"]
    order = dict(X=["NW", "NE", "SW", "SE"], Z=["NW", "SW", "NE", "SE"])
    join = lambda qs: " ".join(map(str, qs))  # noqa: E731
    out = []
    for rnd in range(rounds):
        q = int(rng.integers(0, n))
        out += [f"T {q}", f"DEPOLARIZE1({p}) {q}", "H " + join(xs), f"DEPOLARIZE1({p}) " + join(xs)]
        for step in range(4):
            pairs = []
            for a, (typ, at) in zip(anc, faces):
                if order[typ][step] in at:
                    q = at[order[typ][step]]
                    pairs += [a, q] if typ == "X" else [q, a]
            out += ["CX " + join(pairs), f"DEPOLARIZE2({p}) " + join(pairs)]
        out += ["H " + join(xs), f"DEPOLARIZE1({p}) " + join(xs), f"X_ERROR({p}) " + join(anc), "MR " + join(anc)]
        for i, (typ, _) in enumerate(faces):
            if rnd:
                out.append(f"DETECTOR rec[-{m - i}] rec[-{2 * m - i}]")
            elif typ == "Z":
                out.append(f"DETECTOR rec[-{m - i}]")
    out += [f"X_ERROR({p}) " + join(range(n)), "M " + join(range(n))]
    for i, (typ, at) in enumerate(faces):
        if typ == "Z":
            out.append("DETECTOR " + " ".join(f"rec[-{n - q}]" for q in sorted(at.values())) + f" rec[-{n + m - i}]")
    out.append("OBSERVABLE_INCLUDE(0) " + " ".join(f"rec[-{n - q}]" for q in range(d)))
    return "\n".join(out)
