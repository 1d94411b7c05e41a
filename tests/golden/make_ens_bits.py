"""Digests of the batched mixed-precision form's results on an MI355X, one per
case and quantity: its numbers have no reference outside this library, so the
bits themselves are kept (ens_bits.json), and a change of a kernel that is not
meant to change results is compared with them.  Recorded with the tracer
transport as separate kernels (edgvar3, trcadv1, trcadv2, trcadv3) and the
global sums as one thread per column.

    python tests/golden/make_ens_bits.py       records them again (on the GPU)
"""
import hashlib
import json
import os

import numpy as np

FILE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "ens_bits.json")
NOISE, PERTURB, LOGNORMAL = 1, 2, 4
FIELDS = ("us", "vs", "dp", "pr", "ex", "ph", "mp", "ws", "sdot", "tr", "trdp", "psrf")
# name: level, nvl, ntra, members, mode, flux scheme, class-B tracers, land, fused transport, synth flags, steps
CASES = {
    "G2 x 64 full": (2, 64, 2, 3, 0, 1, 0, False, False, NOISE | PERTURB, 9),
    "G3 x 38 mass_adv class B": (3, 38, 3, 2, 0, 2, 2, False, False, NOISE | PERTURB, 14),
    "G3 x 64 transport land": (3, 64, 4, 2, 1, 1, 0, True, False, NOISE | LOGNORMAL, 8),
    "G3 x 33 transport land fused": (3, 33, 5, 2, 1, 1, 0, True, True, NOISE, 6),
    "G4 x 64 full land": (4, 64, 4, 2, 0, 1, 0, True, False, NOISE | PERTURB, 24),
    "G4 x 50 mass_adv transport": (4, 50, 7, 1, 1, 2, 0, False, False, NOISE | LOGNORMAL, 8),
}


def digests(case):
    """{quantity: digest of its bytes, every member's in turn} of a case's run."""
    from fimocn_subx_realtime_hera_apr2020_amd import fimhip, state
    level, nvl, ntra, members, mode, scheme, ntrb, land, fused, flags, steps = CASES[case]
    g = fimhip.icos_grid(level)
    th, ds = state.vertical_tables(nvl)
    own = 5760.0 / 2 ** (level - 1)
    e = fimhip.Ensemble(g, members, nvl, ntra, min(480.0, own) if mode else min(240.0, own * 2.0 / 3.0), th, ds)
    try:
        e.set_flux_scheme(scheme)
        if ntrb:
            e.set_class_b(ntrb, 3)
        if fused:
            e.set_fused(True)
        for m in range(members):
            e.synth(m, seed=11, flags=flags)
            if land:
                e.set_wet(m, np.sin(3 * np.asarray(g.lon) + m) + np.cos(2 * np.asarray(g.lat)) > -0.5)
            if ntrb:
                e.load_class_b(m, np.random.default_rng(m).uniform(0.5, 1.5, (ntrb, g.nip, nvl)))
        e.init_state(not mode)
        e.step(steps, mode)
        out = dict(zip(("mass", "totals", "mass32", "totals32"), ([a] for a in e.globsum())))
        for f in FIELDS + (("trb",) if ntrb else ()):
            out[f] = [e.download(m, f) for m in range(members)]
    finally:
        e.close()
    return {f: hashlib.sha256(b"".join(np.ascontiguousarray(a, np.float64).tobytes() for a in v)).hexdigest()[:16]
            for f, v in out.items()}


if __name__ == "__main__":
    with open(FILE, "w") as f:
        json.dump({c: digests(c) for c in CASES}, f, indent=1)
        f.write("\n")
