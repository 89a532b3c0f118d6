"""The tridiagonal reduction and the back-transformation at the edges of their tiles.

Stacks of H2 molecules (one AO per atom, a helium atom for odd counts) give
systems of every AO count: around the 16-column phases and 32-row tiles of the
register reduction, the 192-column switch between its two forms, the
16-reflector blocks and 16-row tiles of the back-transformation, and the
256-AO limit of the register kernels.  Energies, forces and charges against the
oracle at the package's bars.
"""
import numpy as np
import pytest

from oracle import oracle as O
from xtbloom_amd import interface, library, workloads

pytestmark = pytest.mark.gpu

E_TOL, F_TOL, Q_TOL = 1e-7, 1e-6, 1e-6


def stack(n, rng):
    """n atoms with one AO each: H2 molecules on a grid, one He when n is odd."""
    z, xyz = [], []
    for m in range(n // 2):
        c = 5.0 * np.array([m % 5, (m // 5) % 5, m // 25]) + rng.normal(0.0, 0.1, 3)
        u = rng.normal(size=3)
        u *= 0.5 * (1.40 + rng.uniform(-0.05, 0.05)) / np.linalg.norm(u)
        z += [1, 1]
        xyz += [c - u, c + u]
    if n % 2:
        z.append(2)
        xyz.append(np.array([-5.0, -5.0, 0.0]))
    return dict(Z=np.array(z, np.int32), xyz=np.array(xyz), charge=0.0, uhf=0)


@pytest.mark.parametrize("sizes", [
    [1, 2, 3, 4, 5, 6],                       # no, one or a few reflectors
    [14, 15, 16, 17, 18, 19, 31, 32, 33, 34],  # first phases and row tiles, one or two WY blocks
    [47, 48, 49, 63, 64, 65, 66, 95, 97],
    [127, 128, 129, 130, 175, 176, 177],
    [190, 191, 192, 193, 194, 195],           # the switch between the two forms
    [208, 223, 225, 240, 254, 255, 256],
    [257, 258, 259, 272, 288, 289],           # teams of nine and ten workgroups
    [353, 448, 449, 513],                     # row tiles per wavefront of the back-transformation
], ids=lambda s: f"{s[0]}-{s[-1]}")
def test_sizes_against_the_oracle(sizes):
    check(sizes)


def test_teams_that_leave_at_the_gate(monkeypatch):
    """A closed gate: every team leaves before it writes anything and one workgroup
    per system reduces the matrices instead."""
    monkeypatch.setenv("XTBLOOM_AMD_TEAMS", "0")
    check([258, 289, 353])


def check(sizes):
    rng = np.random.default_rng(sizes[0])
    b = workloads.from_systems([stack(n, rng) for n in sizes])
    ctx = interface.Context("hip", 0)
    try:
        print("case reduction sizes", sizes, flush=True)
        out = interface.compute_arrays(ctx, b.atom_offsets, b.atomic_numbers, b.positions,
                                       b.molecular_charges, b.unpaired_electrons)
    finally:
        ctx.close()
    ref = O.batch(b.atom_offsets, b.atomic_numbers, b.positions, b.molecular_charges,
                  b.unpaired_electrons, threads=4)
    assert np.all(out.per_system_status == 0) and np.all(ref["status"] == 0)
    assert np.abs(out.scc_iterations - ref["iterations"]).max() <= 1
    assert np.abs(out.energies - ref["energies"]).max() <= E_TOL
    assert np.abs(out.forces + ref["gradient"]).max() <= F_TOL
    assert np.abs(out.charges - ref["charges"]).max() <= Q_TOL


def test_result_depends_on_the_system_alone(monkeypatch):
    """64 systems of 302 AOs take 640 team members, more than the chip holds at once:
    the bits of one lane are those of two lanes, and of systems computed alone."""
    rng = np.random.default_rng(64)
    systems = [workloads.alkane(50, rng) for _ in range(64)]
    b = workloads.from_systems(systems)
    ctx = interface.Context("hip", 0)

    def run(batch):
        return interface.compute_arrays(ctx, batch.atom_offsets, batch.atomic_numbers, batch.positions,
                                        batch.molecular_charges, batch.unpaired_electrons)

    try:
        print("case 64 systems of 302 AOs: one lane, two lanes, alone", flush=True)
        monkeypatch.setenv("XTBLOOM_AMD_LANES", "1")
        one = run(b)
        assert np.all(one.per_system_status == 0)
        monkeypatch.setenv("XTBLOOM_AMD_LANES", "2")
        two = run(b)
        monkeypatch.setenv("XTBLOOM_AMD_LANES", "1")
        for name in ("energies", "charges", "scc_iterations", "per_system_status"):
            assert np.array_equal(getattr(two, name), getattr(one, name)), name
        for i in (0, 40, 63):
            alone = run(workloads.from_systems([systems[i]]))
            a0, a1 = b.atom_offsets[i], b.atom_offsets[i + 1]
            assert alone.energies[0] == one.energies[i] and np.array_equal(alone.charges, one.charges[a0:a1])
            assert alone.scc_iterations[0] == one.scc_iterations[i]
    finally:
        ctx.close()
    ref = O.batch(b.atom_offsets[:3], b.atomic_numbers, b.positions, b.molecular_charges[:2],
                  b.unpaired_electrons[:2], threads=2)
    assert np.abs(one.energies[:2] - ref["energies"]).max() <= E_TOL
    a1 = b.atom_offsets[2]
    assert np.abs(one.forces[:a1] + ref["gradient"][:a1]).max() <= F_TOL


def test_closed_gate_changes_no_bit(monkeypatch):
    """The one workgroup that reduces a system whose team left at the gate forms every
    sum as the team does; that it ran shows in the time of the reduction (a team of 40
    workgroups against one)."""
    rng = np.random.default_rng(1280)
    b = workloads.from_systems([workloads.alkane(213, rng), workloads.alkane(50, rng), stack(257, rng)])
    ctx = interface.Context("hip", 0)

    def run():
        return interface.compute_arrays(ctx, b.atom_offsets, b.atomic_numbers, b.positions, b.molecular_charges,
                                        b.unpaired_electrons, determinism=library.DETERMINISM_REPRODUCIBLE,
                                        kernel_stats=["tridiag"])

    try:
        print("case gate: 1280, 302 and 257 AOs by teams", flush=True)
        team = run()
        monkeypatch.setenv("XTBLOOM_AMD_TEAMS", "0")
        print("case gate: the same, gates closed", flush=True)
        solo = run()
    finally:
        ctx.close()
    assert np.all(team.per_system_status == 0)
    for name in ("energies", "forces", "charges", "scc_iterations", "per_system_status"):
        assert np.array_equal(getattr(solo, name), getattr(team, name)), name
    ms = [o.extension["kernel_stats"]["tridiag"]["ms"] for o in (team, solo)]
    print("reduction: teams %.1f ms, one workgroup %.1f ms" % tuple(ms), flush=True)
    assert ms[1] > 3.0 * ms[0]
