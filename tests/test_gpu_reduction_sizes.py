"""The tridiagonal reduction and the back-transformation at the edges of their tiles.

Stacks of H2 molecules (one AO per atom, a hydrogen atom for odd counts) give
systems of every AO count: around the 16-column phases and 32-row tiles of the
register reduction, the 192-column switch between its two forms, the
16-reflector blocks and 16-row tiles of the back-transformation, and the
256-AO limit of the register kernels.  Energies, forces and charges against the
oracle.  Molecules of 640 to 1280 AOs: the edges of the teams' classes and the
switches at 1024.
"""
import numpy as np
import pytest

from oracle import oracle as O
from xtbloom_amd import interface, library, workloads

pytestmark = pytest.mark.gpu

# Same iterations on both sides, so only rounding separates them: an eigenvector
# carries n eps |H| / gap <= 1280 * 2.2e-16 * 10 / 0.1 = 3e-11 of its neighbours, which
# enters the density to first order and the forces with derivatives of order 1; the
# SCC's amplification is below 10.  1e-9 is above that and two orders below an error
# of the package's bars.
E_TOL, F_TOL, Q_TOL = 1e-9, 1e-9, 1e-9


def stack(n, rng):
    """n hydrogen atoms, one AO each: H2 molecules on a grid and one atom when n is odd."""
    xyz = []
    for m in range(n // 2):
        c = 5.0 * np.array([m % 5, (m // 5) % 5, m // 25]) + rng.normal(0.0, 0.1, 3)
        u = rng.normal(size=3)
        u *= 0.5 * (1.40 + rng.uniform(-0.05, 0.05)) / np.linalg.norm(u)
        xyz += [c - u, c + u]
    if n % 2:
        xyz.append(np.array([-5.0, -5.0, 0.0]))
    return dict(Z=np.ones(n, np.int32), xyz=np.array(xyz), charge=0.0, uhf=n % 2)


def molecule(n, rng):
    """n >= 19 AOs, closed shell: the largest alkane (odd n: alkyl amine) that fits and
    H2 molecules 8 bohr and more beside it."""
    k = (n - 7) // 6 if n % 2 else (n - 2) // 6
    s = workloads.alkane(k, rng, substituent="NH2" if n % 2 else None)
    left = n - (6 * k + (7 if n % 2 else 2))
    if left == 0:
        return s
    rest = stack(left, rng)["xyz"]
    beside = rest + s["xyz"].min(axis=0) - rest.max(axis=0) - np.array([0.0, 8.0, 0.0])
    return dict(s, Z=np.concatenate([s["Z"], np.ones(left, np.int32)]).astype(np.int32),
                xyz=np.concatenate([s["xyz"], beside]))


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


def test_team_classes_against_the_oracle():
    """The first and last size of each class of teams; 1025 and above also switch the
    conditioning estimate and the back-transformation."""
    check([640, 641, 832, 833, 1024, 1025, 1280], molecule, threads=8)


def test_teams_that_leave_at_the_gate(monkeypatch):
    """A closed gate: every team leaves before it writes anything and one workgroup
    per system reduces the matrices instead."""
    monkeypatch.setenv("XTBLOOM_AMD_TEAMS", "0")
    check([258, 289, 353])


def check(sizes, make=stack, threads=4):
    rng = np.random.default_rng(sizes[0])
    b = workloads.from_systems([make(n, rng) for n in sizes])
    assert [O.basis_counts(b.system(i)["Z"])[1] for i in range(len(sizes))] == list(sizes)
    ctx = interface.Context("hip", 0)
    try:
        print("case reduction sizes", sizes, flush=True)
        out = interface.compute_arrays(ctx, b.atom_offsets, b.atomic_numbers, b.positions,
                                       b.molecular_charges, b.unpaired_electrons)
    finally:
        ctx.close()
    ref = O.batch(b.atom_offsets, b.atomic_numbers, b.positions, b.molecular_charges,
                  b.unpaired_electrons, threads=threads)
    assert np.all(out.per_system_status == 0) and np.all(ref["status"] == 0)
    print("|dE| %.1e |dF| %.1e |dq| %.1e" % (np.abs(out.energies - ref["energies"]).max(),
                                             np.abs(out.forces + ref["gradient"]).max(),
                                             np.abs(out.charges - ref["charges"]).max()), flush=True)
    assert np.abs(out.scc_iterations - ref["iterations"]).max() <= 1
    assert np.abs(out.energies - ref["energies"]).max() <= E_TOL
    assert np.abs(out.forces + ref["gradient"]).max() <= F_TOL
    assert np.abs(out.charges - ref["charges"]).max() <= Q_TOL


def test_result_depends_on_the_system_alone(monkeypatch):
    """64 systems of 302 AOs take 320 team members, more than the chip holds at once:
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
    b = workloads.from_systems([workloads.alkane(k, rng) for k in (213, 150, 108, 50)] + [stack(257, rng)])
    ctx = interface.Context("hip", 0)

    def run():
        return interface.compute_arrays(ctx, b.atom_offsets, b.atomic_numbers, b.positions, b.molecular_charges,
                                        b.unpaired_electrons, determinism=library.DETERMINISM_REPRODUCIBLE,
                                        kernel_stats=["tridiag"])

    try:
        print("case gate: 1280, 902, 650, 302 and 257 AOs by teams", flush=True)
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


def test_gate_failure_shortens_later_waits(monkeypatch):
    """Gates that no count fills: the first round waits 0.2 s, the others 20 ms each, and
    the result is that of the teams."""
    rng = np.random.default_rng(5)
    b = workloads.from_systems([workloads.alkane(50, rng), workloads.alkane(45, rng)])
    ctx = interface.Context("hip", 0)

    def run():
        return interface.compute_arrays(ctx, b.atom_offsets, b.atomic_numbers, b.positions, b.molecular_charges,
                                        b.unpaired_electrons, kernel_stats=["tridiag"])

    try:
        team = run()
        monkeypatch.setenv("XTBLOOM_AMD_TEAMS", "never")
        print("case gates that never fill, 302 and 272 AOs", flush=True)
        held = run()
    finally:
        ctx.close()
    rounds = int(team.scc_iterations.max())
    assert np.array_equal(held.energies, team.energies) and np.array_equal(held.charges, team.charges)
    ms = held.extension["kernel_stats"]["tridiag"]["ms"]
    print("reduction of %d rounds: %.0f ms" % (rounds, ms), flush=True)
    # 200 + 20 (rounds - 1) ms of waiting and one workgroup's work, below 20 ms a round
    assert 200.0 <= ms <= 200.0 + 40.0 * rounds
