"""The calls whose speed counts: GFN2-xTB energies, forces and charges through
the public entry points, from one small molecule to one of more than a
thousand orbitals.

A case names the entry point (``api``), the molecules (``kind``, ``batch``,
``kmin``..``kmax`` carbons of an alkane chain) and the options.  Molecules,
point charges and batch sizes are those of ``xtbloom_amd.workloads`` (the
benchmark's configurations) and of the GPU tests, with other counts.  ``draw``
gives more cases of the same ranges.
"""
import math

import numpy as np
import torch

from xtbloom_amd import interface, library, workloads
from xtbloom_amd.torch import xtbloom_torch

FLAGS = library.COMPUTE_ENERGY | library.COMPUTE_FORCES | library.COMPUTE_ATOMIC_CHARGES
R_CCL = 3.37  # bohr, a C-Cl bond (1.78 angstrom)
SCC_ROUNDS = 10  # of a FRESH start: alkanes and water take 9 to 13
WARM_ROUNDS = 7  # of a WARM start after a step of WARM_STEP
WARM_STEP = 0.005  # bohr, the displacement of an atom between two steps of a trajectory


def listed():
    return [
        # one water molecule through the Calculator: an interactive call, or one
        # energy of a script that loops over small molecules; latency only
        dict(name="water", api="calculator", kind="water", batch=1, kmin=0, kmax=0),
        # a few small molecules in one call (the smallest benchmark configuration)
        dict(name="water8", api="arrays", kind="water", batch=8, kmin=0, kmax=0),
        # one ordinary organic molecule of 62 atoms: an optimizer's or a
        # trajectory's single evaluation, host arrays in and out
        dict(name="c20_single", api="arrays", kind="alkane", batch=1, kmin=20, kmax=20),
        # 128 conformers of one molecule, device buffers (conformer ranking)
        dict(name="c20_128", api="tensors", kind="alkane", batch=128, kmin=20, kmax=20),
        # the same molecules as parallel trajectories: a fixed-topology plan,
        # every step a WARM start at a moved geometry
        dict(name="c20_128_md", api="plan_warm", kind="alkane", batch=128, kmin=20, kmax=20),
        # 512 uneven molecules of 8 to 116 atoms, device buffers: the benchmark's
        # headline batch, dataset labelling
        dict(name="ragged512", api="tensors", kind="ragged", batch=512, kmin=2, kmax=38),
        # uneven molecules, each in 500 point charges of a solvent, energies and
        # their gradients through autograd, forward and backward (learned potentials, QM/MM)
        dict(name="qmmm256_grad", api="autograd", kind="ragged", batch=256, kmin=6, kmax=26,
             waters=167),
        # open shells with two spin channels (radical reactions), host arrays
        dict(name="radicals96", api="arrays", kind="radical", batch=96, kmin=1, kmax=24),
        # molecules with a d shell (chlorine) in a uniform field, list of
        # structures through the batch calculator, dipole moments too
        dict(name="chloro_field48", api="batch", kind="chloro", batch=48, kmin=2, kmax=20,
             field=0.002),
        # periodic QM/MM coupling: b + A q per molecule, bit-reproducible mode
        dict(name="periodic64", api="arrays", kind="ragged", batch=64, kmin=3, kmax=30,
             operator=True, reproducible=True),
        # long chains of 242 to 482 orbitals in 1000 solvent charges: few
        # molecules, each above the sizes whose matrices fit one CU's registers
        dict(name="long16", api="tensors", kind="long", batch=16, kmin=40, kmax=80, waters=333),
        # one molecule of more than a thousand orbitals
        dict(name="c190_single", api="arrays", kind="alkane", batch=1, kmin=190, kmax=190),
    ]


def draw(rng):
    def between(lo, hi):  # spread over the logarithm
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    what = rng.choice(["water", "small", "ragged", "ragged", "uniform", "md", "grad", "radical",
                       "chloro", "periodic", "long", "single"])
    if what == "water":
        return dict(api=rng.choice(["arrays", "tensors"]), kind="water", batch=between(1, 512),
                    kmin=0, kmax=0)
    if what == "small":
        k = between(2, 45)
        return dict(api=rng.choice(["calculator", "arrays", "tensors"]), kind="alkane", batch=1,
                    kmin=k, kmax=k)
    if what == "ragged":
        kmin = between(2, 16)
        return dict(api=rng.choice(["tensors", "arrays", "batch"]), kind="ragged",
                    batch=between(2, 512), kmin=kmin, kmax=between(kmin, 42))
    if what == "uniform":
        k = between(3, 42)
        return dict(api="tensors", kind="alkane", batch=between(2, 384), kmin=k, kmax=k)
    if what == "md":
        k = between(3, 42)
        return dict(api="plan_warm", kind="alkane", batch=between(1, 256), kmin=k, kmax=k)
    if what == "grad":
        kmin = between(3, 12)
        return dict(api="autograd", kind="ragged", batch=between(1, 256), kmin=kmin,
                    kmax=between(kmin, 38), waters=between(5, 250))
    if what == "radical":
        kmin = between(1, 6)
        return dict(api="arrays", kind="radical", batch=between(1, 128), kmin=kmin,
                    kmax=between(max(kmin, 2), 36))
    if what == "chloro":
        kmin = between(2, 8)
        return dict(api="batch", kind="chloro", batch=between(1, 96), kmin=kmin,
                    kmax=between(kmin, 34), field=round(rng.uniform(0.0005, 0.004), 5))
    if what == "periodic":
        kmin = between(2, 8)
        return dict(api="arrays", kind="ragged", batch=between(1, 96), kmin=kmin,
                    kmax=between(kmin, 38), operator=True,
                    reproducible=bool(rng.randrange(2)))
    if what == "long":
        kmin = between(40, 60)
        return dict(api="tensors", kind="long", batch=between(1, 20), kmin=kmin,
                    kmax=between(kmin, 82), waters=between(30, 333))
    k = between(80, 186)
    return dict(api="arrays", kind="alkane", batch=1, kmin=k, kmax=k)


def _radical(k, rng):
    """An alkyl radical CkH(2k+1), or OH for k = 1: one unpaired electron."""
    if k < 2:
        z = np.array([8, 1], np.int32)
        xyz = np.array([[0.0, 0.0, 0.0], [1.83, 0.1, -0.05]]) + rng.normal(0.0, 0.02, (2, 3))
        return dict(Z=z, xyz=xyz, charge=0.0, uhf=1)
    s = workloads.alkane(k, rng)
    return dict(Z=s["Z"][:-1], xyz=s["xyz"][:-1], charge=0.0, uhf=1)


def _chloroalkane(k, rng):
    """An alkane with its last hydrogen replaced by chlorine along the C-H bond."""
    s = workloads.alkane(k, rng)
    z, xyz = s["Z"].copy(), s["xyz"].copy()
    carbons = np.flatnonzero(z == 6)
    c = carbons[np.argmin(np.linalg.norm(xyz[carbons] - xyz[-1], axis=1))]
    bond = xyz[-1] - xyz[c]
    z[-1] = 17
    xyz[-1] = xyz[c] + bond * (R_CCL / np.linalg.norm(bond))
    return dict(s, Z=z, xyz=xyz)


def _solvent(xyz, rng, waters):
    """Three-site water molecules (-0.834, +0.417, +0.417 e) as bare point
    charges around a solute: no site nearer than 4 bohr to any of its atoms, the
    oxygens up to 15 bohr from one."""
    h = 1.81 * np.array([[math.cos(0.912), math.sin(0.912), 0.0],
                         [math.cos(0.912), -math.sin(0.912), 0.0]])
    found = np.zeros((0, 3, 3))
    while len(found) < waters:
        d = rng.normal(size=(waters, 3))
        d *= (rng.uniform(4.0 ** 3, 15.0 ** 3, size=(waters, 1)) ** (1.0 / 3.0) /
              np.linalg.norm(d, axis=1, keepdims=True))
        o = xyz[rng.integers(0, len(xyz), size=waters)] + d
        turn = np.linalg.qr(rng.normal(size=(waters, 3, 3)))[0]
        sites = np.concatenate([o[:, None, :], o[:, None, :] + h @ turn], axis=1)
        gap = ((sites[:, :, None, :] - xyz) ** 2).sum(axis=3).min(axis=(1, 2))
        found = np.concatenate([found, sites[gap >= 16.0]])
    return dict(pc_xyz=found[:waters].reshape(-1, 3), pc_q=np.tile([-0.834, 0.417, 0.417], waters),
                pc_gamma=np.full(3 * waters, workloads.POINT_CHARGE_GAMMA))


def batch_of(case, seed):
    """The case's molecules as a packed ragged batch: the compositions belong to
    the case, the geometries and the surroundings to the seed."""
    rng = np.random.default_rng([int(seed), 20])
    kind, count, kmin, kmax = case["kind"], case["batch"], case["kmin"], case["kmax"]
    sizes = np.random.default_rng([count, kmin, kmax])
    systems = []
    for i in range(count):
        k = int(sizes.integers(kmin, kmax + 1))
        if count > 1 and i < 2:
            k = (kmax, kmin)[i]  # the range's ends are in every batch
        if kind == "water":
            s = workloads.water(rng)
        elif kind == "radical":
            s = _radical(k, rng)
        elif kind == "chloro":
            s = _chloroalkane(k, rng)
        else:
            sub = None
            if kind == "ragged" and sizes.random() < 0.5:
                sub = "OH" if sizes.random() < 0.5 else "NH2"
            s = workloads.alkane(k, rng, substituent=sub)
        if case.get("waters"):
            s.update(_solvent(s["xyz"], rng, case["waters"]))
        systems.append(s)
    return workloads.from_systems(systems), rng


def prepare(case, seed):
    batch, rng = batch_of(case, seed)
    api = case["api"]
    state = dict(api=api, batch=batch)
    if api == "calculator":
        s = batch.system(0)
        state["calc"] = interface.Calculator("GFN2-xTB", s["Z"], s["xyz"])
        return state
    if api == "batch":
        field = case.get("field")
        members = []
        for i in range(batch.batch_size):
            s = batch.system(i)
            direction = rng.normal(size=3)
            e = None if field is None else field * direction / np.linalg.norm(direction)
            members.append(interface.Structure(s["Z"], s["xyz"], efield=e))
        state["calc"] = interface.BatchCalculator(members)
        return state
    ctx = interface.Context("hip", 0)
    state["ctx"] = ctx
    args = dict(atom_offsets=batch.atom_offsets, numbers=batch.atomic_numbers,
                positions=batch.positions, charges=batch.molecular_charges,
                uhf=batch.unpaired_electrons)
    if batch.point_offsets is not None:
        args.update(point_offsets=batch.point_offsets, point_positions=batch.point_positions,
                    point_values=batch.point_charges, point_gammas=batch.point_gammas)
    if api == "arrays":
        if case["kind"] == "radical":
            args["spin_channels"] = np.full(batch.batch_size, 2, np.int32)
        if case.get("operator"):
            sizes = np.diff(batch.atom_offsets)
            roff = np.zeros(batch.batch_size + 1, np.int64)
            roff[1:] = np.cumsum(sizes * sizes)
            mats = []
            for n in sizes:
                a = rng.normal(scale=0.01, size=(n, n))
                mats.append((0.5 * (a + a.T) + 0.05 * np.eye(n)).ravel())
            args.update(atomic_potential_shifts=rng.normal(scale=0.01, size=int(sizes.sum())),
                        charge_response_offsets=roff, charge_response_matrix=np.concatenate(mats))
        if case.get("reproducible"):
            args["determinism"] = library.DETERMINISM_REPRODUCIBLE
        state["args"] = args
        return state
    dev = torch.device("cuda", 0)
    state["args"] = {k: torch.from_numpy(np.array(v)).to(dev) for k, v in args.items()}
    if api == "tensors":
        state["out"] = None
    elif api == "autograd":
        a = state["args"]
        a["positions"].requires_grad_()
        a["point_positions"].requires_grad_()
        a["point_values"].requires_grad_()
        state["weights"] = torch.from_numpy(rng.normal(size=batch.batch_size)).to(dev)
    elif api == "plan_warm":
        # a trajectory after its first step: converged at the geometry it comes from
        state["plan"] = interface.Plan(ctx, batch.atom_offsets, batch.atomic_numbers,
                                       batch.positions, batch.molecular_charges,
                                       batch.unpaired_electrons, flags=FLAGS)
        a = state["args"]
        state["here"] = a.pop("positions")
        step = rng.normal(0.0, WARM_STEP, batch.positions.shape)
        state["there"] = state["here"] + torch.from_numpy(step).to(dev)
        interface.compute_tensors(ctx, positions=state["here"], flags=FLAGS, plan=state["plan"], **a)
    return state


def _arrays(out):
    d = dict(energies=out.energies, forces=out.forces, charges=out.charges,
             iterations=out.scc_iterations, converged=out.scc_converged,
             status=out.per_system_status)
    if out.point_charge_forces is not None:
        d["point_charge_forces"] = out.point_charge_forces
    return d


def _tensors(out):
    return {k: out[k] for k in ("energies", "forces", "charges", "point_charge_forces",
                                "scc_iterations", "scc_converged", "per_system_status")
            if k in out}


def run(state):
    api = state["api"]
    if api == "calculator":
        r = state["calc"].singlepoint()
        return dict(energy=r.energy, forces=r.forces, charges=r.charges,
                    iterations=r.scc_iterations, converged=r.scc_converged)
    if api == "batch":
        r = state["calc"].compute()
        return {k: r.get(k) for k in ("energies", "forces", "charges", "dipole_moments",
                                      "scc_iterations", "scc_converged", "scc_status")
                if r.get(k) is not None}
    if api == "arrays":
        return _arrays(interface.compute_arrays(state["ctx"], **state["args"]))
    if api == "tensors":
        # the caller's output tensors, allocated by the first call
        a = state["args"]
        flags = FLAGS | library.COMPUTE_POINT_CHARGE_FORCES if "point_values" in a else FLAGS
        state["out"], _ = interface.compute_tensors(state["ctx"], flags=flags,
                                                    outputs=state["out"], **a)
        return _tensors(state["out"])
    a = state["args"]
    if api == "autograd":
        e, f = xtbloom_torch(a["positions"], a["numbers"], a["atom_offsets"], a["charges"],
                             a["uhf"], context=state["ctx"], point_offsets=a["point_offsets"],
                             point_positions=a["point_positions"],
                             point_values=a["point_values"], point_gammas=a["point_gammas"])
        loss = (state["weights"] * e).sum()
        grads = torch.autograd.grad(loss, (a["positions"], a["point_positions"],
                                           a["point_values"]))
        return dict(energies=e.detach(), forces=f.detach(), grad_positions=grads[0],
                    grad_point_positions=grads[1], grad_point_values=grads[2])
    # two steps of a trajectory: there and back, each a WARM start
    steps = []
    for where in ("there", "here"):
        out, _ = interface.compute_tensors(state["ctx"], positions=state[where], flags=FLAGS,
                                           plan=state["plan"],
                                           scc_start_mode=library.SCC_START_WARM, **a)
        steps.append(_tensors(out))
    return steps


def work(case):
    """Inputs read and outputs written once; the flops of the dense algebra per
    system, (25/3) k n^3 + (7/3) n^3 for n orbitals and k SCC rounds (Householder
    reduction 4/3, back-transformation 2, products 5, and the overlap factor)."""
    batch, _ = batch_of(case, 0)
    z = batch.atomic_numbers
    orbitals = np.where(z == 1, 1, np.where(z == 17, 9, 4))
    n = np.add.reduceat(orbitals, batch.atom_offsets[:-1]).astype(float)
    atoms, systems = len(z), batch.batch_size
    points = 0 if batch.point_charges is None else len(batch.point_charges)
    moved = atoms * (4 + 24 + 24 + 8) + systems * (8 + 8 + 4 + 8 + 5) + points * (24 + 8 + 8 + 32)
    if case.get("operator"):
        moved += 8 * (atoms + int((np.diff(batch.atom_offsets) ** 2).sum()))
    channels = 2 if case["kind"] == "radical" else 1
    rounds = SCC_ROUNDS
    flops = float((n ** 3).sum()) * (channels * 25.0 / 3.0 * rounds + 7.0 / 3.0)
    if case["api"] == "plan_warm":
        moved *= 2
        flops = 2.0 * float((n ** 3).sum()) * (25.0 / 3.0 * WARM_ROUNDS + 7.0 / 3.0)
    return {"bytes": float(moved), "flops": flops}


def tolerance(case):
    """With the atoms of every molecule in another order (so every sum too), the
    listed cases and 45 drawn ones changed by at most 5e-11 of an output's norm
    and 1e-9 of its largest deviation, growing with the molecule, and no
    iteration count changed."""
    return {"rel": 4e-10, "max": 8e-9}


def exact(case, seed):
    """None: the outputs are the end of a whole self-consistent GFN2-xTB
    calculation (integrals, D4, mixing, forces and their parameter tables),
    which plain torch does not hold; all of it already runs in 64 bits."""
    return None
