"""Oracle results at the size switches above 1280 AOs (tests/golden/switch_sizes.npz).

    python tests/golden/make_switch_fixture.py

One molecule each of 1281, 1536, 1537, 2048 and 2049 AOs through
``oracle.singlepoint`` with the default options (a few minutes on one core
each); the geometries are stored with the results.
"""
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
sys.path.insert(0, ROOT)

import numpy as np  # noqa: E402

from oracle import oracle as O  # noqa: E402
from tests.test_gpu_reduction_sizes import molecule  # noqa: E402
from xtbloom_amd import workloads  # noqa: E402

SIZES = (1281, 1536, 1537, 2048, 2049)


def main():
    systems = [molecule(n, np.random.default_rng(n)) for n in SIZES]
    assert [O.basis_counts(s["Z"])[1] for s in systems] == list(SIZES)
    b = workloads.from_systems(systems)
    r = O.batch(b.atom_offsets, b.atomic_numbers, b.positions, b.molecular_charges, b.unpaired_electrons,
                threads=len(SIZES))
    assert np.all(r["status"] == 0)
    np.savez_compressed(os.path.join(ROOT, "tests", "golden", "switch_sizes.npz"), sizes=np.array(SIZES, np.int32),
             atom_offsets=b.atom_offsets, Z=b.atomic_numbers.astype(np.int32), xyz=b.positions,
             energies=r["energies"], gradient=r["gradient"], charges=r["charges"], iterations=r["iterations"])
    print("energies", r["energies"].tolist(), "iterations", r["iterations"].tolist())


if __name__ == "__main__":
    main()
