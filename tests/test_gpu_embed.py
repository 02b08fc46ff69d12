"""Device start-geometry embedder (csrc/embed.hip) against the host embedder (csrc/embed.c)
it moves onto the GPU, from the same seeds:

* the restraint energy (restated here in numpy from its definition: equality springs
  100 (d - d0)^2, lower-bound walls 10 (d_min - d)^2 for d < d_min) of the noise-free device
  geometries is as small as the host's (the two agree conformer by conformer when their
  FP64 relaxations take the same steps), and bond lengths are as close to their MMFF r0;
* two runs give identical coordinates (fixed-point gradient sums, fixed-order energies);
* noise N(0, sigma) is added with the right spread;
* BFGS from device starts converges as from host starts, to energies of the same size.
"""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def restraint_energy(params, z, x):
    from mlxmolkit_archive_amd.embed import restraints
    ri, rj, d0, kind = restraints(params, np.asarray(z))
    p = x.reshape(-1, 3).astype(np.float64)
    d = np.linalg.norm(p[ri] - p[rj], axis=1)
    eq = kind == 0
    wall = ~eq & (d < d0)
    return float(np.sum(100.0 * (d[eq] - d0[eq]) ** 2) + np.sum(10.0 * (d[wall] - d0[wall]) ** 2))


def _split(params, counts, x):
    out, off = [], 0
    for p, c in zip(params, counts):
        for _ in range(c):
            out.append(x[off:off + 3 * p.n_atoms])
            off += 3 * p.n_atoms
    return out


def test_device_embedder_satisfies_restraints_like_host():
    from mlxmolkit_archive_amd import molgen, workloads
    from mlxmolkit_archive_amd.embed import embed, embed_device
    mols = molgen.generate("ragged", 24, seed=molgen.SEED_BASE + 3)
    params = workloads._typed((mols, "MMFF94"))
    z = [m.atomic_numbers() for m in mols]
    counts = [3] * len(mols)
    seeds = np.arange(sum(counts), dtype=np.uint64) + np.uint64(99)
    xd = embed_device(params, z, counts, seeds=seeds, noise=0.0)
    xd2 = embed_device(params, z, counts, seeds=seeds, noise=0.0)
    torch.cuda.synchronize()
    xd, xd2 = xd.cpu().numpy(), xd2.cpu().numpy()
    assert np.array_equal(xd, xd2) and np.isfinite(xd).all()
    xh = embed(params, z, counts, seeds=seeds, noise=0.0)
    conf_p = [p for p, c in zip(params, counts) for _ in range(c)]
    conf_z = [zz for zz, c in zip(z, counts) for _ in range(c)]
    ed = np.array([restraint_energy(p, zz, x) for p, zz, x in zip(conf_p, conf_z, _split(params, counts, xd))])
    eh = np.array([restraint_energy(p, zz, x) for p, zz, x in zip(conf_p, conf_z, _split(params, counts, xh))])
    # bond lengths against the MMFF r0 targets (springs compete with the walls, so neither
    # embedder meets every target exactly)
    def worst_bond(xs):
        out = []
        for p, x in zip(conf_p, _split(params, counts, xs)):
            q = x.reshape(-1, 3)
            out.append(np.abs(np.linalg.norm(q[p.bond_idx1] - q[p.bond_idx2], axis=1) - p.bond_r0).max())
        return np.array(out)
    bd, bh = worst_bond(xd), worst_bond(xh)
    same = np.isclose(ed, eh, rtol=1e-6, atol=1e-6)
    print(f"\nrestraint energy per conformer: device median {np.median(ed):.3f} max {ed.max():.3f}; "
          f"host median {np.median(eh):.3f} max {eh.max():.3f}; equal for {same.sum()}/{len(ed)} conformers; "
          f"worst bond |d - r0| device {bd.max():.3f} host {bh.max():.3f} A")
    assert np.median(ed) <= 1.1 * np.median(eh) + 0.05
    assert np.percentile(ed, 90) <= 1.25 * np.percentile(eh, 90) + 0.5
    assert np.median(bd) <= np.median(bh) + 0.02


def test_device_embedder_noise_and_minimization():
    from mlxmolkit_archive_amd import engine, molgen, workloads
    from mlxmolkit_archive_amd.embed import embed_device
    mols = molgen.generate("medium", 12, seed=molgen.SEED_BASE + 4)
    params = workloads._typed((mols, "MMFF94"))
    z = [m.atomic_numbers() for m in mols]
    counts = [2] * len(mols)
    seeds = np.arange(sum(counts), dtype=np.uint64) + np.uint64(7)
    x0 = embed_device(params, z, counts, seeds=seeds, noise=0.0).cpu().numpy()
    x1 = embed_device(params, z, counts, seeds=seeds, noise=0.1)
    dx = x1.cpu().numpy() - x0
    assert abs(dx.std() - 0.1) < 0.01 and abs(dx.mean()) < 0.01
    db = engine.device_batch(params, counts)
    res = engine.NkRunner(db, max_iters=2000, grad_tol=1e-4, ls_grad=True).run(x1)
    torch.cuda.synchronize()
    st = res.status.cpu().numpy()
    e = res.energy.cpu().numpy()
    print(f"\nBFGS from device starts: status0 {np.mean(st == 0):.3f}, mean iterations "
          f"{res.counters.cpu().numpy()[:, 0].mean():.1f}, energy range {e.min():.1f}..{e.max():.1f}")
    assert np.mean(st == 0) >= 0.95 and np.isfinite(e).all()


def _chain(n):
    """Restraint table of an n-atom zigzag: 1-2 and 1-3 springs, walls between atoms 3 to 9 apart."""
    i, j, d = [], [], []
    for k in range(n):
        for s in range(1, 10):
            if k + s < n:
                i.append(k), j.append(k + s), d.append(1.5 if s == 1 else 2.5 if s == 2 else -3.0)
    ij = np.array(i, np.uint32) | (np.array(j, np.uint32) << 16)
    return ij.astype(np.uint32), np.array(d, np.float32)


@pytest.mark.parametrize("n", [1, 2, 20, 65, 131])
def test_embedding_does_not_depend_on_the_batch(n):
    """A molecule alone, and beside one so large that its coordinates leave no LDS for the waves'
    queues of active restraints: the same geometry. The two kernels add the same energies in
    another order, so they take the same steps unless two energies agree to rounding; 1e-5 A
    allows one float rounding of a coordinate (2^-23 of at most 40 A). Up to 1,279 atoms fit."""
    from types import SimpleNamespace
    from mlxmolkit_archive_amd.embed import embed_device
    big = 1279
    tabs = [_chain(n), _chain(big)]
    ps = [SimpleNamespace(n_atoms=n), SimpleNamespace(n_atoms=big)]
    seeds = np.array([5, 6, 7], np.uint64)
    alone = embed_device(ps[:1], [None], [2], seeds=seeds[:2], noise=0.1, tables=tabs[:1]).cpu().numpy()
    both = embed_device(ps, [None] * 2, [2, 1], seeds=seeds, noise=0.1, tables=tabs).cpu().numpy()
    assert alone.shape == (6 * n,) and np.isfinite(both).all()
    assert np.abs(alone - both[:6 * n]).max() <= 1e-5
    with pytest.raises(RuntimeError, match="too large"):
        embed_device([SimpleNamespace(n_atoms=big + 1)], [None], [1], seeds=seeds[:1], tables=[_chain(n)])
