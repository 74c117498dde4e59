"""Real space on cell grids (the half-shell kernel: each unordered pair once,
the reaction added to the partner) against the oracle's Realteil
(realpart.c:124-167): dense cells of several 64-particle chunks next to
sparse ones, clusters that wrap across the periodic boundary, both cell
sizes (side rcut / 2, and side rcut for sparse systems), the device entry
point accumulating into the caller's arrays, and the mixed form."""
import ctypes
import math

import numpy as np
import pytest

from conftest import cell_geometry, cells_of, rel_err

pytestmark = pytest.mark.gpu


def corner_cluster(n_cluster, n_background, L, sigma, seed, centre=(0.0, 0.0, 0.0)):
    """A Gaussian cluster about `centre` (folded into the box, so at a corner
    it spans the periodic boundary on all three axes) plus a uniform
    background; charges +-1, neutral."""
    rng = np.random.default_rng(seed)
    c = rng.normal(0.0, sigma, (n_cluster, 3)) + np.asarray(centre)
    b = rng.uniform(0.0, L, (n_background, 3))
    p = np.mod(np.concatenate([c, b]), L)
    p[p >= L] = 0.0
    n = n_cluster + n_background
    q = np.where(np.arange(n) % 2 == 0, 1.0, -1.0)
    if n % 2:
        q[-1] = 0.0
    return {"x": p[:, 0].copy(), "y": p[:, 1].copy(), "z": p[:, 2].copy(), "q": q, "L": float(L)}


def lattice(side, L, seed):
    """side^3 particles in site order, jittered: no two closer than 0.4 sites."""
    rng = np.random.default_rng(seed)
    site = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)
    p = (site + 0.5 + 0.6 * (rng.uniform(size=site.shape) - 0.5)) * (L / side)
    q = np.where(np.arange(len(p)) % 2 == 0, 1.0, -1.0)
    return {"x": p[:, 0].copy(), "y": p[:, 1].copy(), "z": p[:, 2].copy(), "q": q, "L": float(L)}


class DeviceRealteil:
    """realteil_device of `solver` on device copies of a system."""

    def __init__(self, solver, s, rcut, alpha):
        import torch

        self.solver, self.rcut, self.alpha = solver, rcut, alpha
        self.n, self.L = len(s["q"]), s["L"]
        self.dev = {k: torch.empty(self.n, dtype=torch.float64, device="cuda") for k in "xyzq"}
        self.fr = torch.zeros(3 * self.n, dtype=torch.float64, device="cuda")
        self.en = torch.zeros(1, dtype=torch.float64, device="cuda")
        self.put(s)

    def put(self, s):
        import torch

        self.solver.synchronize()
        for k in "xyzq":
            self.dev[k].copy_(torch.tensor(s[k]))
        torch.cuda.synchronize()

    def run(self, calls=1):
        """Forces (3, n) and energy, summed over `calls` calls."""
        import torch

        for _ in range(calls):
            self.solver.realteil_device(self.n, self.L, *[self.dev[k].data_ptr() for k in "xyzq"], self.rcut,
                                        self.alpha, self.fr.data_ptr(), self.en.data_ptr())
        self.solver.synchronize()
        out = self.fr.cpu().numpy().reshape(3, self.n).copy(), float(self.en.item())
        self.fr.zero_()
        self.en.zero_()
        torch.cuda.synchronize()
        return out


def on_cells(pkg, s, rcut, alpha, reach, prec_name="FP64"):
    """Real-space forces, energy and cells per side of `s` (below 7
    particles per cell of side rcut / 2 on average) on a cell list of the given
    reach: the list is made by a first call, for uniform positions (reach 1)
    or for a cluster (reach 2), and kept for `s`."""
    rng = np.random.default_rng(1)
    n, L = len(s["q"]), s["L"]
    first = rng.uniform(0.0, L if reach == 1 else L / 16, (3, n))
    solver = pkg.Solver(0, pkg.HostSystem.from_dict(s), pkg.parameters(16, 3, alpha, rcut),
                        getattr(pkg, prec_name))
    dev = DeviceRealteil(solver, dict(s, x=first[0], y=first[1], z=first[2]), rcut, alpha)
    dev.run()
    dev.put(s)
    f, e = dev.run()
    nc, got = cells_of(pkg, solver)
    assert got == reach
    solver.close()
    return f, e, nc


def cell_counts(s, nc):
    """Particles per cell of a grid of nc cells per side."""
    L = s["L"]
    c = np.minimum((np.stack([s["x"], s["y"], s["z"]], 1) * nc / L).astype(int), nc - 1)
    return np.bincount((c[:, 0] * nc + c[:, 1]) * nc + c[:, 2], minlength=nc ** 3)


@pytest.mark.parametrize("L,n_background,centre,reach", [
    (14.0, 2500, (0.0, 0.0, 0.0), 2), (14.0, 2500, (7.0, 0.3, 13.9), 2),
    (30.0, 1000, (0.0, 0.0, 0.0), 1), (30.0, 1000, (29.5, 15.0, 0.2), 1)])
def test_wrapped_dense_cluster(pkg, orc, L, n_background, centre, reach):
    """A cluster across the box corner / faces: cells of up to several
    hundred particles (several chunks; the candidate search on the matrix
    cores), sparse background cells (the vector search), image shifts inside
    dense cell pairs; with cells of side rcut / 2 and of side rcut."""
    rcut, alpha = 3.0, 1.0
    s = corner_cluster(2500 if reach == 2 else 2000, n_background, L, 0.9, seed=31, centre=centre)
    f, e, nc = on_cells(pkg, s, rcut, alpha, reach)
    cnt = cell_counts(s, nc)
    assert nc >= 2 * reach + 1 and cnt.max() > 128 and np.sum((cnt > 0) & (cnt <= 4)) > 50
    system = pkg.HostSystem.from_dict(s)
    forces = pkg.realteil(system, rcut, alpha)
    fr_ref, e_ref = orc.realteil(s, rcut, alpha)
    err = max(rel_err(forces.real(), fr_ref), rel_err(f, fr_ref))
    print("reach %d, max cell %d, rel err %.2e, energy %.15e vs %.15e" % (
        reach, cnt.max(), err, system.c.energy, e_ref))
    assert err < 1e-13
    assert abs(system.c.energy - e_ref) <= 1e-12 * abs(e_ref)
    assert abs(e - e_ref) <= 1e-12 * abs(e_ref)


@pytest.mark.parametrize("reach,nc", [(1, 3), (2, 7)])
def test_single_dense_cell_of_many_chunks(pkg, orc, reach, nc):
    """One cell of ~600 particles (ten chunks: the item's own chunk, later
    chunks of its cell, earlier ones left to their own items) in an
    otherwise sparse box."""
    L, rcut, alpha = 12.0, 3.0, 1.2
    rng = np.random.default_rng(5)
    side = L / nc
    cell = rng.uniform(1 * side + 1e-3, 2 * side - 1e-3, (600, 3))
    rest = rng.uniform(0.0, L, (300, 3))
    p = np.concatenate([cell, rest])
    q = np.where(np.arange(900) % 2 == 0, 1.0, -1.0)
    s = {"x": p[:, 0].copy(), "y": p[:, 1].copy(), "z": p[:, 2].copy(), "q": q, "L": L}
    assert cell_counts(s, nc).max() >= 600
    f, e, got_nc = on_cells(pkg, s, rcut, alpha, reach)
    assert got_nc == nc
    system = pkg.HostSystem.from_dict(s)
    forces = pkg.realteil(system, rcut, alpha)
    fr_ref, e_ref = orc.realteil(s, rcut, alpha)
    assert rel_err(forces.real(), fr_ref) < 1e-13
    assert abs(system.c.energy - e_ref) <= 1e-12 * abs(e_ref)
    assert rel_err(f, fr_ref) < 1e-13
    assert abs(e - e_ref) <= 1e-12 * abs(e_ref)


def test_newton_third_law(pkg):
    """Each unordered pair enters both partners with opposite sign, so the
    real-space forces of a periodic system sum to zero (to rounding)."""
    L, rcut, alpha = 14.0, 3.0, 1.0
    s = corner_cluster(2000, 500, L, 1.2, seed=8, centre=(7.0, 7.0, 7.0))
    forces = pkg.realteil(pkg.HostSystem.from_dict(s), rcut, alpha)
    f = forces.real()
    assert np.abs(f.sum(axis=1)).max() < 1e-10 * np.abs(f).sum()


@pytest.mark.parametrize("prec_name", ["FP64", "MIXED"])
def test_device_form_accumulates_and_mixed_is_close(pkg, orc, prec_name):
    """The device entry point (both precision forms) adds the real-space
    forces to the caller's array and the energy to its scalar; the mixed form
    has the FP64 form's pair set (its energy agrees to FP32 rounding) and
    forces within 1e-6 of the force norm (its pair energies are summed in
    FP32 per lane, hence 1e-5 on the energy)."""
    import torch

    L, rcut, alpha = 14.0, 3.0, 1.0
    s = corner_cluster(2500, 700, L, 0.9, seed=12)
    n = len(s["q"])
    fr_ref, e_ref = orc.realteil(s, rcut, alpha)
    prec = getattr(pkg, prec_name)
    solver = pkg.Solver(3, pkg.HostSystem.from_dict(s), pkg.parameters(16, 5, alpha, rcut), prec)
    dev = {k: torch.tensor(np.asarray(s[k]), dtype=torch.float64, device="cuda") for k in "xyzq"}
    fr = torch.full((3 * n,), 2.0, dtype=torch.float64, device="cuda")
    en = torch.full((1,), 5.0, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    solver.realteil_device(n, L, *[dev[k].data_ptr() for k in "xyzq"], rcut, alpha, fr.data_ptr(),
                           en.data_ptr())
    solver.synchronize()
    got = fr.cpu().numpy().reshape(3, n) - 2.0
    e = float(en.item()) - 5.0
    solver.close()
    err = rel_err(got, fr_ref)
    print("%s: rel err %.2e, energy rel %.2e" % (prec_name, err, abs(e - e_ref) / abs(e_ref)))
    if prec_name == "FP64":
        assert err < 1e-13
        assert abs(e - e_ref) <= 1e-12 * abs(e_ref)
    else:
        assert err < 1e-6
        assert abs(e - e_ref) <= 1e-5 * abs(e_ref)


@pytest.mark.parametrize("m,reach", [(400, 1), (1400, 2)])
def test_pairs_at_the_cutoff(pkg, orc, m, reach):
    """Pairs placed within 1e-9 of rcut on either side, in all directions and
    across cell and box boundaries: the candidate search (FP16 operands in
    units of the cell side, with a margin) passes all of them and the exact
    FP64 test keeps exactly the reference's ones; both cell sizes."""
    L, rcut, alpha = 12.0, 3.0, 0.8
    assert cell_geometry(2 * m, L, rcut)[1] == reach
    rng = np.random.default_rng(77)
    a = rng.uniform(0.0, L, (m, 3))
    u = rng.normal(size=(m, 3))
    u /= np.linalg.norm(u, axis=1)[:, None]
    eps = np.where(np.arange(m) % 2 == 0, -1e-9, 1e-9)
    b = a + (rcut * (1.0 + eps))[:, None] * u
    p = np.mod(np.concatenate([a, b]), L)
    p[p >= L] = 0.0
    q = np.concatenate([np.ones(m), -np.ones(m)])
    s = {"x": p[:, 0].copy(), "y": p[:, 1].copy(), "z": p[:, 2].copy(), "q": q, "L": L}
    system = pkg.HostSystem.from_dict(s)
    forces = pkg.realteil(system, rcut, alpha)
    fr_ref, e_ref = orc.realteil(s, rcut, alpha)
    assert rel_err(forces.real(), fr_ref) < 1e-13
    assert abs(system.c.energy - e_ref) <= 1e-12 * abs(e_ref)


@pytest.mark.parametrize("m,reach", [(400, 1), (1400, 2)])
def test_pairs_at_the_cutoff_mixed(pkg, orc, m, reach):
    """The mixed form on the pairs of test_pairs_at_the_cutoff: their FP32
    squared distances fall inside the band around rcut^2, where the FP64 test
    decides on the FP64 positions with the pair's image shift (many of the
    pairs wrap across the box).  One pair decided the other way would move
    its two particles' forces by the pair force at rcut, f_c = 3.4e-4: each
    particle's error is held to 1e-5 of its force plus f_c / 10 (FP32
    rounding stays near 1e-7 of the force), besides the mixed form's 1e-6
    on the norm."""
    import torch

    L, rcut, alpha = 12.0, 3.0, 0.8
    assert cell_geometry(2 * m, L, rcut)[1] == reach
    rng = np.random.default_rng(78)
    a = rng.uniform(0.0, L, (m, 3))
    u = rng.normal(size=(m, 3))
    u /= np.linalg.norm(u, axis=1)[:, None]
    eps = np.where(np.arange(m) % 2 == 0, -1e-9, 1e-9)
    b = a + (rcut * (1.0 + eps))[:, None] * u
    p = np.mod(np.concatenate([a, b]), L)
    p[p >= L] = 0.0
    q = np.concatenate([np.ones(m), -np.ones(m)])
    s = {"x": p[:, 0].copy(), "y": p[:, 1].copy(), "z": p[:, 2].copy(), "q": q, "L": L}
    n = 2 * m
    fr_ref, e_ref = orc.realteil(s, rcut, alpha)
    solver = pkg.Solver(3, pkg.HostSystem.from_dict(s), pkg.parameters(16, 5, alpha, rcut), pkg.MIXED)
    dev = {k: torch.tensor(np.asarray(s[k]), dtype=torch.float64, device="cuda") for k in "xyzq"}
    fr = torch.zeros(3 * n, dtype=torch.float64, device="cuda")
    en = torch.zeros(1, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    solver.realteil_device(n, L, *[dev[k].data_ptr() for k in "xyzq"], rcut, alpha, fr.data_ptr(),
                           en.data_ptr())
    solver.synchronize()
    got = fr.cpu().numpy().reshape(3, n)
    e = float(en.item())
    solver.close()
    err = rel_err(got, fr_ref)
    fc = (math.erfc(alpha * rcut) / rcut + 2.0 * alpha / math.sqrt(math.pi) * math.exp(-(alpha * rcut) ** 2)) / rcut**2
    dev_i = np.linalg.norm(got - fr_ref, axis=0)
    bound_i = 1e-5 * np.linalg.norm(fr_ref, axis=0) + 0.1 * fc
    print("mixed at the cutoff (m %d, reach %d): rel err %.2e, worst particle %.2e of its bound"
          % (m, reach, err, (dev_i / bound_i).max()))
    assert (dev_i <= bound_i).all()
    assert err < 1e-6
    assert abs(e - e_ref) <= 1e-5 * abs(e_ref)


def test_stage_ring_pair_kernel_times(pkg):
    """The per-step pair-kernel times of the stage ring: positive, within the
    step's real-space stage (which also holds the cell list), and 0 for a
    step without real space."""
    import torch

    L, rcut, alpha = 14.0, 3.0, 1.0
    s = corner_cluster(2500, 700, L, 0.9, seed=14)
    n = len(s["q"])
    solver = pkg.Solver(3, pkg.HostSystem.from_dict(s), pkg.parameters(16, 5, alpha, rcut), pkg.MIXED)
    dev = {k: torch.tensor(np.asarray(s[k]), dtype=torch.float64, device="cuda") for k in "xyzq"}
    f, fk, fr = (torch.zeros(3 * n, dtype=torch.float64, device="cuda") for _ in range(3))
    ptr = [dev[k].data_ptr() for k in "xyzq"]
    torch.cuda.synchronize()
    solver.stage_ring_start(3)
    for rc in (rcut, rcut, 0.0):
        solver.calculate_forces_device(n, L, *ptr, rc, alpha, f.data_ptr(), fk.data_ptr(), fr.data_ptr(),
                                       None)
    stages = solver.stage_ring_read(3)
    pairs = solver.stage_ring_read_pairs(3)
    solver.stage_ring_start(0)
    solver.close()
    print(stages[:, 4], pairs)
    assert len(pairs) == 3
    assert all(0.0 < pairs[k] <= stages[k, 4] for k in (0, 1))
    assert pairs[2] == 0.0


@pytest.mark.parametrize("prec_name", ["FP64", "MIXED"])
@pytest.mark.parametrize("cells,per_cell,units", [(3, 37, 16), (6, 9, 8), (7, 8, 4), (8, 8, 2), (13, 4, 1), (16, 3, 1),
                                                  (17, 3, 1)])
def test_items_dealt_to_several_wavefronts(pkg, orc, cells, per_cell, units, prec_name):
    """Systems of few work items, whose neighbour cells are dealt out to 16,
    8, 4, 2 or one wavefront per item (items from 27 to above 4096, one cell
    of 150 particles among them so that items of one cell differ in chunks):
    sums of up to 16 shares per particle and of the energy, so the tolerances
    are those of the other real-space tests (FP64 1e-13, energy 1e-12; mixed
    1e-6 by the fixed-point quantum at these densities' closest pairs, kept
    above 0.05, energy 1e-5)."""
    rcut, alpha = 3.0, 1.0
    L = rcut * cells * 1.001
    rng = np.random.default_rng(100 + cells)
    side = int(round((per_cell * cells ** 3) ** (1.0 / 3.0)))
    lattice = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)
    p = (lattice + 0.5 + 0.6 * (rng.uniform(size=lattice.shape) - 0.5)) * (L / side)
    p = np.concatenate([p, rng.uniform(0.05, 2.9, (150, 3))])
    gap = np.linalg.norm(p[-150:, None] - p[None], axis=2)
    gap[np.arange(150), np.arange(len(p) - 150, len(p))] = 1.0
    p = np.delete(p, len(p) - 150 + np.nonzero(gap.min(1) < 0.05)[0], axis=0)
    n = len(p)
    q = np.where(np.arange(n) % 2 == 0, 1.0, -1.0)
    s = {"x": p[:, 0].copy(), "y": p[:, 1].copy(), "z": p[:, 2].copy(), "q": q, "L": float(L)}
    fr_ref, e_ref = orc.realteil(s, rcut, alpha, cells=True)
    f, e, nc = on_cells(pkg, s, rcut, alpha, 1, prec_name)
    assert nc == cells
    items = int(((cell_counts(s, nc) + 63) // 64).sum())
    dealt = 1
    while dealt < 16 and items * dealt < 1024:
        dealt *= 2
    assert dealt == units
    err = rel_err(f, fr_ref)
    print("cells %d n %d items %d %s rel err %.2e energy %.2e" % (cells, n, items, prec_name, err, abs(e / e_ref - 1)))
    assert err < (1e-13 if prec_name == "FP64" else 1e-6)
    assert abs(e - e_ref) <= (1e-12 if prec_name == "FP64" else 1e-5) * abs(e_ref)


@pytest.mark.parametrize("prec_name", ["FP64", "MIXED"])
@pytest.mark.parametrize("layout", ["dense", "clustered", "sparse"])
def test_cell_size_follows_the_clustering(pkg, orc, layout, prec_name):
    """Cells of side rcut / 2 for a dense uniform system (18 per such cell)
    and for one that is sparse on average but clustered (its mean per cell is
    below the sparse one's), cells of side rcut for the sparse one: all
    against the oracle (FP64 1e-13; mixed 1e-6 with closest pairs above 0.05)."""
    import torch

    rcut, alpha = 3.0, 1.0
    rng = np.random.default_rng(11)
    L, side = {"dense": (12.0, 19), "clustered": (30.0, 14), "sparse": (18.0, 14)}[layout]
    lattice = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)
    box = 6.0 if layout == "clustered" else L
    p = (lattice + 0.5 + 0.6 * (rng.uniform(size=lattice.shape) - 0.5)) * (box / side)
    if layout == "clustered":
        p = np.mod(p - 2.0, L)  # across the box corner
    n = len(p)
    s = {"x": p[:, 0].copy(), "y": p[:, 1].copy(), "z": p[:, 2].copy(),
         "q": np.where(np.arange(n) % 2 == 0, 1.0, -1.0), "L": L}
    fr_ref, _ = orc.realteil(s, rcut, alpha, cells=True)
    solver = pkg.Solver(0, pkg.HostSystem.from_dict(s), pkg.parameters(16, 3, alpha, rcut),
                        getattr(pkg, prec_name))
    dev = {k: torch.tensor(s[k], dtype=torch.float64, device="cuda") for k in "xyzq"}
    fr = torch.zeros(3 * n, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    solver.realteil_device(n, L, *[dev[k].data_ptr() for k in "xyzq"], rcut, alpha, fr.data_ptr(), None)
    solver.synchronize()
    err = rel_err(fr.cpu().numpy().reshape(3, n), fr_ref)
    print("%s %s rel err %.2e" % (layout, prec_name, err))
    assert cells_of(pkg, solver)[1] == (1 if layout == "sparse" else 2)
    assert err < (1e-13 if prec_name == "FP64" else 1e-6)
    solver.close()


@pytest.mark.parametrize("held", ["nothing", "unreadable", "zeros"])
def test_init_reads_sizes_only(pkg, orc, held):
    """Init takes the particle count and the box length of a system whose
    arrays are absent, not readable by the host, or placeholders; the cell
    size follows the positions of the first real-space call (uniform and
    sparse here: side rcut)."""
    rcut, alpha = 3.0, 1.0
    s = lattice(12, 18.0, seed=3)
    system = pkg.HostSystem.from_dict(dict(s, **{k: np.zeros_like(s[k]) for k in "xyz"}))
    if held == "nothing":
        system.c.p, system.c.q = None, None
    elif held == "unreadable":
        nowhere = ctypes.cast(ctypes.c_void_p(8), ctypes.POINTER(ctypes.c_double))
        system.c.p.contents.x = system.c.p.contents.y = system.c.p.contents.z = system.c.q = nowhere
    solver = pkg.Solver(7, system, pkg.parameters(16, 3, alpha, rcut))
    fr, _ = DeviceRealteil(solver, s, rcut, alpha).run()
    assert cells_of(pkg, solver)[1] == 1
    assert rel_err(fr, orc.realteil(s, rcut, alpha, cells=True)[0]) < 1e-13
    solver.close()


@pytest.mark.parametrize("side", [32, 63, 64])
def test_lattice_order_is_not_clustered(pkg, side):
    """Particles in the site order of a lattice (the usual start of a
    simulation), whose rows the sample's runs of side^3 / 4096 particles
    divide or nearly divide: uniform, so cells of side rcut at 3.4 particles
    per cell of side rcut / 2."""
    s = lattice(side, float(side), seed=4)
    solver = pkg.Solver(0, pkg.HostSystem.from_dict(s), pkg.parameters(16, 3, 1.0, 3.0))
    DeviceRealteil(solver, s, 3.0, 1.0).run()
    assert cells_of(pkg, solver)[1] == 1
    solver.close()


@pytest.mark.parametrize("per_cell,clustering,reach", [(6, 1.0, 1), (8, 1.0, 2), (11, 1.0, 2), (2, 3.0, 1),
                                                       (2, 4.0, 2), (0.5, 100.0, 2), (0.5, 1.0, 1)])
def test_cell_size_rule(pkg, per_cell, clustering, reach):
    """Cells of side rcut / 2 from 7 particles in a typical particle's cell
    on; clustering 1 is what the batch assumes."""
    L, rcut = 30.3, 3.0  # 20 cells of side rcut / 2, 10 of side rcut
    n = int(per_cell * 8000)
    lib = pkg.lib()
    lib.p3mk_cells_create.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_int] + [ctypes.c_double] * 3
    lib.p3mk_cells_geometry.restype = None
    lib.p3mk_cells_geometry.argtypes = [ctypes.c_void_p, ctypes.POINTER(ctypes.c_int), ctypes.POINTER(ctypes.c_int)]
    lib.p3mk_cells_destroy.restype, lib.p3mk_cells_destroy.argtypes = None, [ctypes.c_void_p]
    cells, nc, got = ctypes.c_void_p(), ctypes.c_int(), ctypes.c_int()
    assert lib.p3mk_cells_create(ctypes.byref(cells), n, L, rcut, clustering) == 0
    lib.p3mk_cells_geometry(cells, ctypes.byref(nc), ctypes.byref(got))
    lib.p3mk_cells_destroy(cells)
    assert (nc.value, got.value) == ((10, 1) if reach == 1 else (20, 2))
    if clustering == 1.0:
        assert cell_geometry(n, L, rcut) == (nc.value, got.value)


def test_cell_size_follows_changed_positions(pkg, orc):
    """A system that clusters and spreads out again: the list's cell size is
    the new positions' within 2 x 64 calls, and the forces are the oracle's
    before, at and after the change."""
    rcut, alpha = 3.0, 1.0
    spread = lattice(14, 27.0, seed=6)
    tight = dict(spread)
    for k in "xyz":
        tight[k] = np.mod(spread[k] * 0.25 - 2.0, 27.0)  # spacing 0.48, across the box corner
    ref = {id(s): orc.realteil(s, rcut, alpha, cells=True)[0] for s in (spread, tight)}
    solver = pkg.Solver(0, pkg.HostSystem.from_dict(spread), pkg.parameters(16, 3, alpha, rcut))
    dev = DeviceRealteil(solver, spread, rcut, alpha)
    for s, before, after in ((spread, 1, 1), (tight, 1, 2), (spread, 2, 1)):
        dev.put(s)
        assert rel_err(dev.run()[0], ref[id(s)]) < 1e-13
        assert cells_of(pkg, solver)[1] == before
        dev.run(130)
        dev.run(2)
        assert cells_of(pkg, solver)[1] == after
        assert rel_err(dev.run()[0], ref[id(s)]) < 1e-13
    solver.close()
