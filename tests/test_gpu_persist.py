"""The Krylov loops that run in one kernel on small lattices (mh_persist.hip):
every shape of the dispatch (lanes per site, threads per workgroup) at ragged
sizes and at the edges of its range, on both parities.

The FP64 CG is compared with the oracle's CG on the same links where that is
quick: iteration counts within one, solutions within the residual times the
condition number of the operator, 1 / (4 m^2) (times 10); everywhere its true
residual, which other kernels compute, has to meet the target.  A mixed solve
on a lattice above the one-kernel range of the mixed CG still goes through the
sloppy iterations."""
import ctypes

import numpy as np
import pytest

import ks_oracle as ko
import milc_qcd_amd as mq

pytestmark = pytest.mark.gpu

# Vh = 128, 648, 4096 | 6000, 8192 | 13824, 16384 | 21168, 65536 | 68040, 131072
SIZES = [(4, 4, 4, 4), (6, 6, 6, 6), (8, 8, 8, 16), (10, 10, 10, 12), (8, 8, 16, 16), (12, 12, 12, 16),
         (16, 8, 16, 16), (18, 6, 14, 28), (16, 16, 16, 32), (18, 18, 14, 30), (16, 16, 32, 32)]


@pytest.mark.parametrize("dims", SIZES)
@pytest.mark.parametrize("parity", [mq.EVEN, mq.ODD])
def test_cg_one_kernel(dims, parity):
    mass, resid = 0.1, 1e-10
    print(f"one-kernel CG {dims} parity {parity}", flush=True)
    with mq.Lattice(dims) as G:
        G.dev_gauge_hisq(1400)
        G.dev_source(1401, parity, 0)
        it, st = G.dev_invert(0, 1, mass, parity, resid, 0)
        assert st["converged"] and st["resid"] < resid
        # the same solve again, bit for bit
        G.dev_invert(0, 2, mass, parity, resid, 0)
        assert G.dev_diff(1, 2) == 0.0
        itm, stm = G.dev_invert(0, 3, mass, parity, resid, 2)
        assert stm["converged"] and stm["resid"] < resid
        if G.V > 30000:
            return
        fat, lng = G.dev_read_links()
        src, x = G.dev_read(0, parity), G.dev_read(1, parity)
        L = ko.Lattice(dims)
        ref, it_ref, _ = L.congrad(fat, lng, src, mass, resid, parity=parity, max_iters=20000)
        s = L.parity_slice(parity)
        assert abs(it - it_ref) <= 1
        assert np.linalg.norm(x[s] - ref[s]) < 10 * resid / (4 * mass ** 2) * np.linalg.norm(ref[s])


def test_mixed_cg_above_the_one_kernel_range():
    dims = (16, 16, 16, 32)  # Vh = 65536
    with mq.Lattice(dims) as G:
        G.dev_gauge_hisq(1402)
        G.dev_source(1403, mq.EVEN, 0)
        _, ref = G.dev_invert(0, 1, 0.05, mq.EVEN, 1e-11, 0)
        for mixed in (1, 2):
            _, st = G.dev_invert(0, 2, 0.05, mq.EVEN, 1e-10, mixed)
            assert st["converged"] and st["resid"] < 1e-10
            assert G.dev_diff(2, 1) < 10 * 1e-10 / (4 * 0.05 ** 2)


OFFSETS = [4 * 0.05 ** 2 + 1e-4 * 10 ** (4 * i / 11) for i in range(12)]


# 206, 524 and 512 blocks of 256 sites in the update kernel: remainders over the
# 8 XCDs with a last block of 8 and of 248 sites; an even split
@pytest.mark.parametrize("dims", [(18, 18, 18, 18), (18, 18, 18, 46), (16, 16, 32, 32)])
def test_update_kernel_block_order(dims):
    """A block order that missed or repeated sites would leave the true residual,
    which other kernels compute, above the target.  Two solutions lie within
    the sum of their residuals times the condition number 1 / (4 m^2) (times 10)."""
    mass, resid = 0.05, 1e-9
    print(f"update kernel {dims}", flush=True)
    with mq.Lattice(dims) as G:
        G.dev_gauge_hisq(1404)
        G.dev_source(1405, mq.EVEN, 0)
        G.dev_invert(0, 1, mass, mq.EVEN, resid, 0)
        for mixed in (1, 2):
            _, st = G.dev_invert(0, 2, mass, mq.EVEN, resid, mixed)
            assert st["converged"] and st["resid"] < resid
            assert G.dev_diff(2, 1) < 10 * 2 * resid / (4 * mass ** 2)


@pytest.mark.parametrize("dims", SIZES)
@pytest.mark.parametrize("mixed", [0, 1])
def test_multishift_one_kernel(dims, mixed):
    """Three and twelve shifts against single-mass solves to a hundredth of the
    target; a repeat is bit-identical."""
    resid = 1e-9
    print(f"one-kernel multi-shift {dims} mixed {mixed}", flush=True)
    with mq.Lattice(dims) as G:
        G.dev_gauge_hisq(1404)
        G.dev_source(1405, mq.EVEN, 0)
        for offs in (OFFSETS[5:2:-1], OFFSETS):
            n = len(offs)
            _, _, conv = G.dev_multishift(0, offs, resid, mixed, out_slot0=1)
            assert conv
            G.dev_multishift(0, offs, resid, mixed, out_slot0=20)
            for j in (0, 1, n - 1):
                assert G.dev_diff(1 + j, 20 + j) == 0.0
                G.dev_invert(0, 40, 0.5 * offs[j] ** 0.5, mq.EVEN, resid / 100, 0)
                assert G.dev_diff(1 + j, 40) < 10 * resid / offs[j]


@pytest.mark.parametrize("n", [1, 2, 31, 32])
def test_multishift_one_kernel_shift_counts_and_retirement(n, small_form):
    """In one kernel and launch by launch: shift counts at the ends of the table, the smallest offset last or first,
    heavy shifts whose zeta underflows (retired), and iteration caps inside and
    at the edge of a window, against the oracle's multi-shift CG."""
    dims = (6, 4, 8, 6)
    L = ko.Lattice(dims)
    U = L.rephase(L.gauge_random(1406))
    fat, lng, _ = L.hisq_links(U)
    src = L.gaussian_vector(1407, ko.EVEN)
    offs = [0.04 * 1.9 ** (j if n % 2 else n - 1 - j) for j in range(n)]
    s = L.parity_slice(ko.EVEN)
    with mq.Lattice(dims) as G:
        G.set_small_lattice_form(small_form)
        G.set_links(fat, lng)
        for cap in (3000, 2, 9, 10):
            ref, it_ref, _ = L.multicg_offset(fat, lng, src, offs, 1e-10, max_iters=cap, nrestart=1)
            ksp = [mq.KsParam(offset=o) for o in offs]
            qic = [mq.QuarkInvertControl(max=cap, nrestart=1, resid=1e-10) for _ in offs]
            x = G.ks_multicg_offset_field(src, ksp, qic, mixed=0)
            assert qic[0].final_iters == it_ref
            for a, b in zip(x, ref):
                assert np.linalg.norm(a[s] - b[s]) < 1e-9 * max(np.linalg.norm(b[s]), 1e-300)


@pytest.mark.parametrize("dims,nsrc", [((6, 4, 8, 6), 1), ((6, 4, 8, 6), 4), ((6, 4, 8, 6), 5), ((6, 4, 8, 6), 6),
                                       ((6, 4, 8, 6), 7), ((8, 8, 16, 16), 4), ((8, 8, 16, 16), 5), ((8, 8, 16, 16), 6),
                                       ((12, 12, 12, 16), 3), ((12, 12, 12, 16), 4), ((12, 12, 12, 16), 5),
                                       ((12, 12, 12, 16), 6), ((6, 4, 8, 6), 9), ((6, 4, 8, 6), 12),
                                       ((12, 12, 12, 24), 2), ((12, 12, 12, 24), 3), ((16, 16, 16, 24), 2)])
def test_block_calls_on_both_sides_of_the_dispatch(dims, nsrc):
    """Block CG (with an initial guess) and block multi-shift of one and three
    shifts, just where the sources are solved one after another and just where
    they go as a batch: true residuals and single-source solutions."""
    resid, mass = 1e-9, 0.1
    print(f"block calls {dims} x {nsrc}", flush=True)
    with mq.Lattice(dims) as G:
        G.dev_gauge_hisq(1410)
        fat, lng = G.dev_read_links()
        E = G.parity_slice(mq.EVEN)
        srcs = []
        for s in range(nsrc):
            G.dev_source(1411 + s, mq.EVEN, s)
            srcs.append(G.dev_read(s, mq.EVEN))
        G.set_links(fat, lng)
        qic = mq.QuarkInvertControl(max=3000, nrestart=1, parity=mq.EVEN, resid=resid)
        dests = [0.3 * v for v in srcs]
        _, res = G.ks_congrad_block_parity(srcs, dests, qic, mass)
        assert max(res) < resid
        for offs in ([4 * mass ** 2], [4 * mass ** 2, 0.3, 2.0]):
            st = G.dev_multishift_block(list(range(nsrc)), offs, 1e-7, resid, out_slot0=20)
            assert st["converged"] and max(st["true_rel"]) < resid
            for s in range(nsrc):
                for j, o in enumerate(offs):
                    G.dev_invert(s, 63, 0.5 * o ** 0.5, mq.EVEN, resid / 100, 0)
                    x = 20 + s * len(offs) + j
                    assert G.dev_diff(x, 63) < 10 * resid / o
                    if j == 0:
                        ref = G.dev_read(63, mq.EVEN)
                        assert np.linalg.norm(dests[s][E] - ref[E]) < 10 * resid / o * np.linalg.norm(ref[E])


@pytest.mark.parametrize("nsrc", [2, 7])
def test_block_multishift_slots_may_overlap(nsrc):
    """Solutions over slots of the sources, one source after another (2) and as
    a batch (7): every source is read before a solution is written, so the
    solutions are bit for bit those of separate slots."""
    offs = [0.04, 0.3]
    with mq.Lattice((6, 4, 8, 6)) as G:
        G.dev_gauge_hisq(1420)
        for first in (0, 1):  # solutions from slot `first` on
            for s in range(nsrc):
                G.dev_source(1421 + s, mq.EVEN, s)
            src = list(range(nsrc))
            G.dev_multishift_block(src, offs, 1e-7, 1e-9, out_slot0=40)
            G.dev_multishift_block(src, offs, 1e-7, 1e-9, out_slot0=first)
            for k in range(nsrc * len(offs)):
                assert G.dev_diff(first + k, 40 + k) == 0.0, (first, k)


@pytest.mark.parametrize("nsrc", [2, 7])
def test_block_calls_on_aliased_host_arrays(nsrc):
    """The same for host arrays: solution s in the array of source s + 1 (which is
    then also the CG's initial guess)."""
    dims, mass = (6, 4, 8, 6), 0.1
    offs = [4 * mass ** 2, 0.3]
    with mq.Lattice(dims) as G:
        G.dev_gauge_hisq(1430)
        G.set_links(*G.dev_read_links())
        srcs = []
        for s in range(nsrc):
            G.dev_source(1431 + s, mq.EVEN, 0)
            srcs.append(G.dev_read(0, mq.EVEN))
        qic = mq.QuarkInvertControl(max=3000, nrestart=1, parity=mq.EVEN, resid=1e-9)
        ref = [srcs[(s + 1) % nsrc].copy() for s in range(nsrc)]
        G.ks_congrad_block_parity([v.copy() for v in srcs], ref, qic, mass)
        a = [v.copy() for v in srcs]
        G.ks_congrad_block_parity(a, [a[(s + 1) % nsrc] for s in range(nsrc)], qic, mass)
        for s in range(nsrc):
            assert np.array_equal(a[(s + 1) % nsrc], ref[s]), s

        ref = G.ks_multicg_offset_block(srcs, offs, mq.EVEN, 1e-7, 1e-9)[0]
        a = [v.copy() for v in srcs]
        x = [[a[(s + 1) % nsrc], np.zeros_like(a[0])] for s in range(nsrc)]
        ptr = lambda fields: (ctypes.c_void_p * len(fields))(*[f.ctypes.data for f in fields])
        rc = G.lib.milc_hip_multishift_invert_block(
            2, nsrc, 2, (ctypes.c_double * 2)(*offs), mq.ks.InvArgs(3000, 0, 1, 0.0, 1.0, 0), (ctypes.c_double * 1)(1e-7),
            1e-9, G.fat.ctypes.data, G.lng.ctypes.data, ptr(a), ptr([f for xs in x for f in xs]),
            (ctypes.c_double * (2 * nsrc))(), ctypes.byref(ctypes.c_int(0)))
        assert rc > 0
        E = G.parity_slice(mq.EVEN)
        for s in range(nsrc):
            for j in range(2):
                assert np.array_equal(x[s][j][E], ref[s][j][E]), (s, j)


@pytest.mark.parametrize("nsrc", [2, 7])
def test_block_calls_without_a_target_run_to_the_cap(nsrc):
    """A target whose square is zero is never met: max_iter iterations and no
    convergence, on either side of the dispatch."""
    with mq.Lattice((6, 4, 8, 6)) as G:
        G.dev_gauge_hisq(1440)
        G.set_links(*G.dev_read_links())
        for s in range(nsrc):
            G.dev_source(1441 + s, mq.EVEN, s)
        src = G.dev_read(0, mq.EVEN)
        for resid in (0.0, 1e-170):
            qic = mq.QuarkInvertControl(max=24, nrestart=1, parity=mq.EVEN, resid=resid)
            dests = [np.zeros_like(src) for _ in range(nsrc)]
            it, res = G.ks_congrad_block_parity([src] * nsrc, dests, qic, 0.1)
            assert 24 <= it <= 25 and qic.converged == 0
            assert 0 < max(res) < 1e-2
        st = G.dev_multishift_block(list(range(nsrc)), [0.04, 0.5], 1e-6, 1e-170, max_iters=60, out_slot0=20)
        assert st["converged"] == 0 and 0 < max(st["true_rel"]) < 1e-9
        if nsrc == 2:
            _, _, conv = G.dev_multishift(0, [0.04, 0.5], 1e-170, 1, out_slot0=20)
            assert not conv
            G.dev_invert(0, 30, 0.1, mq.EVEN, 1e-12, 0)
            assert G.dev_diff(20, 30) < 1e-9


@pytest.mark.parametrize("nsrc", [2, 7])
def test_block_multishift_takes_an_offset_of_zero(nsrc):
    """(-D D) x = b, offset 0, is a positive system too: accepted on either side
    of the dispatch."""
    with mq.Lattice((4, 4, 4, 4)) as G:
        G.dev_gauge_hisq(1450)
        for s in range(nsrc):
            G.dev_source(1451 + s, mq.EVEN, s)
        st = G.dev_multishift_block(list(range(nsrc)), [0.0, 0.5], 1e-6, 1e-9, out_slot0=20)
        assert st["converged"] and max(st["true_rel"]) < 1e-9


@pytest.mark.parametrize("nsrc", [2, 7])
def test_block_multishift_counts_stage_and_refinement(nsrc):
    """On either side of the dispatch the device call counts the multi-shift's
    iterations and those of each shift's refinement apart and the host call
    returns their sum.  A target below what FP64 reaches (about 4e-16 |b|) needs
    refinement, up to the cap."""
    offs, cap = [0.04, 0.5], 200
    with mq.Lattice((6, 4, 8, 6)) as G:
        G.dev_gauge_hisq(1460)
        for s in range(nsrc):
            G.dev_source(1461 + s, mq.EVEN, s)
        st = G.dev_multishift_block(list(range(nsrc)), offs, 1e-6, 1e-16, max_iters=cap)
        print(st)
        assert st["converged"] == 0 and max(st["true_rel"]) < 1e-14
        assert st["iters"] == st["ms_iters"] < cap
        assert all(cap <= it <= cap + 1 for it in st["refine_iters"])
        fat, lng = G.dev_read_links()
        srcs = [G.dev_read(s, mq.EVEN) for s in range(nsrc)]
        G.set_links(fat, lng)
        _, _, it = G.ks_multicg_offset_block(srcs, offs, mq.EVEN, 1e-6, 1e-16, max_iter=cap)
        assert it == st["ms_iters"] + sum(st["refine_iters"])


@pytest.mark.parametrize("dims", [(4, 4, 4, 4), (10, 10, 10, 12), (18, 6, 14, 28), (16, 16, 16, 32)])
def test_given_up_solves_go_on_launch_by_launch(dims):
    """A one-kernel solve that gives up waiting (form 2: at the first poll) is
    finished by the loops of larger lattices (form 0), with the restarts and
    iterations of those: bit for bit the same solutions and counts."""
    print(f"given up {dims}", flush=True)
    offs = OFFSETS[::4]
    out = []
    with mq.Lattice(dims) as G:
        G.dev_gauge_hisq(1470)
        G.dev_source(1471, mq.EVEN, 0)
        for k, form in enumerate((0, 2)):
            G.set_small_lattice_form(form)
            it, st = G.dev_invert(0, 1 + k, 0.1, mq.EVEN, 1e-10, 0)
            itc, stc = G.dev_invert(0, 3 + k, 0.1, mq.EVEN, 1e-10, 0, max_iter=7)
            itm, _, conv = G.dev_multishift(0, offs, 1e-9, 0, out_slot0=10 + 4 * k)
            assert st["converged"] and conv and st["resid"] < 1e-10
            out.append((it, st["reliable_updates"], itc, stc["converged"], itm))
        assert out[0] == out[1]
        for a in (1, 3):
            assert G.dev_diff(a, a + 1) == 0.0
        for j in range(len(offs)):
            assert G.dev_diff(10 + j, 14 + j) == 0.0
        # where the small lattice's form is chosen for a mixed solve
        it, st = G.dev_invert(0, 3, 0.1, mq.EVEN, 1e-10, 2)
        assert st["converged"] and st["resid"] < 1e-10
        itm, _, conv = G.dev_multishift(0, offs, 1e-9, 1, out_slot0=20)
        assert conv
        for j in range(len(offs)):
            assert G.dev_diff(20 + j, 10 + j) < 10 * 2e-9 / offs[j]


def test_small_lattice_form_is_checked_and_belongs_to_the_context():
    """Values other than 0, 1 and 2 are refused, and a new context starts with 1:
    a single source's block multi-shift has no stencil variant (-1) there."""
    dims, variant = (4, 4, 4, 4), []
    for form in (0, None):
        with mq.Lattice(dims) as G:
            assert G.lib.milc_hip_set_small_lattice_form(3) == -2
            assert G.lib.milc_hip_set_small_lattice_form(-1) == -2
            if form is not None:
                G.set_small_lattice_form(form)
            G.dev_gauge_hisq(1480)
            G.dev_source(1481, mq.EVEN, 0)
            st = G.dev_multishift_block([0], [0.1, 0.5], 1e-6, 1e-9)
            assert st["converged"]
            variant.append(st["variant"])
    assert variant[0] >= 0 and variant[1] == -1
