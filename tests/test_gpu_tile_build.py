"""The device tile builder at the sizes where it branches: tiles of one to
128 particles with a ragged last one, rows longer than the 256 entries that
are put in order, partners spread over the whole system (the hashed set) or
in a few runs of slots (the paged one), rows of very different lengths, open
and periodic boxes. The tiles must equal the host model's (ljgpu_make_tiles_*)
and the forces over them, whose entry order is the slices' own, the oracle's.
"""
import ctypes
import functools

import numpy as np
import pytest

import lj_gpu_amd as G
import oracle as O
from helpers import FP64_TOL, normwise

MIXED_TOL = 2.0e-6  # normwise, FP32 force scalars with FP64 sums

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    if G.device_count() < 1:
        pytest.skip("no HIP device")
    c = G.Context(0)
    yield c
    c.close()


@functools.lru_cache(maxsize=None)
def system(name):
    """(q, box, full list, oracle force)."""
    rng = np.random.default_rng(5)
    if name == "ragged":        # vacancies, shuffled: N = 859
        q, box = G.lattice_periodic(6, 1.0, 3)
        q = q[rng.permutation(q.shape[0])[:-5]]
    elif name == "long_rows":   # about 300 partners: rows past the order's limit
        q, box = G.lattice_periodic(6, 2.0, 3)
    elif name == "mixed_rows":  # rows of about 140 to 310 entries in one box
        q, box = G.lattice_periodic(8, 2.0, 3)
        keep = (q[:, 0] < 0.5 * box) | (rng.random(q.shape[0]) < 0.4)
        q = q[keep]
    elif name == "scattered":   # open box in a shuffled index order
        q, box = G.lattice_reference(1.0, 22.0), 0.0
        q = q[rng.permutation(q.shape[0])]
    else:                       # open box in lattice order
        assert name == "open"
        q, box = G.lattice_reference(0.5, 22.0), 0.0
    q = np.ascontiguousarray(q)
    full = G.makepair(q, box, G.LIST_FULL)
    f = np.zeros_like(q)
    O.force_aos(O.CSR(full.number_of_partners, full.pointer, full.sorted_list, "full"), q, f, 1.0,
                O.CL2, box, steps=1, method="full")
    return q, box, full, f


@pytest.mark.parametrize("name", ["ragged", "long_rows", "mixed_rows", "scattered", "open"])
@pytest.mark.parametrize("lanes,unroll,tile", [(4, 4, 64), (4, 2, 48), (4, 4, 1), (2, 1, 128),
                                               (8, 2, 32), (64, 1, 16)])
def test_built_tiles_and_their_forces(ctx, name, lanes, unroll, tile):
    q, box, full, f = system(name)
    print(f"{name} lanes={lanes} unroll={unroll} tile={tile}", flush=True)
    ctx.set_kernel_config(lanes, 256, unroll)
    ctx.set_tiling(tile)
    ctx.set_half_mode(G.HALF_AUTO)
    dq, dp = ctx.array(q), ctx.zeros(q.shape)
    ctx.build_list(dq, q.shape[0], box, G.LIST_FULL)
    for steps in (1, 20):
        dp.zero()
        ctx.force_aos_f64(dq, dp, 1.0 / steps, G.CL2, box, steps)
        ctx.sync()
        assert normwise(dp.download(), f) < FP64_TOL
    t = ctx.get_tiles()
    used = ctx.list_info().tile_particles
    order, member = ctx.get_tile_order()
    assert order == (G.TILE_ORDER_SPATIAL if box > 0 else G.TILE_ORDER_INDEX)
    h = G.make_tiles(full, used, member=member, q=q, box=box, cl2=G.CL2)
    if np.all(h.desc[:-1, 1] == used):
        np.testing.assert_array_equal(t.desc, h.desc)
        np.testing.assert_array_equal(t.stage, h.stage)
        np.testing.assert_array_equal(t.local, h.local)
    # Inspection left the evaluated layout as it was.
    dp.zero()
    ctx.force_aos_f64(dq, dp, 1.0, G.CL2, box, 1)
    ctx.sync()
    assert normwise(dp.download(), f) < FP64_TOL


@pytest.mark.parametrize("name", ["ragged", "long_rows", "mixed_rows", "scattered", "open"])
@pytest.mark.parametrize("layout", ["aos", "soa", "aos3"])
@pytest.mark.parametrize("tile", [64, 16, 1])
def test_atomic_half_lists_over_tiles(ctx, name, layout, tile):
    """Half lists scattered to both particles: over tiles where partners are
    shared (LDS sums, one addition to memory per staged partner), else the
    untiled kernel; reported as untiled either way."""
    q, box, full, f = system(name)
    n = q.shape[0]
    print(f"{name} {layout} tile={tile}", flush=True)
    ctx.set_kernel_config(4, 256, 4)
    ctx.set_tiling(tile)
    ctx.set_half_mode(G.HALF_ATOMIC)
    if layout == "soa":
        dq = [ctx.array(np.ascontiguousarray(q[:, c])) for c in range(3)]
        dp = [ctx.zeros(n) for _ in range(3)]
        build, force = ctx.build_list_soa, ctx.force_soa_f64
    else:
        w = 4 if layout == "aos" else 3
        dq, dp = ctx.array(np.ascontiguousarray(q[:, :w])), ctx.zeros((n, w))
        build = ctx.build_list if w == 4 else ctx.build_list_aos3
        force = ctx.force_aos_f64 if w == 4 else ctx.force_aos3_f64
    build(dq, n, box, G.LIST_HALF)
    for steps in (1, 5, 20):
        for a in dp if layout == "soa" else [dp]:
            a.zero()
        force(dq, dp, 1.0 / steps, G.CL2, box, steps)
        ctx.sync()
        p = np.stack([a.download() for a in dp], 1) if layout == "soa" else dp.download()
        assert normwise(p, f) < FP64_TOL
    assert ctx.list_info().tile_particles == 0 and ctx.get_tiles() is None
    ctx.set_half_mode(G.HALF_AUTO)


@pytest.mark.parametrize("tile,resident", [(64, 0), (4, 0), (1, 1)])
@pytest.mark.parametrize("graphs", [True, False])
def test_launches_of_several_evaluations(ctx, tile, resident, graphs):
    """A launch over tiles carries several evaluations of a call (in one chain
    for 14 tiles, two for 215 or 859, a persistent grid of fewer workgroups than
    tiles included): bit for bit what as many calls of one give."""
    q, box, full, _ = system("ragged")
    n = q.shape[0]
    print(f"tile={tile} resident={resident} graphs={graphs}", flush=True)
    ctx.set_kernel_config(4, 256, 4)
    ctx.set_tiling(tile, resident_per_cu=resident)
    ctx.set_half_mode(G.HALF_AUTO)
    ctx.set_graphs(graphs)
    dq, da, db = ctx.array(q), ctx.zeros(q.shape), ctx.zeros(q.shape)
    ctx.build_list(dq, n, box, G.LIST_FULL)
    for steps in (2, 3, 5, 10, 17, 300):
        da.zero()
        db.zero()
        ctx.force_aos_f64(dq, da, 1e-3, G.CL2, box, steps)
        for _ in range(steps):
            ctx.force_aos_f64(dq, db, 1e-3, G.CL2, box, 1)
        ctx.sync()
        np.testing.assert_array_equal(da.download(), db.download())
    ctx.set_graphs(True)
    ctx.set_tiling(64)


@pytest.mark.parametrize("cells", [22, 24])
@pytest.mark.parametrize("soa", [False, True])
def test_many_rounds_of_tiles(ctx, cells, soa):
    """Systems of more than four rounds of tiles (55,296 particles in tiles of
    4: 13,824 tiles) take slot-order copies from ten evaluations on and more
    of them per launch than smaller ones (42,592): bit for bit what as many
    calls of one give."""
    q, box = G.lattice_periodic(cells, 0.5, 3)
    n = q.shape[0]
    print(f"cells={cells} soa={soa}", flush=True)
    ctx.set_kernel_config(4, 256, 4)
    ctx.set_tiling(4)
    ctx.set_half_mode(G.HALF_AUTO)
    if soa:
        dq = [ctx.array(np.ascontiguousarray(q[:, c])) for c in range(3)]
        da, db = ([ctx.zeros(n) for _ in range(3)] for _ in range(2))
        build, force = ctx.build_list_soa, ctx.force_soa_f64
    else:
        dq, da, db = ctx.array(q), ctx.zeros(q.shape), ctx.zeros(q.shape)
        build, force = ctx.build_list, ctx.force_aos_f64
    build(dq, n, box, G.LIST_FULL)
    for steps in (9, 10, 11):
        force(dq, da, 1e-3, G.CL2, box, steps)
        for _ in range(steps):
            force(dq, db, 1e-3, G.CL2, box, 1)
    ctx.sync()
    for a, b in zip(da if soa else [da], db if soa else [db]):
        np.testing.assert_array_equal(a.download(), b.download())
    ctx.set_tiling(64)


@pytest.mark.parametrize("copies", [1, 7, 255, 256])
@pytest.mark.parametrize("others", [0, 1, 40])
def test_rows_that_repeat_a_partner(ctx, copies, others):
    """A caller's list may name a partner many times: up to all 256 entries of
    a row that is put in order are then in one class. The untiled kernel's
    momenta."""
    n = 400
    q, box = G.lattice_periodic(5, 0.8, 3)
    q = np.ascontiguousarray(q[:n])
    rows = [np.zeros(0, np.int32) for _ in range(n)]
    others = min(others, 256 - copies)
    for i in range(0, n, 3):
        rows[i] = np.concatenate([np.full(copies, (i + 1) % n, np.int32),
                                  np.array([(i + 2 + k) % n for k in range(others)], np.int32)])
    nop = np.array([len(r) for r in rows], np.int32)
    ptr = np.concatenate([[0], np.cumsum(nop)[:-1]]).astype(np.int32)
    csr = G.CSR(nop, ptr, np.concatenate(rows).astype(np.int32), G.LIST_FULL)
    print(f"copies={copies} others={others}", flush=True)
    ctx.set_kernel_config(4, 256, 4)
    ctx.set_half_mode(G.HALF_AUTO)
    out = []
    for tile in (64, 0):
        ctx.set_tiling(tile)
        ctx.set_list(csr)
        dq, dp = ctx.array(q), ctx.zeros(q.shape)
        ctx.force_aos_f64(dq, dp, 1e-3, G.CL2, box, 1)
        ctx.sync()
        out.append(dp.download())
    ctx.set_tiling(64)
    assert np.abs(out[1]).max() > 0
    assert normwise(out[0], out[1]) < FP64_TOL


@pytest.mark.parametrize("name", ["ragged", "long_rows", "open"])
@pytest.mark.parametrize("lanes,unroll", [(4, 4), (8, 2)])
def test_kahan_sums_have_slices_of_their_own(ctx, name, lanes, unroll):
    """Kahan sums run over rows in the bank-class order, made on first use,
    beside the other kernels' slices: neither changes the other's momenta."""
    q, box, full, _ = system(name)
    ctx.set_kernel_config(lanes, 256, unroll)
    ctx.set_tiling(64)
    ctx.set_half_mode(G.HALF_AUTO)
    dq = ctx.array(q)

    def momenta(accum):
        dp = ctx.zeros(q.shape)
        if accum is None:
            ctx.force_aos_f64(dq, dp, 1e-3, G.CL2, box, 3)
        else:
            ctx.force_aos_mixed(dq, dp, 1e-3, G.CL2, box, 3, accum)
        ctx.sync()
        return dp.download()

    out = []
    for order in ([None, G.ACCUM_KAHAN_F32, None, G.ACCUM_F64], [G.ACCUM_KAHAN_F32, None, None,
                                                                 G.ACCUM_F64]):
        ctx.build_list(dq, q.shape[0], box, G.LIST_FULL)
        got = [momenta(a) for a in order]
        out.append({a: g for a, g in zip(order, got)})
        f64 = [g for a, g in zip(order, got) if a is None]
        np.testing.assert_array_equal(f64[0], f64[1])
    for a in out[0]:
        np.testing.assert_array_equal(out[0][a], out[1][a])
    ctx.set_kernel_config(4, 256, 4)


def half_tile(ctx):
    """Particles per tile of the installed atomic half list; 0: untiled kernel."""
    query = G.lib().ljgpu_internal_half_tile
    query.argtypes = [ctypes.c_void_p, ctypes.POINTER(ctypes.c_int32)]
    t = ctypes.c_int32(-1)
    assert query(ctx.handle, ctypes.byref(t)) == G.OK
    return t.value


@pytest.mark.parametrize("name", ["ragged", "mixed_rows", "scattered", "open"])
@pytest.mark.parametrize("tile", [64, 16, 1])
def test_which_kernel_an_atomic_half_list_takes(ctx, name, tile):
    """Tiles where they stage at most half as many partners as the list has
    entries, the untiled kernel elsewhere (scattered particles, tiles of one);
    Kahan sums always take the untiled kernel's order of entries."""
    q, box, _, f = system(name)
    n = q.shape[0]
    ctx.set_kernel_config(4, 256, 4)
    ctx.set_half_mode(G.HALF_ATOMIC)
    dq, dp = ctx.array(q), ctx.zeros(q.shape)
    kahan = []
    for t in (tile, 0):
        ctx.set_tiling(t)
        ctx.build_list(dq, n, box, G.LIST_HALF)
        used = half_tile(ctx)
        print(f"{name} tile={t} used={used}", flush=True)
        assert used == (t if name != "scattered" and t > 1 else 0)
        for accum, tol in ((None, FP64_TOL), (G.ACCUM_F64, MIXED_TOL), (G.ACCUM_KAHAN_F32, None)):
            dp.zero()
            if accum is None:
                ctx.force_aos_f64(dq, dp, 1.0, G.CL2, box, 1)
            else:
                ctx.force_aos_mixed(dq, dp, 1.0, G.CL2, box, 1, accum)
            ctx.sync()
            if tol is None:
                kahan.append(dp.download())
            else:
                assert normwise(dp.download(), f) < tol
    # FP32 sums in another order differ by about 1e-7, the additions to memory by rounding.
    assert normwise(kahan[0], kahan[1]) < FP64_TOL
    ctx.set_tiling(64)
    ctx.set_half_mode(G.HALF_AUTO)


@pytest.mark.parametrize("buffer", [1, 2])
@pytest.mark.parametrize("device_list", [True, False])
def test_half_list_whose_tiles_find_no_room(buffer, device_list):
    """Where the tiles' force sums (or their staged particles) cannot be
    allocated, the list is installed all the same and takes the untiled kernel,
    call after call; after a smaller list that is tiled, too. With room again, a
    new list is tiled."""
    q, box, _, f = system("ragged")
    small, small_box = G.lattice_periodic(5, 0.5, 3)
    c = G.Context(0)
    try:
        limit = G.lib().ljgpu_internal_limit
        limit.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_size_t]
        c.set_half_mode(G.HALF_ATOMIC)
        half = G.makepair(q, box, G.LIST_HALF)
        dq, dp = c.array(q), c.zeros(q.shape)

        def install():
            if device_list:
                c.build_list(dq, q.shape[0], box, G.LIST_HALF)
            else:
                c.set_list(half)

        def check(tile):
            for steps in (1, 5, 20):
                dp.zero()
                c.force_aos_f64(dq, dp, 1.0 / steps, G.CL2, box, steps)
                c.sync()
                assert half_tile(c) == tile
                assert normwise(dp.download(), f) < FP64_TOL

        assert limit(c.handle, buffer, 64) == G.OK
        install()
        check(0)
        assert limit(c.handle, buffer, 2**64 - 1) == G.OK
        c.build_list(c.array(small), small.shape[0], small_box, G.LIST_HALF)
        assert half_tile(c) == 64
        assert limit(c.handle, buffer, 64) == G.OK
        install()
        check(0)
        assert limit(c.handle, buffer, 2**64 - 1) == G.OK
        install()
        check(64)
    finally:
        c.close()


def exact_force(q, box, half):
    """Force of every pair of a half list inside the cutoff in extended
    precision, and per particle sum(|24 s^4| + |48 s^7|) r, s = 1 / r^2."""
    i = np.repeat(np.arange(q.shape[0]), half.number_of_partners)
    j = half.sorted_list
    x = q[:, :3].astype(np.longdouble)
    d = x[j] - x[i]
    d -= np.longdouble(box) * np.rint(d / np.longdouble(box))
    r2 = (d * d).sum(1)
    i, j, d, r2 = (a[r2 <= G.CL2] for a in (i, j, d, r2))
    s = 1 / r2
    df = 24 * s ** 4 - 48 * s ** 7
    weight = (24 * s ** 4 + 48 * s ** 7) * np.sqrt(r2)
    f = np.zeros_like(x)
    scale = np.zeros(q.shape[0], np.longdouble)
    for c in range(3):
        np.add.at(f[:, c], i, df * d[:, c])
        np.add.at(f[:, c], j, -df * d[:, c])
    np.add.at(scale, i, weight)
    np.add.at(scale, j, weight)
    return f, scale


@pytest.mark.parametrize("corner", [0.0, 0.5])
@pytest.mark.parametrize("tile", [64, 16, 0])
def test_half_list_forces_lose_nothing_at_a_face(ctx, corner, tile):
    """A dense block of particles across the corner of a box 30 times its size
    (or in the middle of it): positions shifted into a tile's frame must not be
    rounded at the box's magnitude, which moves every pair by 256 u (u = 2^-53) and
    its force by 14 * 256 u / r. Rounded once each: differences u, r^2 4 u, its
    reciprocal 6 u, the seventh power and products 45 u; a row's additions 80 u."""
    q, side = G.lattice_periodic(6, 1.0, 3)
    box = 300.0
    # Positions on the grid of the largest ones: wrapping them is exact.
    x = np.rint((q[:, :3] - side / 2 + corner * box) * 2.0**44) / 2.0**44
    rng = np.random.default_rng(11)
    q = np.zeros_like(q)
    q[:, :3] = np.where(x < 0, x + box, x)
    # and, below that grid, bits of their own
    low = q[:, :3] < 16.0
    q[:, :3] += np.where(low, rng.uniform(0, 2.0**-45, low.shape), 0.0)
    half = G.makepair(q, box, G.LIST_HALF)
    f, scale = exact_force(q, box, half)
    ctx.set_kernel_config(4, 256, 4)
    ctx.set_tiling(tile)
    ctx.set_half_mode(G.HALF_ATOMIC)
    dq, dp = ctx.array(q), ctx.zeros(q.shape)
    ctx.build_list(dq, q.shape[0], box, G.LIST_HALF)
    assert half_tile(ctx) == tile
    ctx.force_aos_f64(dq, dp, 1.0, G.CL2, box, 1)
    ctx.sync()
    off = np.abs(dp.download()[:, :3] - f).max(1) / (scale * 2.0**-53)
    print(f"corner={corner} tile={tile} error {float(off.max()):.1f} u", flush=True)
    # The untiled kernel rounds differences across a face, up to the box's ulp / 2.
    assert off.max() < (125 if tile or corner else 125 + 14 * 256)
    ctx.set_tiling(64)
    ctx.set_half_mode(G.HALF_AUTO)


def momenta_of(c, q, box, kind, steps=1):
    dq, dp = c.array(q), c.zeros(q.shape)
    if kind == "f64":
        c.force_aos_f64(dq, dp, 1e-3, G.CL2, box, steps)
    else:
        accum = G.ACCUM_F64 if kind == "mixed" else G.ACCUM_KAHAN_F32
        c.force_aos_mixed(dq, dp, 1e-3, G.CL2, box, steps, accum)
    c.sync()
    return dp.download()


@pytest.mark.parametrize("before", ["kahan", "stage_offsets", "get_tiles"])
@pytest.mark.parametrize("lanes,unroll", [(8, 2), (4, 4), (64, 1)])
def test_rows_keep_their_order_whatever_ran_before(before, lanes, unroll):
    """Kahan sums, offsets staged in LDS and tile inspection take the rows in the
    bank-class order; the launches that follow over the same list, in another
    shape, give what they give in a context that did none of these."""
    q, box, _, _ = system("mixed_rows")
    out = []
    for disturbed in (False, True):
        c = G.Context(0)
        try:
            dq = c.array(q)
            c.build_list(dq, q.shape[0], box, G.LIST_FULL)
            if disturbed:
                if before == "kahan":
                    momenta_of(c, q, box, "kahan")
                elif before == "get_tiles":
                    c.get_tiles()
                else:
                    c.set_tiling(64, stage_offsets=True)
                    momenta_of(c, q, box, "f64")
                    c.set_tiling(64)
            c.set_kernel_config(lanes, 256, unroll)
            print(f"{before} lanes={lanes} disturbed={disturbed}", flush=True)
            got = [momenta_of(c, q, box, k) for k in ("f64", "mixed", "kahan", "f64")]
            got.append(c.get_tiles().local)
            out.append(got + [momenta_of(c, q, box, k) for k in ("kahan", "f64")])
        finally:
            c.close()
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
    np.testing.assert_array_equal(out[0][0], out[0][3])
    np.testing.assert_array_equal(out[0][2], out[0][5])


@pytest.mark.parametrize("installed", [False, True])
def test_force_calls_do_not_allocate(installed):
    """Once a list is built on the device (or, installed from the host, has had
    its first force call), force calls of any precision take no more device
    memory: what a list of 4.6 million entries needs for Kahan sums comes with
    the list."""
    info = G.lib().hipMemGetInfo  # of the HIP runtime that the library is linked with
    info.argtypes = [ctypes.POINTER(ctypes.c_size_t)] * 2

    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert info(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value

    q, box = G.lattice_periodic(20, 1.0, 3)
    full = G.makepair(q, box, G.LIST_FULL) if installed else None
    warm, c = G.Context(0), G.Context(0)
    try:
        for x in (warm, c):  # the first context loads the kernels
            dq, dp = x.array(q), x.zeros(q.shape)
            if installed:
                x.set_list(full)
                x.force_aos_f64(dq, dp, 1e-3, G.CL2, box, 1)
            else:
                x.build_list(dq, q.shape[0], box, G.LIST_FULL)
            x.sync()
            was = free()
            for steps in (1, 3, 20):
                x.force_aos_f64(dq, dp, 1e-3, G.CL2, box, steps)
                x.force_aos_mixed(dq, dp, 1e-3, G.CL2, box, steps, G.ACCUM_F64)
                x.force_aos_mixed(dq, dp, 1e-3, G.CL2, box, steps, G.ACCUM_KAHAN_F32)
            x.sync()
            taken = was - free()
            print(f"installed={installed} taken {taken}", flush=True)
        assert taken == 0
    finally:
        warm.close()
        c.close()


@pytest.mark.parametrize("lanes,tile,used", [(2, 512, 256), (2, 257, 256), (2, 256, 256),
                                             (4, 1000, 256)])
@pytest.mark.parametrize("installed", [False, True])
def test_half_lists_in_tiles_of_more_rows_than_their_kernel_takes(ctx, lanes, tile, used, installed):
    """The half-list kernel has four lanes a row, whatever the configured
    number: tiles of more than 256 rows become tiles of 256 where those fit (a
    gas; dense tiles are halved until they do)."""
    q, box = G.lattice_periodic(6, 0.1, 2)
    half = G.makepair(q, box, G.LIST_HALF)
    f, _ = exact_force(q, box, half)
    ctx.set_kernel_config(lanes, 256, 4)
    ctx.set_tiling(tile)
    ctx.set_half_mode(G.HALF_ATOMIC)
    dq, dp = ctx.array(q), ctx.zeros(q.shape)
    if installed:
        ctx.set_list(half)
    else:
        ctx.build_list(dq, q.shape[0], box, G.LIST_HALF)
    for steps in (1, 20):
        dp.zero()
        ctx.force_aos_f64(dq, dp, 1.0 / steps, G.CL2, box, steps)
        ctx.sync()
        assert half_tile(ctx) == used
        assert normwise(dp.download(), f.astype(float)) < FP64_TOL
    ctx.set_kernel_config(4, 256, 4)
    ctx.set_tiling(64)
    ctx.set_half_mode(G.HALF_AUTO)


@pytest.mark.parametrize("tiles,tiled", [(0, True), (25, True), (150, False)])
def test_half_lists_with_some_scattered_tiles(ctx, tiles, tiled):
    """Of the 500 tiles of an open lattice in its own order, some hold
    particles from all over it: up to an eighth of them the list is tiled (their
    sets hashed), beyond it takes the untiled kernel."""
    q = G.lattice_reference(0.5, 40.0)
    n = q.shape[0]
    rng = np.random.default_rng(2)
    at = np.arange(64 * tiles)
    to = rng.choice(np.arange(64 * tiles, n), at.size, replace=False)
    order = np.arange(n)
    order[at], order[to] = to, at
    q = np.ascontiguousarray(q[order])
    half = G.makepair(q, 0.0, G.LIST_HALF)
    f, _ = exact_force(q, 1e9, half)
    ctx.set_kernel_config(4, 256, 4)
    ctx.set_tiling(64)
    ctx.set_half_mode(G.HALF_ATOMIC)
    dq, dp = ctx.array(q), ctx.zeros(q.shape)
    ctx.build_list(dq, n, 0.0, G.LIST_HALF)
    used = half_tile(ctx)
    print(f"n={n} scattered tiles={tiles}: tile {used}", flush=True)
    assert (used > 0) == tiled and (tiles > 0 or used == 64)
    for steps in (1, 20):
        dp.zero()
        ctx.force_aos_f64(dq, dp, 1.0 / steps, G.CL2, 0.0, steps)
        ctx.sync()
        assert normwise(dp.download(), f.astype(float)) < FP64_TOL
    ctx.set_half_mode(G.HALF_AUTO)


@functools.lru_cache(maxsize=None)
def scattered_system():
    """27,436 particles of an open box in a shuffled order, and the first one's
    row over all 215 pages of slots: sets of every tile size are hashed."""
    q = G.lattice_reference(0.5, 38.0)
    n = q.shape[0]
    q = np.ascontiguousarray(q[np.random.default_rng(7).permutation(n)])
    full = G.makepair(q, 0.0, G.LIST_FULL)
    row = np.arange(1, n, n // 250).astype(np.int32)
    lst = np.concatenate([row, full.sorted_list[full.number_of_partners[0]:]]).astype(np.int32)
    nop = full.number_of_partners.copy()
    nop[0] = row.size
    ptr = np.concatenate([[0], np.cumsum(nop)[:-1]]).astype(np.int32)
    return q, G.CSR(nop, ptr, lst, G.LIST_FULL)


@pytest.mark.parametrize("tile,used", [(64, 32), (16, 16), (5, 5), (4, 4), (3, 3), (2, 2), (1, 1)])
def test_tiles_of_scattered_partners(ctx, tile, used):
    """Hashed sets of 20 words (ranked against each other) to 1,300 (sorted), on
    both sides of the change at 192: the host model's tiles, the untiled kernel's
    forces. Tiles of 64 have too many words and become 32."""
    q, csr = scattered_system()
    ctx.set_kernel_config(4, 256, 4)
    ctx.set_half_mode(G.HALF_AUTO)
    dq, p = ctx.array(q), []
    for t in (0, tile):
        ctx.set_tiling(t)
        ctx.set_list(csr)
        dp = ctx.zeros(q.shape)
        ctx.force_aos_f64(dq, dp, 1.0, G.CL2, 0.0, 1)
        ctx.sync()
        p.append(dp.download())
    print(f"tile={tile} used={ctx.list_info().tile_particles} "
          f"staged {ctx.list_info().tile_max_stage}", flush=True)
    assert ctx.list_info().tile_particles == used
    assert normwise(p[1], p[0]) < FP64_TOL
    t, h = ctx.get_tiles(), G.make_tiles(csr, used, q=q, box=0.0, cl2=G.CL2)
    np.testing.assert_array_equal(t.desc, h.desc)
    np.testing.assert_array_equal(t.stage, h.stage)
    np.testing.assert_array_equal(t.local, h.local)
    ctx.set_tiling(64)


@pytest.mark.parametrize("accum", [G.ACCUM_F64, G.ACCUM_KAHAN_F32])
@pytest.mark.parametrize("name", ["ragged", "open"])
@pytest.mark.parametrize("tile,resident", [(64, 0), (4, 1)])
def test_mixed_launches_of_several_evaluations(ctx, accum, name, tile, resident):
    """As test_launches_of_several_evaluations for mixed precision with either
    kind of sum, whose kernels keep their own form of the loop over evaluations."""
    q, box, _, _ = system(name)
    ctx.set_kernel_config(4, 256, 4)
    ctx.set_tiling(tile, resident_per_cu=resident)
    ctx.set_half_mode(G.HALF_AUTO)
    dq, da, db = ctx.array(q), ctx.zeros(q.shape), ctx.zeros(q.shape)
    ctx.build_list(dq, q.shape[0], box, G.LIST_FULL)
    for steps in (2, 5, 17, 100):
        ctx.force_aos_mixed(dq, da, 1e-3, G.CL2, box, steps, accum)
        for _ in range(steps):
            ctx.force_aos_mixed(dq, db, 1e-3, G.CL2, box, 1, accum)
        ctx.sync()
        np.testing.assert_array_equal(da.download(), db.download())
    ctx.set_tiling(64)


@pytest.mark.parametrize("cells", [14, 15])
@pytest.mark.parametrize("layout", ["aos", "soa", "aos3"])
@pytest.mark.parametrize("kind", [G.LIST_FULL, G.LIST_HALF])
def test_copies_in_slot_order_around_one_round_of_tiles(ctx, cells, layout, kind):
    """10,976 and 13,500 particles in tiles of 4 are 0.9 and 1.1 rounds of tiles of
    256 compute units; from one round on shorter calls run over copies of the
    arrays in slot order: bit for bit what as many calls of one step give."""
    q, box = G.lattice_periodic(cells, 0.5, 3)
    q = np.ascontiguousarray(q[np.random.default_rng(cells).permutation(q.shape[0])])
    n = q.shape[0]
    ctx.set_kernel_config(4, 256, 4)
    ctx.set_tiling(4)
    ctx.set_half_mode(G.HALF_AUTO)
    if layout == "soa":
        dq = [ctx.array(np.ascontiguousarray(q[:, c])) for c in range(3)]
        da, db = ([ctx.zeros(n) for _ in range(3)] for _ in range(2))
        build, force = ctx.build_list_soa, ctx.force_soa_f64
    else:
        w = 4 if layout == "aos" else 3
        dq, da, db = ctx.array(np.ascontiguousarray(q[:, :w])), ctx.zeros((n, w)), ctx.zeros((n, w))
        build = ctx.build_list if w == 4 else ctx.build_list_aos3
        force = ctx.force_aos_f64 if w == 4 else ctx.force_aos3_f64
    build(dq, n, box, kind)
    for steps in (3, 4, 5, 6, 7, 9, 10, 15, 16):
        force(dq, da, 1e-3, G.CL2, box, steps)
        for _ in range(steps):
            force(dq, db, 1e-3, G.CL2, box, 1)
        ctx.sync()
        for a, b in zip(*(([x] if layout != "soa" else x) for x in (da, db))):
            np.testing.assert_array_equal(a.download(), b.download())
    ctx.set_tiling(64)


@pytest.mark.parametrize("unroll", [1, 2, 4])
@pytest.mark.parametrize("gap", [1e-30, 1e-40, 1e-50])
def test_particles_that_all_but_coincide(ctx, gap, unroll):
    """Two particles so close that s = 1 / r^2 overflows in the fourth power: the
    tiled kernel's momenta are the untiled one's, infinite in the pair's
    directions, and finite for the others."""
    q, box = G.lattice_periodic(6, 0.5, 3)
    q = q.copy()
    # a pair at the origin, nobody else within reach of the overflow
    q[0, :3] = 0.0
    q[1, :3] = gap * np.array([1.0, 2.0, 3.0])
    full = G.makepair(q, box, G.LIST_FULL)
    ctx.set_half_mode(G.HALF_AUTO)
    ctx.set_kernel_config(4, 256, unroll)
    p = []
    for tile in (0, 64):
        ctx.set_tiling(tile)
        ctx.set_list(full)
        dq, dp = ctx.array(q), ctx.zeros(q.shape)
        ctx.force_aos_f64(dq, dp, 1e-3, G.CL2, box, 1)
        ctx.sync()
        p.append(dp.download()[:, :3])
    print(f"gap {gap}: {p[0][0]} {p[1][0]}", flush=True)
    assert not np.isnan(p[0]).any() and not np.isnan(p[1]).any()
    big = np.abs(p[0]) > 1e100
    np.testing.assert_array_equal(np.isinf(p[0]), np.isinf(p[1]))
    np.testing.assert_array_equal(np.sign(p[0][big]), np.sign(p[1][big]))
    assert big[:2].all() and not big[2:].any()
    assert normwise(p[1][2:], p[0][2:]) < FP64_TOL
    ctx.set_kernel_config(4, 256, 4)
    ctx.set_tiling(64)
