"""CPU checks of how a conv call uses its workspace (q8_debug_conv_plan).

A plan is asked for over swept geometries (ranks, groups, strides, dilations,
short and long contractions, ui8 operands and zero points, prepacked weights),
workspace sizes and alignments, and what its passes write is worked out here
from the route alone: never more than the workspace that was accepted.
Nothing is launched."""
import ctypes as C
import os
import random

import pytest

DIRECT, FRAME, MATRIX = 0, 1, 2


@pytest.fixture(scope="module")
def lib():
    from mlfw_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.fail("libq8hip.so is not built: run `python -m mlfw_amd.build`")
    return _lib


def arr(v):
    return (C.c_int64 * len(v))(*v)


def geom(xs, ws, st, lo, hi, dl, g):
    return (len(xs) - 2, arr(xs), arr(ws), arr(st), arr(lo), arr(hi), arr(dl), g)


def asked(lib, args):
    need = C.c_size_t(0)
    assert lib.load().q8_quantized_conv_workspace(*args, C.byref(need)) == lib.Q8_OK
    return need.value


def plan(lib, args, ws_at, ws_bytes, xd=0, zx=0, wd=0, zw=0, taps=0):
    """(route, images, groups, bytes), None where the call is refused."""
    r, nb, gc, b = C.c_int(), C.c_int64(), C.c_int64(), C.c_size_t()
    rc = lib.load().q8_debug_conv_plan(*args, xd, zx, wd, zw, taps, C.c_void_p(ws_at), ws_bytes, C.byref(r),
                                       C.byref(nb), C.byref(gc), C.byref(b))
    assert rc in (lib.Q8_OK, lib.Q8_ERR_INVALID), lib.load().q8_last_error()
    return (r.value, nb.value, gc.value, b.value) if rc == lib.Q8_OK else None


def written(case, route, nb, gc, ws_at, taps):
    """Workspace bytes that a pass of nb images and gc groups writes, at least."""
    xs, ws, st, lo, hi, dl, g = case
    if route == DIRECT:
        return 0
    pad = -ws_at % 16
    kc, kn = ws[1], 1
    P, E = 1, 1
    for i in range(len(xs) - 2):
        k, d = ws[2 + i], dl[i]
        p = (xs[2 + i] + lo[i] + hi[i] - (k - 1) * d - 1) // st[i] + 1
        P, E, kn = P * p, E * ((p - 1) * st[i] + (k - 1) * d + 1), kn * k
    kc *= kn
    if route == FRAME:
        assert ws[1] % 16 == 0
        return pad + nb * gc * E * ws[1] + (0 if taps or kn == 1 else ws[0] * kc)
    return pad + nb * gc * P * (-(-kc // 16) * 16)


def random_case(rng):
    d = rng.choice([1, 2, 2, 2, 3])
    g = rng.choice([1, 1, 1, 2, 4])
    cg = rng.choice([1, 3, 8, 10, 16, 16, 16, 24, 32, 48, 64, 96, 128])
    o = g * rng.choice([4, 8, 9, 16, 17, 64, 130])
    n = rng.choice([1, 1, 2, 3, 7, 40])
    big = {1: 6000, 2: 112, 3: 24}[d]
    S = [rng.randint(1, big) for _ in range(d)]
    K, st, dl, lo, hi = [], [], [], [], []
    for i in range(d):
        k, dil, a, b = rng.choice([1, 1, 2, 3, 3, 5]), rng.choice([1, 1, 2]), rng.randint(0, 2), rng.randint(0, 2)
        if (k - 1) * dil + 1 > S[i] + a + b:
            k = 1
        K.append(k), st.append(rng.choice([1, 1, 2, 3])), dl.append(dil), lo.append(a), hi.append(b)
    return ([n, g * cg, *S], [o, cg, *K], st, lo, hi, dl, g)


SHORT = [   # few taps of 16 channels, enough work for the GEMM: the frame is smaller than the matrix
    ([1, 16, 112, 112], [64, 16, 1, 3], [1, 1], [0, 1], [0, 1], [1, 1], 1),
    ([1, 16, 6000], [64, 16, 3], [1], [1], [1], [1], 1),
    ([2, 16, 6000], [128, 16, 2], [1], [0], [0], [1], 1),
    ([1, 32, 3000], [256, 32, 1], [1], [0], [0], [1], 1),
]


def test_passes_stay_inside_the_workspace(lib):
    rng = random.Random(7)
    routes = set()
    for case in SHORT + [random_case(rng) for _ in range(600)]:
        args = geom(*case)
        want = asked(lib, args)
        kn = 1
        for k in case[1][2:]:
            kn *= k
        for xd, zx, wd, zw in ((0, 0, 0, 0), (1, 117, 0, 0), (0, -128, 1, 3), (1, 300, 0, 0)):
            taps = int(case[1][1] % 16 == 0 and kn > 1 and rng.random() < 0.5 and xd == wd == 0)
            for at in (0, 0x1000, 0x1001, 0x1008, 0x100f):
                for size in (want, want // 2, want - 1, want + 15, rng.randint(0, want + 64), 0):
                    if size < 0 or (at == 0 and size):
                        continue
                    p = plan(lib, args, at, size, xd, zx, wd, zw, taps)
                    if p is None:
                        assert size < want and (xd, zx, wd, zw) == (0, 0, 0, 0), (case, at, size)
                        continue
                    route, nb, gc, b = p
                    routes.add(route)
                    assert b <= size, (case, at, size, p)
                    assert written(case, route, nb, gc, at, taps) <= b, (case, at, size, p)
                    assert (route == DIRECT) == (nb == 0 and gc == 0)
    assert routes == {DIRECT, FRAME, MATRIX}


@pytest.mark.parametrize("case", SHORT)
def test_short_contraction_with_the_workspace_it_asks_for(lib, case):
    """An aligned workspace of the size asked for takes the frame; one that
    starts between 16-byte boundaries may not have room for it, and then no
    pass writes past its end."""
    args = geom(*case)
    want = asked(lib, args)
    assert want > 0
    assert plan(lib, args, 0x1000, want)[0] == FRAME
    for at in (0x1001, 0x1008, 0x100f):
        route, nb, gc, b = plan(lib, args, at, want)
        assert max(b, written(case, route, nb, gc, at, 0)) <= want


def test_workspace_asked_for_and_least_accepted(lib):
    """No more is asked for than one batch (128 MiB, or one image of one group
    where that is larger), the weight rows and 1 MiB of partial sums; a symmetric conv is accepted
    with one image of one group, and refused below."""
    rng = random.Random(11)
    many_groups = ([2, 256, 512, 512], [256, 8, 3, 3], [1, 1], [1, 1], [1, 1], [1, 1], 32)
    deep = ([4, 64, 12, 12], [32, 64, 3, 3], [1, 1], [1, 1], [1, 1], [1, 1], 1)      # long contraction, few tiles
    for case in [many_groups, deep] + [random_case(rng) for _ in range(300)]:
        args = geom(*case)
        want = asked(lib, args)
        xs, ws, g = case[0], case[1], case[6]
        kc = ws[1]
        for k in ws[2:]:
            kc *= k
        kn = kc // ws[1]
        frame = ws[1] % 16 == 0 and kc <= 65536 and kn <= 1024
        weight = ws[0] * (kc if frame and kn > 1 else -(-kc // 16) * 16)
        unit = written(case, FRAME if frame else MATRIX, 1, 1, 0, 1)
        assert want <= max(128 << 20, unit) + 512 + weight + 256 + (1 << 20), case
        if kc < 64:
            continue
        least = unit + (ws[0] * kc + 255) // 256 * 256 * (frame and kn > 1)
        assert least <= want, case
        assert plan(lib, args, 0x1000, least) is not None, case
        assert plan(lib, args, 0x1000, least - 1) is None, case
    # every group of every image in one pass where that is within a batch
    assert plan(lib, geom(*deep), 0x1000, asked(lib, geom(*deep)))[1:3] == (4, 1)
    r, nb, gc, b = plan(lib, geom(*many_groups), 0x1000, asked(lib, geom(*many_groups)))
    assert r == MATRIX and nb == 1 and 1 < gc < 32


def test_part_of_a_batch_or_one_thread_per_output(lib):
    """A workspace for part of the batch is used while its passes are fewer
    than the one-thread kernel's time is worth; below one image the affine
    call runs that kernel and the symmetric one is refused."""
    big = geom([16, 64, 56, 56], [64, 64, 3, 3], [1, 1], [1, 1], [1, 1], [1, 1], 1)
    one = 58 * 58 * 64 + 64 * 576
    for kind in ((0, 0, 0, 0), (1, 117, 0, 0)):
        assert plan(lib, big, 0x1000, one, *kind)[:3] == (FRAME, 1, 1)
    assert plan(lib, big, 0x1000, one - 1) is None
    assert plan(lib, big, 0x1000, one - 1, 1, 117)[0] == DIRECT
    tiny = geom([1000, 16, 7, 7], [16, 16, 3, 3], [1, 1], [1, 1], [1, 1], [1, 1], 1)
    one = 9 * 9 * 16 + 16 * 144
    assert plan(lib, tiny, 0x1000, asked(lib, tiny), 1, 117)[:3] == (FRAME, 1000, 1)
    assert plan(lib, tiny, 0x1000, one, 1, 117)[0] == DIRECT      # 1000 passes for 0.1 ms of work


def test_frame_launches_stay_within_the_grid(lib):
    """More channel tiles than grid.z takes, and more 64 x 64 tiles than a
    launch: fewer groups or images a pass, as a launch per group once did."""
    wide = geom([1, 128 * 40000, 1], [40000 * 17, 128, 1], [1], [0], [0], [1], 40000)
    r, nb, gc, b = plan(lib, wide, 0x1000, 1 << 33)
    assert r == FRAME and 0 < gc * 128 <= 64 * 65535
    points = geom([65535, 32768, 1], [17, 32768, 1], [1], [0], [0], [1], 1)
    r, nb, gc, b = plan(lib, points, 0x1000, 1 << 33)
    assert r == FRAME and 0 < nb * 512 <= 1 << 23
