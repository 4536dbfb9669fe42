"""The rules that choose the kernel of a prefill matmul from 64 tokens on: host
functions of the library, called on shapes alone (no launch, no GPU). Each listed
shape was measured on the kernel it takes and on the one it would take otherwise."""
import ctypes as C

import pytest


class Group(C.Structure):
    """MatmulGroupLaunch of nightrun_amd/csrc/nrq_launch.h."""
    _fields_ = [("w", C.c_void_p * 3), ("y", C.c_void_p * 3), ("rows", C.c_int * 3), ("nmat", C.c_int),
                ("xs", C.c_void_p), ("bpr", C.c_int), ("batch", C.c_int), ("stream", C.c_void_p)]


def group(rows, bpr, batch):
    g = Group(nmat=len(rows), xs=1 << 20, bpr=bpr, batch=batch)
    for i, r in enumerate(rows):
        g.w[i], g.y[i], g.rows[i] = 16 << 20 | i << 30, 17 << 20 | i << 30, r
    return g


def rule(name, *extra):
    from nightrun_amd import _lib

    fn = getattr(_lib.lib(), name)
    fn.restype = C.c_bool
    fn.argtypes = [C.POINTER(Group), *extra]
    return fn


@pytest.mark.parametrize("rows,bpr,batch,takes", [
    ((9728, 9728), 10, 512, True), ((9728, 9728), 10, 63, False), ((127, 9728), 10, 512, False),
    ((2560,), 38, 512, False),  # rows of 32 blocks and more
    ((5120,), 10, 256, True), ((4992,), 10, 224, False),  # 320 workgroups, 273
    ((3473,), 23, 340, True), ((4463, 6013), 31, 110, False), ((3759,), 30, 424, True),  # 308, 328, 420
    ((3616, 168, 4323), 22, 233, False), ((2472, 268, 7968), 8, 258, False),  # a round more than the rows fill
    ((4480,), 19, 405, True), ((6770,), 20, 419, True)])
def test_q4k_route(rows, bpr, batch, takes):
    fits = rule("_ZN3nrq8mmk_fitsERKNS_17MatmulGroupLaunchEb", C.c_bool)
    assert fits(C.byref(group(rows, bpr, batch)), False) == takes


@pytest.mark.parametrize("rows,bpr,batch,tall", [
    ((8192, 8192), 64, 512, None), ((545, 758), 67, 224, None), ((1300, 984), 303, 215, None),  # no short one
    ((3000, 40, 3200), 34, 67, None), ((6, 5198), 46, 314, (5198,)), ((4870, 41), 75, 188, (4870,)), ((9769, 12), 269, 135, (9769,)),
    ((62, 4121, 2383), 48, 135, (4121, 2383)), ((10000, 40, 10100), 24, 130, (10000, 10100)), ((5, 9), 64, 512, None)])
def test_q8_0_group_with_short_matrices(rows, bpr, batch, tall):
    """Groups stay one launch, except that matrices of fewer rows than a tile go alone
    where the others are large enough; a group without such a matrix never splits."""
    fits = rule("_ZN3nrq18mm8_fits_but_shortERKNS_17MatmulGroupLaunchEPS0_", C.POINTER(Group))
    g, h = group(rows, bpr, batch), Group()
    assert fits(C.byref(g), C.byref(h)) == (tall is not None)
    if tall:
        keep = [i for i, r in enumerate(rows) if r in tall]
        assert tuple(h.rows[:h.nmat]) == tall
        assert [(h.w[k], h.y[k]) for k in range(h.nmat)] == [(g.w[i], g.y[i]) for i in keep]
        assert (h.xs, h.bpr, h.batch) == (g.xs, bpr, batch)


@pytest.mark.parametrize("rows,bpr,batch,takes", [
    ((8192, 8192), 64, 512, True), ((8192, 8192), 64, 63, False), ((63, 8192), 64, 512, False),
    ((3072,), 64, 128, True), ((2048,), 64, 128, False),  # 96 workgroups, 64
    # odd rows: two tiles of 32 x 32 per CU, and stages of 1.6 times the row
    ((4266,), 35, 85, False), ((4643,), 145, 84, False), ((4102,), 23, 118, True), ((1191,), 141, 395, True),
    ((9908,), 9, 262, False),
    # below 1024 rows
    ((225,), 320, 371, False), ((370,), 308, 455, False), ((604,), 192, 277, True), ((674,), 76, 305, True), ((967,), 50, 244, False),
    ((732,), 55, 354, True), ((517,), 33, 456, False), ((742,), 307, 344, True), ((709,), 18, 227, False),
    ((512,), 64, 512, True), ((512,), 64, 256, False), ((600,), 256, 300, True), ((972,), 18, 415, True)])
def test_q8_0_route(rows, bpr, batch, takes):
    fits = rule("_ZN3nrq8mm8_fitsERKNS_17MatmulGroupLaunchEb", C.c_bool)
    assert fits(C.byref(group(rows, bpr, batch)), False) == takes
