"""A caller's own global matrices on the matrix-core passes against the VALU kernels of the same engine
(GPU tests): full matrices, small entries where the basis has zeros, fuller face permutations."""
import ctypes as C

import numpy as np
import pytest

from seissol_amd import _capi
from seissol_amd._capi import check, lib, ptr
from seissol_amd.kernels import Engine, global_matrices, num_basis, num_face_basis
from test_gpu_mx import random_layer, run_local, run_neighbor

pytestmark = pytest.mark.gpu

REAL = {"fp64": 1e-12, "fp32": 5e-5}  # the bounds of test_gpu_mx.py


def engine(order, arith, family, gm):
    eng = Engine(order, arith)
    eng.set_layout(0, "compact")
    if arith in REAL:
        eng.set_kernels(family)
    check(lib().sdg_engine_set_global_matrices(eng.handle, gm.ctypes.data), "sdg_engine_set_global_matrices")
    return eng


def layer(eng, order, arith, n):
    """random_layer with neighbours, sides and orientations of every kind"""
    import torch
    a = random_layer(eng, order, arith, n, 0, "compact", 40 + order, setup=True)
    gen = torch.Generator(device="cuda").manual_seed(n)
    draw = lambda hi, shape, t: torch.randint(0, hi, shape, generator=gen, device="cuda").to(t)
    a["neighbors"] = draw(n, (n, 4), torch.int32)
    a["relations"] = torch.stack([draw(4, (n, 4), torch.uint8), draw(3, (n, 4), torch.uint8)], -1)
    a["aminus"] = torch.rand((n, 4, 81), generator=gen, device="cuda", dtype=a["dofs"].dtype) * 2 - 1
    v = a["view"]
    v.aminus, v.face_neighbors, v.face_relations = ptr(a["aminus"]), ptr(a["neighbors"]), ptr(a["relations"])
    return a


def call(eng, a, part):
    if part == "neighbour":
        run_neighbor(eng, a, False)
    elif part == "neighbour lts":
        run_neighbor(eng, a, True)
    else:
        run_local(eng, a, part, 1)


def compare(order, arith, gm, part, prepare=lambda a: None, n=150, rows=slice(None)):
    """Largest difference of auto and VALU over the largest value of the DOFs' (or integral's) `rows`."""
    import torch
    sides = []
    for family in ("auto", "valu"):
        eng = engine(order, arith, family, gm)
        a = layer(eng, order, arith, n)
        prepare(a)
        call(eng, a, part)
        torch.cuda.synchronize()
        sides.append(a["integrated" if part == "ader" else "dofs"][:, :, rows].clone())
    assert float(sides[1].abs().max()) > 0
    err = float((sides[0] - sides[1]).abs().max() / sides[1].abs().max())
    print(f"{arith} order={order} {part}: {err:.1e}", flush=True)
    return err


@pytest.mark.parametrize("arith", ["fp64", "fp32"])
@pytest.mark.parametrize("order", [3, 5, 6, 7])
def test_full_matrices(gpu, order, arith):
    # every entry of every matrix but fP: no k-step may be skipped
    g = global_matrices(order)
    rng = np.random.default_rng(order)
    for k in ("kDivM", "kDivMT", "rDivM", "fMrT", "rT"):
        g[k][:] = rng.uniform(-1, 1, g[k].shape)  # views of the flat array
    for part in ("ader", "local", "lts", "neighbour", "neighbour lts"):
        assert compare(order, arith, g["flat"], part) < REAL[arith], part


# a single entry of 5e-14 of the matrix's largest where the basis has a zero, seen alone: all other
# inputs that reach its row are zero
@pytest.mark.parametrize("arith", ["fp64", "fp32"])
@pytest.mark.parametrize("part", ["ader", "local", "neighbour"])
def test_small_entries_of_a_caller_count(gpu, arith, part):
    order = 5
    B = num_basis(order)
    g = global_matrices(order)
    if part == "ader":  # derivative 1: the last row of the second row tile from the first column
        row, col = num_basis(order - 1) - 1, 0
        g["kDivMT"][:, row, :] = 0
        g["kDivMT"][:, row, col] = 5e-14 * np.abs(g["kDivMT"]).max()

        def prepare(a):
            a["dofs"][:, :, 1:] = 0
    elif part == "local":  # volume: the first row from the last column
        row, col = 0, B - 1
        g["kDivM"][:, row, :] = 0
        g["kDivM"][:, row, col] = 5e-14 * np.abs(g["kDivM"]).max()

        def prepare(a):
            a["integrated"][:, :, :-1] = 0
            a["dofs"].zero_()
            a["aplus"].zero_()
    else:  # face rows: U has row 0 only, fP takes it to the last row with the small entry alone
        row, col = slice(None), 0
        g["rT"][:, 1:] = 0
        g["fP"][:, :, 0] = 0
        g["fP"][:, -1, 0] = 5e-14 * np.abs(g["fP"]).max()

        def prepare(a):
            a["dofs"].zero_()
    assert compare(order, arith, g["flat"], part, prepare, rows=row) < REAL[arith]


@pytest.mark.parametrize("arith", ["fp64", "fp32", "f16x3", "bf16x3"])
@pytest.mark.parametrize("order", [4, 6])
def test_fuller_face_permutations(gpu, order, arith):
    # more than `order` entries in a row: FP32 engines run the VALU neighbour pass, the others refuse
    g = global_matrices(order)
    g["fP"][1, 2] = 0.5
    assert num_face_basis(order) > order
    if arith == "fp32":
        for part in ("local", "neighbour", "neighbour lts"):
            assert compare(order, arith, g["flat"], part) < REAL[arith]
    else:
        with pytest.raises(_capi.SdgError, match="more than `order` non-zeros"):
            engine(order, arith, "auto", g["flat"])


@pytest.mark.parametrize("arith", ["fp64", "fp32", "f16x3", "bf16x6"])
def test_the_generated_matrices_given_back_change_nothing(gpu, arith):
    import torch
    order, n = 6, 150
    sides = []
    for again in (False, True):
        eng = Engine(order, arith)
        eng.set_layout(0, "compact")
        if again:
            gm = global_matrices(order)["flat"]
            check(lib().sdg_engine_set_global_matrices(eng.handle, gm.ctypes.data), "sdg_engine_set_global_matrices")
        a = layer(eng, order, arith, n)
        call(eng, a, "lts")
        call(eng, a, "neighbour lts")
        torch.cuda.synchronize()
        sides.append(a)
    for k in ("dofs", "integrated", "derivatives"):
        assert torch.equal(sides[0][k], sides[1][k]), k
