"""The matrix-core passes in the engine's real type against the VALU kernels
of the same engine (GPU tests): predictor, local integral and the fused LTS
pass, every order they serve, ragged layers and enough workgroups to put the
memory system under load."""
import ctypes as C

import pytest

from seissol_amd import _capi
from seissol_amd._capi import check, lib, ptr
from seissol_amd.kernels import Engine, global_matrices, num_basis, num_face_basis, padded_face_basis
from seissol_amd.proxy import DeviceLayer, make_setup, run_proxy

pytestmark = pytest.mark.gpu


def random_layer(eng, order, arith, n, align, star, seed, setup=False):
    """Arrays of random values (the kernels are linear maps of the DOFs: no mesh is needed)."""
    import torch
    rt = torch.float64 if arith == "fp64" else torch.float32
    ld, reals, dsize = C.c_int32(), C.c_int64(), C.c_int64()
    check(lib().sdg_layout_sizes(eng.handle, C.byref(ld), C.byref(reals), C.byref(dsize)), "sdg_layout_sizes")
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *shape: torch.rand(shape, generator=gen, device="cuda", dtype=rt) * 2 - 1
    a = dict(dofs=rnd(n, 9, ld.value), integrated=rnd(n, 9, ld.value), derivatives=rnd(n, dsize.value),
             star=rnd(n, 3, 24 if star == "compact" else 81), aplus=rnd(n, 4, 81))
    if setup:
        bits = torch.randint(0, 8, (n,), generator=gen, device="cuda", dtype=torch.int32) << 8
        a["setup"] = bits.to(torch.int16)
    a["view"] = _capi.Layer(n, ptr(a["dofs"]), ptr(a["integrated"]), ptr(a["derivatives"]), ptr(a["star"]),
                            ptr(a["aplus"]), None, None, None, None, None, ptr(a.get("setup")), 0, 0, 0)
    return a


def run_local(eng, a, part, reset):
    import torch
    coeffs = (C.c_double * 8)(1.0, 0.5, 0.2, 0.1, 0.05, 0.02, 0.01, 0.005)
    s, view = torch.cuda.current_stream().cuda_stream, C.byref(a["view"])
    if part == "ader":
        check(lib().sdg_compute_batched_ader(eng.handle, coeffs, 1.0, view, s), part)
    elif part == "local":
        check(lib().sdg_compute_batched_integral(eng.handle, view, s), part)
    else:
        check(lib().sdg_compute_local_integration(eng.handle, coeffs, 1.0, view, reset, s), part)
    torch.cuda.synchronize()


def same(a, b, keys, tol, what):
    import torch
    for k in keys:
        assert torch.isfinite(a[k]).all(), (what, k)
        err = float((a[k] - b[k]).abs().max() / b[k].abs().max())
        print(f"{what} {k}: largest difference / largest value {err:.1e}", flush=True)
        assert err < tol, (what, k)


# sums of at most 3 * 84 products in O - 1 <= 6 nested steps: 1e4 roundings at the very most
@pytest.mark.parametrize("arith,tol", [("fp64", 1e-12), ("fp32", 5e-5)])
@pytest.mark.parametrize("order", [3, 4, 5, 6, 7])
def test_local_passes_equal_the_valu_kernels(gpu, order, arith, tol):
    for n, align, star, part, reset in ((1, 0, "dense", "ader", 1), (17, 128, "compact", "local", 1),
                                        (333, 0, "compact", "lts", 1), (333, 128, "dense", "lts", 0)):
        print(f"mx {arith} order={order} n={n} align={align} {star} {part}", flush=True)
        sides = []
        for family in ("auto", "valu"):
            eng = Engine(order, arith)
            eng.set_layout(align, star)
            eng.set_kernels(family)
            a = random_layer(eng, order, arith, n, align, star, 7 * order + n, setup=part == "lts")
            run_local(eng, a, part, reset)
            sides.append(a)
        same(*sides, ("dofs", "integrated", "derivatives"), tol, f"{part} n={n}")


@pytest.mark.parametrize("arith,tol", [("fp64", 1e-12), ("fp32", 5e-5)])
def test_local_pass_under_memory_load(gpu, arith, tol):
    # thousands of workgroups with all their stores in flight
    sides = []
    for family in ("auto", "valu"):
        eng = Engine(6, arith)
        eng.set_kernels(family)
        a = random_layer(eng, 6, arith, 50_000, 0, "dense", 3, setup=True)
        run_local(eng, a, "lts", 0)
        sides.append(a)
    same(*sides, ("dofs", "integrated", "derivatives"), tol, f"{arith} n=50000")


def run_neighbor(eng, a, lts):
    import torch
    time = (C.c_double * 8)(1.0, 0.5, 0.2, 0.1, 0.05, 0.02, 0.01, 0.005)
    sub = (C.c_double * 8)(0.5, 0.4, 0.3, 0.2, 0.1, 0.05, 0.02, 0.01)
    s, view = torch.cuda.current_stream().cuda_stream, C.byref(a["view"])
    if lts:
        check(lib().sdg_compute_neighboring_integration(eng.handle, time, sub, view, s), "neighbour lts")
    else:
        check(lib().sdg_compute_batched_neighbors_integral(eng.handle, view, s), "neighbour")
    torch.cuda.synchronize()


# n, alignment, sides drawn from [0, sides), LTS: one element; ragged; one side only (full
# groups); every side; enough elements for every CU
@pytest.mark.parametrize("arith,tol", [("fp64", 1e-12), ("fp32", 5e-5)])
@pytest.mark.parametrize("order", [3, 4, 5, 6, 7])
def test_neighbour_pass_equals_the_valu_kernels(gpu, order, arith, tol):
    import torch
    for n, align, sides, lts in ((1, 0, 4, False), (17, 128, 4, True), (333, 0, 1, False), (333, 0, 2, True),
                                 (9001, 128, 4, True), (9001, 0, 4, False)):
        print(f"mx neighbour {arith} order={order} n={n} align={align} sides={sides} lts={lts}", flush=True)
        results = []
        for family in ("auto", "valu"):
            eng = Engine(order, arith)
            eng.set_layout(align, "compact")
            eng.set_kernels(family)
            a = random_layer(eng, order, arith, n, align, "compact", 5 * order + n, setup=True)
            gen = torch.Generator(device="cuda").manual_seed(n)
            draw = lambda hi, shape, t: torch.randint(0, hi, shape, generator=gen, device="cuda").to(t)
            a["neighbors"] = draw(n, (n, 4), torch.int32)
            a["relations"] = torch.stack([draw(sides, (n, 4), torch.uint8), draw(3, (n, 4), torch.uint8)], -1)
            a["types"] = (draw(8, (n, 4), torch.int32) == 0).to(torch.uint8)  # some dynamic-rupture faces
            a["aminus"] = torch.rand((n, 4, 81), generator=gen, device="cuda", dtype=a["dofs"].dtype) * 2 - 1
            a["setup"] = draw(1 << 11, (n,), torch.int16)
            v = a["view"]
            v.aminus, v.face_neighbors, v.face_relations = ptr(a["aminus"]), ptr(a["neighbors"]), ptr(a["relations"])
            v.face_types, v.lts_setup = ptr(a["types"]), ptr(a["setup"])
            run_neighbor(eng, a, lts)
            results.append(a)
        same(*results, ("dofs",), tol, f"neighbour n={n} lts={lts}")


# the neighbour pass from face traces (global time stepping); the sums have at
# most O + 9 + 4 * 28 = 128 terms: 128 roundings of 2^-53 / 2^-24
@pytest.mark.parametrize("arith,order,tol", [(a, o, t) for a, t, orders in (
    ("fp64", 1.5e-14, (3, 4, 5, 6, 7)), ("f16x3", 8e-6, (3, 4, 5, 7)), ("bf16x6", 8e-6, (3, 6))) for o in orders])
def test_neighbour_pass_from_traces(gpu, arith, order, tol):
    import torch
    gm = {k: torch.from_numpy(v).cuda() for k, v in global_matrices(order).items() if k in ("rDivM", "fP")}
    B2, B2P = num_face_basis(order), padded_face_basis(order)
    for n, align, dr in ((1, 0, False), (17, 128, True), (333, 0, True), (9001, 0, False)):
        print(f"traces {arith} order={order} n={n} align={align}", flush=True)
        eng = Engine(order, arith)
        eng.set_layout(align, "compact")
        a = random_layer(eng, order, arith, n, align, "compact", 3 * order + n)
        gen = torch.Generator(device="cuda").manual_seed(n)
        draw = lambda hi, shape, t: torch.randint(0, hi, shape, generator=gen, device="cuda").to(t)
        rt = a["dofs"].dtype
        nb, side, h = draw(n, (n, 4), torch.int32), draw(4, (n, 4), torch.uint8), draw(3, (n, 4), torch.uint8)
        types = (draw(8, (n, 4), torch.int32) == 0).to(torch.uint8) if dr else None
        relations = torch.stack([side, h], -1)
        aminus = torch.rand((n, 4, 81), generator=gen, device="cuda", dtype=rt) * 2 - 1
        traces = torch.rand((n, 4, 9, B2P), generator=gen, device="cuda", dtype=rt) * 2 - 1
        v = a["view"]
        v.aminus, v.face_neighbors, v.face_relations = ptr(aminus), ptr(nb), ptr(relations)
        v.face_types, v.face_traces = ptr(types), ptr(traces)
        B = num_basis(order)
        want = a["dofs"][:, :, :B].double()
        for f in range(4):
            u = traces[nb[:, f].long(), side[:, f].long()][:, :, :B2].double()  # [n][q][m]
            u = (gm["fP"][h[:, f].long()] @ u.transpose(1, 2).contiguous()).transpose(1, 2).contiguous()
            w = aminus[:, f].reshape(n, 9, 9).double() @ u                       # [n][p][m]
            if dr:
                w[types[:, f] != 0] = 0
            want = want + w @ gm["rDivM"][f].T.contiguous()
        check(lib().sdg_proxy_run(eng.handle, 2, 1, 1e-3, C.byref(v), torch.cuda.current_stream().cuda_stream), "neigh")
        torch.cuda.synchronize()
        got = a["dofs"][:, :, :B].double()
        err = float((got - want).abs().max() / want.abs().max())
        print(f"  largest difference / largest value {err:.1e}", flush=True)
        assert err < tol


# clusters that step together share a launch: a cluster of one cell, an empty one, ragged ones, and a launch
# of several with another variant's between them, against the VALU kernels cluster by cluster
@pytest.mark.parametrize("arith,tol", [("fp64", 1e-12), ("fp32", 5e-5), ("f16x3", 5e-5)])
@pytest.mark.parametrize("order", [3, 6])
@pytest.mark.parametrize("graph", [False, True])
def test_clusters_in_one_launch_equal_the_valu_kernels(gpu, order, arith, tol, graph):
    import torch
    starts = [0, 100, 101, 101, 134, 150]
    n, C_ = starts[-1], len(starts) - 1
    print(f"clusters {arith} order={order} graph={graph}", flush=True)
    sides = []
    for valu in (False, True):
        eng = Engine(order, arith)
        eng.set_layout(0, "compact")
        a = random_layer(eng, order, arith, n, 0, "compact", 11 * order)
        gen = torch.Generator(device="cuda").manual_seed(order)
        draw = lambda hi, shape, t: torch.randint(0, hi, shape, generator=gen, device="cuda").to(t)
        a["neighbors"] = draw(n, (n, 4), torch.int32)
        a["relations"] = torch.stack([draw(4, (n, 4), torch.uint8), draw(3, (n, 4), torch.uint8)], -1)
        a["aminus"] = torch.rand((n, 4, 81), generator=gen, device="cuda", dtype=a["dofs"].dtype) * 2 - 1
        a["setup"] = draw(1 << 11, (n,), torch.int16)
        for k in ("star", "aplus", "aminus"):
            a[k] *= 0.02  # 16 steps without growth
        v = a["view"]
        v.star, v.aplus, v.aminus = ptr(a["star"]), ptr(a["aplus"]), ptr(a["aminus"])
        v.face_neighbors, v.face_relations, v.lts_setup = ptr(a["neighbors"]), ptr(a["relations"]), ptr(a["setup"])
        handle, cuts = C.c_void_p(), (C.c_int64 * (C_ + 1))(*starts)
        check(lib().sdg_lts_create(C.byref(handle), eng.handle, C.byref(v), C_, cuts, 1e-2), "create")
        for c in range(C_):
            if valu or c == 3:
                check(lib().sdg_lts_set_tile_variant(handle, c, 0, 1), "local variant")
                check(lib().sdg_lts_set_tile_variant(handle, c, 1, 1), "neighbour variant")
        s = torch.cuda.current_stream().cuda_stream
        check((lib().sdg_lts_graph_advance if graph else lib().sdg_lts_advance)(handle, 1, s), "advance")
        torch.cuda.synchronize()
        check(lib().sdg_lts_destroy(handle), "destroy")
        sides.append(a)
    same(*sides, ("dofs", "integrated", "derivatives"), tol, f"clusters {arith}")


# A step's rounding against 64 bits on the same single-precision inputs.  The bounds are the errors that
# the split products the two forms are named after (two scaled fp16 planes, three bf16 planes) had in
# this test: what runs in their place may not be less accurate.
@pytest.mark.parametrize("arith,order,bound", [
    ("f16x3", 3, 1.79e-7), ("f16x3", 4, 1.97e-7), ("f16x3", 5, 2.11e-7), ("f16x3", 6, 2.36e-7), ("f16x3", 7, 2.58e-7),
    ("bf16x6", 4, 1.90e-7), ("bf16x6", 5, 2.12e-7), ("bf16x6", 6, 2.38e-7), ("bf16x6", 7, 2.74e-7)])
def test_a_step_is_as_accurate_as_the_split_products(gpu, arith, order, bound):
    import torch
    print(f"step accuracy {arith} order={order}", flush=True)
    setup = make_setup(order, n=3000, mesh="proxy", seed=17)
    layers = [(eng, DeviceLayer(eng, setup)) for eng in (Engine(order, arith), Engine(order, "fp64"))]
    for k in ("dofs", "star", "aplus", "aminus"):
        getattr(layers[1][1], k).copy_(getattr(layers[0][1], k))
    for eng, layer in layers:
        run_proxy(eng, layer, "all", 1, setup.dt)
    torch.cuda.synchronize()
    got, want = (layer.dofs.double() for _, layer in layers)
    err = float((got - want).norm() / want.norm())
    print(f"  error {err:.3e}, split products {bound:.2e}", flush=True)
    assert err <= bound


# strides of the per-cell operators at which 16 cells are more than 2^31 bytes apart (the padding
# between them is never touched): a ragged tile and more than one
@pytest.mark.parametrize("arith", ["fp64", "fp32", "f16x3"])
@pytest.mark.parametrize("n,megabytes", [(5, 640), (18, 160)])
def test_operators_far_apart_equal_dense_ones(gpu, arith, n, megabytes):
    import torch
    order = 4
    stride = megabytes * 2**20 // (8 if arith == "fp64" else 4)
    print(f"operators {megabytes} MB apart {arith} n={n}", flush=True)
    for part in ("ader", "local", "lts") if arith != "f16x3" else ("proxy", "lts"):
        sides = []
        for far in (False, True):
            eng = Engine(order, arith)
            eng.set_layout(0, "compact")
            a = random_layer(eng, order, arith, n, 0, "compact", n, setup=part == "lts")
            a["traces"] = torch.zeros((n, 4, 9, padded_face_basis(order)), dtype=a["dofs"].dtype, device="cuda")
            v = a["view"]
            if far:
                for k in ("star", "aplus"):
                    dense = a[k].reshape(n, -1)
                    a[k] = torch.empty((n, stride), dtype=dense.dtype, device="cuda")
                    a[k][:, :dense.shape[1]] = dense
                v.star, v.aplus, v.star_stride, v.aplus_stride = ptr(a["star"]), ptr(a["aplus"]), stride, stride
            if part == "proxy":
                v.face_traces = ptr(a["traces"])
                s = torch.cuda.current_stream().cuda_stream
                check(lib().sdg_proxy_run(eng.handle, 1, 1, 1e-3, C.byref(v), s), "local")
                torch.cuda.synchronize()
            else:
                run_local(eng, a, part, 1)
            sides.append(a)
        for k in ("dofs", "integrated", "derivatives", "traces"):
            assert torch.equal(sides[0][k], sides[1][k]), (part, k)
        del sides, a
    torch.cuda.empty_cache()


# the line between the VALU and the matrix-core neighbour pass at ORDER 3 (24 cells per CU in FP64 from
# DOFs, the matrix cores in FP64 with LTS, the VALU in FP32): the same kernel below it, the same values above
@pytest.mark.parametrize("lts", [False, True])
@pytest.mark.parametrize("arith,n,equal", [("fp64", 6144, True), ("fp64", 6145, False), ("fp32", 6145, True)])
def test_neighbour_pass_of_order_3(gpu, arith, n, equal, lts):
    import torch
    print(f"neighbour order=3 {arith} n={n} lts={lts}", flush=True)
    results = []
    for family in ("auto", "valu"):
        eng = Engine(3, arith)
        eng.set_kernels(family)
        a = random_layer(eng, 3, arith, n, 0, "dense", n, setup=True)
        gen = torch.Generator(device="cuda").manual_seed(n)
        draw = lambda hi, shape, t: torch.randint(0, hi, shape, generator=gen, device="cuda").to(t)
        a["neighbors"] = draw(n, (n, 4), torch.int32)
        a["relations"] = torch.stack([draw(4, (n, 4), torch.uint8), draw(3, (n, 4), torch.uint8)], -1)
        a["aminus"] = torch.rand((n, 4, 81), generator=gen, device="cuda", dtype=a["dofs"].dtype) * 2 - 1
        a["setup"] = draw(1 << 11, (n,), torch.int16)
        v = a["view"]
        v.aminus, v.face_neighbors, v.face_relations = ptr(a["aminus"]), ptr(a["neighbors"]), ptr(a["relations"])
        v.lts_setup = ptr(a["setup"])
        run_neighbor(eng, a, lts)
        results.append(a)
    assert torch.equal(results[0]["dofs"], results[1]["dofs"]) == (equal and not (lts and arith == "fp64"))
    same(*results, ("dofs",), 1e-12 if arith == "fp64" else 5e-5, f"neighbour order 3 n={n}")
