"""The work that is timed: VV + critical points and the relation builds, through
the package's public entry points, from one small request to the 12.6 M-cell
benchmark mesh.

Every case is a Kuhn grid of n^3 cubes (6 n^3 cells) from the package's own
generator, or a batch of such grids.  Its fields:

  kind    field      a resident mesh; a pass recomputes VV and the classes
          request    host cells and scalars in, VV and classes out on the host
          buffers    the entry point without allocation, on the caller's buffers
          batch      many meshes in one launch sequence, classes to the host
          relations  a mesh made from cells on the GPU, then its relations
  n       side of the grid (batch: the largest side)
  order   permuted   random vertex ids, random cell order (the benchmark's)
          grid       vertices and cells as the grid generates them (most files)
          cells      random cell order, vertices in grid order
          vertices   random vertex ids, cells in grid order
  split   share of the cells split 1 -> 4 at their centroid (uneven degrees)
  hubs    vertices raised by 64 further splits around them (degrees over 32)
  scalar  the generator's field; f64: float64 scalars instead of float32
  build   relations: what is built, comma separated ("classes": critical points)
  meshes  batch: how many

All outputs are whole numbers (ids, offsets, classes), so they are compared
exactly and no reference in 64 bits is needed.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import tetragpu_amd as tetra
from tetragpu_amd import _native, tuning

RELATIONS = ("TE", "EV", "ET", "TF", "FV", "FE", "FT", "EF", "VT", "TT", "FF", "EE", "VV", "VE",
             "VF")
HUB_SPLITS = 64


def _case(name, kind, n, order="permuted", scalar="uniform", f64=False, split=0.0, hubs=0,
          build="", meshes=1):
    c = {"kind": kind, "n": n, "order": order, "scalar": scalar, "f64": f64, "split": split,
         "hubs": hubs, "build": build, "meshes": meshes}
    return {"name": name, **c} if name else c


def listed():
    return [
        # one small request end to end: upload, validation, launches and the
        # copies back count, the kernels hardly do
        _case("request_6k", "request", 10),
        # the smallest resident mesh of the benchmark (83 k cells): 16 launches
        # and the gaps between them
        _case("field_83k", "field", 24),
        # a caller under a no-allocation rule, its own buffers and stream
        _case("buffers_414k", "buffers", 41, scalar="gaussians"),
        # a mesh as a file stores it, in spatial order, with float64 scalars
        _case("field_grid_1m_f64", "field", 61, order="grid", scalar="gaussians", f64=True),
        # the headline benchmark: 12.6 M cells in random order
        _case("field_12m", "field", 128, scalar="gaussians"),
        # the irregular-degree workload: centroid splits and hub vertices
        _case("field_irregular_8m", "field", 96, scalar="sines", split=0.15, hubs=32),
        # many small meshes of uneven size at once
        _case("batch_96", "batch", 40, meshes=96),
        # edge relations of a large mesh
        _case("edges_5m", "relations", 96, build="TE,EV,VE,EE"),
        # face relations and what is derived from them
        _case("faces_2m", "relations", 72, build="TF,FV,VF,FT,FE,ET,EF,FF"),
        # what a served request asks for next: the cells at each vertex and
        # each cell's neighbours
        _case("followup_2m", "relations", 64, split=0.1, build="VT,TT"),
        # the same on a mesh in file order, where rows lie close together
        _case("followup_grid_1m", "relations", 57, order="grid", split=0.05, build="VT,TT"),
        # every relation and the critical points of a middle-sized mesh with
        # its cells in random order and its vertices in grid order
        _case("all_216k", "relations", 33, order="cells", scalar="gaussians",
              build=",".join(RELATIONS) + ",classes"),
    ]


def _side(rng, lo, hi):
    return int(math.floor(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))


def draw(rng):
    kind = rng.choice(["request", "field", "field", "field", "buffers", "batch", "relations",
                       "relations", "relations"])
    scalar = rng.choice(["uniform", "gaussians", "sines"])
    f64 = rng.random() < 0.3
    split = round(rng.uniform(0.02, 0.15), 3) if rng.random() < 0.5 else 0.0
    order = rng.choice(["permuted", "permuted", "grid", "cells", "vertices"])
    if kind == "request":
        return _case("", kind, _side(rng, 6, 48), order, scalar, f64, split)
    if kind == "field":
        return _case("", kind, _side(rng, 8, 110), order, scalar, f64, split,
                     rng.choice([0, 0, 4, 16]))
    if kind == "buffers":
        return _case("", kind, _side(rng, 6, 50), order, scalar, f64)
    if kind == "batch":
        return _case("", kind, rng.randint(20, 40), "permuted", "uniform", False,
                     meshes=_side(rng, 8, 96))
    build = rng.choice(["TE,EV,VE", "EE", "TF,VF", "TF,FV,FT,FE,ET,EF,FF", "VT,TT", "VT,TT", "VT",
                        "all"])
    if build == "all":
        return _case("", kind, _side(rng, 12, 40), order, scalar, f64, split,
                     build=",".join(RELATIONS) + ",classes")
    # without a field, the seed has to reach the cells: a random order or splits
    if order == "grid" and not split:
        split = 0.05
    return _case("", kind, _side(rng, 12, 72), order, "uniform", False, split, build=build)


def _sides(case):
    """The batch's grid sides, spread over [6, n] by their logarithm."""
    k, n = case["meshes"], case["n"]
    return [int(math.exp(math.log(6) + (math.log(n + 0.99) - math.log(6)) * (i + 0.5) / k))
            for i in range(k)]


def _mesh(case, n, seed):
    # which cells are split decides how large TT and EE get: for relations the
    # splits are the case's own, and the seed gives the order of what is there
    fixed = case["kind"] == "relations" and case["split"] > 0
    shuffled = {"permuted": (True, True), "grid": (False, False), "cells": (False, True),
                "vertices": (True, False)}[case["order"]]
    vertices, cells = (False, False) if fixed else shuffled
    m = tetra.kuhn(n, seed=n if fixed else seed, permute_vertices=vertices, permute_cells=cells,
                   split_fraction=case["split"], n_hubs=case["hubs"],
                   hub_splits=HUB_SPLITS if case["hubs"] else 0, scalar=case["scalar"])
    if fixed:
        _reorder(m, *shuffled, np.random.default_rng(seed))
    return m


def _reorder(m, vertices, cells, rng):
    """Random vertex ids and / or cell order; with neither, 16 pieces of the
    file in random order, as several writers leave them."""
    if vertices:
        ids = rng.permutation(m.n_points).astype(np.int32)
        m.cells = np.sort(ids[m.cells], axis=1)
        m.scalars = m.scalars[np.argsort(ids)]
    if cells:
        m.cells = m.cells[rng.permutation(m.n_cells)]
    if not vertices and not cells:
        pieces = np.array_split(m.cells, 16)
        m.cells = np.concatenate([pieces[i] for i in rng.permutation(len(pieces))])


def _on_gpu(case, mesh):
    dt = torch.float64 if case["f64"] else torch.float32
    return (torch.from_numpy(mesh.cells).cuda(), torch.from_numpy(mesh.scalars).to(dt).cuda())


def prepare(case, seed):
    tetra.init(0)
    tuning.load()
    s = {"case": case}
    if case["kind"] == "batch":
        meshes = [_mesh(case, n, seed * 1009 + i) for i, n in enumerate(_sides(case))]
        s["batch"] = tetra.Batch([(m.cells, m.n_points, m.scalars) for m in meshes])
        s["batch"].use_graph(True)
        return s
    mesh = _mesh(case, case["n"], seed)
    s["V"], s["T"] = mesh.n_points, mesh.n_cells
    if case["kind"] == "request":
        s["cells"] = mesh.cells
        s["scalars"] = mesh.scalars.astype(np.float64 if case["f64"] else np.float32)
        return s
    s["cells"], s["scalars"] = _on_gpu(case, mesh)
    if case["kind"] == "field":
        s["mesh"] = tetra.Mesh(s["cells"].data_ptr(), s["V"], s["scalars"].data_ptr(),
                               on_device=True, n_cells=s["T"], scalars_f64=case["f64"])
    elif case["kind"] == "buffers":
        V, T = s["V"], s["T"]
        s["vv_off"] = torch.zeros(V + 1, dtype=torch.int32, device="cuda")
        s["vv_cols"] = torch.zeros(min(12 * T, V * (V - 1)), dtype=torch.int32, device="cuda")
        s["classes"] = torch.zeros((V, 3), dtype=torch.int32, device="cuda")
        s["status"] = torch.zeros(1, dtype=torch.int32, device="cuda")
    return s


class _DeviceArray:
    """Memory of the library as torch sees it, without a copy."""

    def __init__(self, ptr, shape, typestr):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": typestr,
                                         "strides": None, "version": 2}


def _view(ptr, shape, typestr="<i4"):
    if 0 in shape:
        return torch.zeros(shape, dtype=torch.int64 if typestr == "<i8" else torch.int32)
    return torch.as_tensor(_DeviceArray(ptr, shape, typestr), device="cuda")


def _relation(mesh, name):
    """A built relation's offsets (None for fixed-width ones) and values on the GPU."""
    sh = mesh.shape(name)
    off, off_bytes, val = mesh.relation_device(name)
    o = _view(off, (sh["rows"] + 1,), "<i8" if off_bytes == 8 else "<i4") if off else None
    return o, _view(val, (sh["nnz"], sh["width"]))


def _classes(mesh):
    p = ctypes.c_void_p()
    _native.check(_native.hip().tg_classes_device(mesh.handle, ctypes.byref(p)))
    return _view(p.value, (mesh.n_points, 3))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "field":
        m = state["mesh"]
        m.vv_critpoints()
        return {"VV": _relation(m, "VV"), "classes": _classes(m)}
    if kind == "request":
        with tetra.Mesh(state["cells"], state["V"], state["scalars"]) as m:
            m.vv_critpoints()
            return {"classes": m.classes(), "VV": m.relation("VV")}
    if kind == "buffers":
        # calls share the library's scratch array, so all of them go through
        # one stream, as the entry point asks
        _native.check(_native.hip().tg_vv_critpoints_noalloc(
            state["cells"].data_ptr(), state["T"], state["V"], state["scalars"].data_ptr(),
            int(case["f64"]), state["vv_off"].data_ptr(), state["vv_cols"].data_ptr(),
            state["vv_cols"].numel(), state["classes"].data_ptr(), state["status"].data_ptr(),
            torch.cuda.current_stream().cuda_stream))
        return {k: state[k] for k in ("vv_off", "vv_cols", "classes", "status")}
    if kind == "batch":
        state["batch"].vv_critpoints()
        return {"classes": state["batch"].classes()}
    # relations: the last pass's mesh is let go, as a program that goes
    # through many meshes does
    last = state.pop("mesh", None)
    if last is not None:
        last.close()
    names = case["build"].split(",")
    with_classes = "classes" in names
    m = tetra.Mesh(state["cells"].data_ptr(), state["V"],
                   state["scalars"].data_ptr() if with_classes else None, on_device=True,
                   n_cells=state["T"], scalars_f64=case["f64"])
    state["mesh"] = m
    names = [k for k in names if k != "classes"]
    m.build(tetra.flags(*names))
    if with_classes:
        m.critpoints()
    out = {k: _relation(m, k) for k in names}
    if with_classes:
        out["classes"] = _classes(m)
    return out


def _sizes(n, split, hubs):
    """V, T, E, F of a grid: each 1 -> 4 split adds a vertex, 3 cells, 4 edges, 6 faces."""
    s = round(split * 6 * n ** 3) + hubs * HUB_SPLITS
    return ((n + 1) ** 3 + s, 6 * n ** 3 + 3 * s, 7 * n ** 3 + 9 * n ** 2 + 3 * n + 4 * s,
            12 * n ** 3 + 6 * n ** 2 + 6 * s)


def work(case):
    sides = _sides(case) if case["kind"] == "batch" else [case["n"]]
    total = 0
    for n in sides:
        V, T, E, F = _sizes(n, case["split"], case["hubs"])
        scal = (8 if case["f64"] else 4) * V
        # bytes of each result, offsets included.  TT and EE of an interior
        # cell and edge: 69 cells, 26 edges.
        size = {"TE": 24 * T, "EV": 8 * E, "VE": 4 * (V + 1) + 8 * E, "ET": 8 * (E + 1) + 24 * T,
                "TF": 16 * T, "FV": 12 * F, "VF": 4 * (V + 1) + 12 * F, "FE": 24 * F, "FT": 8 * F,
                "EF": 8 * (E + 1) + 12 * F, "VT": 4 * (V + 1) + 16 * T, "TT": 8 * (T + 1) + 276 * T,
                "FF": 8 * (F + 1) + 48 * T, "EE": 8 * (E + 1) + 104 * E,
                "VV": 4 * (V + 1) + 8 * E, "classes": 12 * V}
        if case["kind"] == "relations":
            names = case["build"].split(",")
            total += 16 * T + (scal if "classes" in names else 0) + sum(size[k] for k in names)
        elif case["kind"] == "batch":
            total += 16 * T + scal + size["VV"] + size["classes"]
        else:
            total += 16 * T + scal + size["VV"] + size["classes"]
    return {"bytes": total, "flops": 0}
