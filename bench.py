"""Benchmark: Galerkin GEP assembly throughput on one MI355X.

Workload (default): the 64x32 waveguide ([0,1]x[0,0.5], 64x32 quads, orders
(6,6), two levels of T refinement on a seeded random 25 % of the leaves per
level, HierPoly, 8x8 Gauss points) - 7784 Elems, 445380 DoFs.

A step is one full assembly (galerkin_sample_gep_hcurl semantics) from the
device-resident flattened Domain to the device-resident upper-triangular CSR
of A and B: elem geometry, DoF signatures, row groups, Gram tables, row
lengths, row_ptr scan and the entry fill. `value` is stored upper-triangular
nonzeros per second (the length of the reference's BTreeMap per second).

Prints one JSON line. The timed steps replay the library's recorded HIP
graphs. `roofline` covers the entry-fill kernel k_fill_flat (the dominant
one): achieved = algorithmic bytes (20 B per stored entry: 4 B column + 8 B A
+ 8 B B) / its duration, measured with HIP events recorded on the assembly
stream around the kernel in the same number of kernel-by-kernel steps;
`traffic` is the HBM bytes per launch from the committed rocprofv3 counter
summary of that kernel. `host_boundary` times the drop-in entry point with
host arrays on both sides. `domain_build` times the host Domain construction
from the workload's Mesh, data-parallel and sequential. `eigensolve` times the
dense GPU eigensolves of assembled GEPs (with LAPACK on the host beside them);
`petsc_writer` the PETSc AIJ files of the assembled GEP (with the oracle's writer
beside it); `fields` the field evaluation over every leaf of the Domain; `sparse_eigensolve`
the sparse shift-invert eigensolve of the workload's GEP near the TE10 cutoff;
`other_workloads` the assembly of the hp-irregular (KOL, 1.78 M DoFs) and 256-guide
configurations at full size, each with its fill roofline and chunk size.
`cpu_baseline` times the oracle (the C++
restatement of the reference algorithm) on a bounded sample of the same
workload on the host cores. `mixed_precision` repeats the measurement with the values
stored in the mixed modes (FP32: 12 B per stored entry; FP32R: FP32 plus a 16-bit residual,
16 B) and states their largest relative entry errors against the FP64 values of the whole
matrix. `assembly_roofline` sets the whole assembly's device time against the output bytes.
"""

from __future__ import annotations

import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "GEP assembly nonzeros/s: mixed-prec vs FP64 GPU at stated rel err; CPU ref"
HBM_PEAK_GBS = 8000.0
BYTES_PER_ENTRY = 20  # col (4) + A (8) + B (8)
# the fill's Gram library placement (fem2d_timing.fill_lib_lds)
FILL_PLACEMENT = {0: "global", 1: "lds"}


def build_workload(name: str):
    from fem_2d_amd import workloads as W

    if name == "waveguide_64x32":
        return W.waveguide_64x32()
    if name == "waveguide_small":
        return W.waveguide_small()
    if name == "precision_study":
        return W.precision_study()
    if name == "hp_irregular":
        return W.hp_irregular()
    if name == "many_waveguides":
        return W.many_waveguides()
    raise SystemExit(f"unknown workload {name}")


def cpu_baseline(w, total_pairs: int, nnz: int, target_s: float):
    """Oracle on the first elems of the same Domain (all host threads up to 16);
    scaled to the full workload through its element-pair count."""
    import oracle

    threads = max(1, min(16, os.cpu_count() or 1))
    n_elems = w.domain.mesh.num_elems
    limit = 64
    while True:
        t0 = time.perf_counter()
        rc, res = oracle.assemble(w.domain.view(), basis=w.basis.code, glq=w.glq, n_threads=threads,
                                  elem_limit=limit)
        dt = time.perf_counter() - t0
        if rc != 0:
            raise RuntimeError(f"oracle failed: {rc}")
        if dt >= target_s or limit >= n_elems:
            break
        limit = min(n_elems, max(limit * 2, int(limit * target_s / max(dt, 1e-3) * 1.1)))
    pairs_per_s = res.pairs / dt
    est_total_s = total_pairs / pairs_per_s
    return {
        "value": nnz / est_total_s,
        "unit": "nonzeros/s",
        "cores": threads,
        "kind": "port",
        "sample": (f"oracle (C++ restatement of galerkin.rs) over elems [0, {limit}) of {n_elems}: "
                   f"{res.pairs} element pairs in {dt:.2f} s on {threads} threads; scaled by the workload's "
                   f"{total_pairs} element pairs"),
        "pairs_per_s": pairs_per_s,
    }


def profiled_traffic(workload: str):
    """HBM bytes per launch of the fill kernel on this workload, from the committed rocprofv3
    --pmc summary (FETCH_SIZE x2 + WRITE_SIZE x1, calibrated on a 1 GiB copy); None if absent."""
    path = os.path.join(ROOT, "profiles", f"k_fill_flat_{workload}.md")
    try:
        for ln in open(path):
            if ln.startswith("traffic_bytes_per_launch:"):
                return int(ln.split(":", 1)[1].strip())
    except OSError:
        pass
    return None


def _max_rel_errors(g32, g64):
    """Largest relative entry error of the FP32-stored values against the FP64 ones, per matrix,
    with the floor sqrt(|d_r d_c|) of the parity definition (entries that cancel to rounding)."""
    import numpy as np

    rows = g64.rows()
    out = {}
    for name, got, ref in (("A", g32.a_val, g64.a_val), ("B", g32.b_val, g64.b_val)):
        diag = np.zeros(g64.n)
        on = rows == g64.col
        diag[rows[on]] = np.abs(ref[on])
        scale = np.maximum(np.abs(ref), np.sqrt(diag[rows] * diag[g64.col]))
        err = np.abs(got - ref)
        ok = scale > 0
        out[name] = float(np.max(err[ok] / scale[ok])) if ok.any() else 0.0
    return out


def mixed_precision(dd, w, args, nnz: int, ms_fp64: float, fill_fp64_ms: float):
    """The same assembly in the mixed storage modes, FP64 arithmetic in both:
    FEM2D_PRECISION_FP32 (A and B stored as FP32, 12 B per stored entry instead of 20) and
    FEM2D_PRECISION_FP32R (FP32 plus a 16-bit residual per value, 16 B per entry). Timed like the
    FP64 steps (graph replays; the fill kernel kernel by kernel); their values are compared with
    the FP64 GPU values of the whole matrix. The byte ratio bounds the fill's speed-up over FP64
    (20/12 and 20/16), the write-bound kernel's roofline."""
    import numpy as np

    import fem_2d_amd as F

    ctx = dd.ctx

    def step(precision):
        return dd.assemble(w.glq, w.basis, F.CurlCurl, F.L2Inner, precision=precision)

    g64 = dd.download(step(F.FP64))
    out_modes = {}
    for name, prec, bpe, desc in (("fp32", F.FP32, 12, "A and B stored as FP32 (FEM2D_PRECISION_FP32)"),
                                  ("fp32r", F.FP32R, 16, "A and B stored as FP32 plus a 16-bit residual "
                                                          "(FEM2D_PRECISION_FP32R)")):
        for _ in range(args.warmup):
            step(prec)
        ctx.synchronize()
        t0 = time.perf_counter()
        for _ in range(args.steps):
            out = step(prec)
        ctx.synchronize()
        ms = (time.perf_counter() - t0) * 1000.0 / args.steps
        ctx.set_graphs(False)
        step(prec)
        fill_ms = []
        for _ in range(args.steps):
            step(prec)
            fill_ms.append(ctx.last_timing()["fill_kernel_ms"])
        ctx.set_graphs(True)
        gm = dd.download(step(prec))
        assert int(out.nnz) == nnz and gm.nnz == nnz
        fill = float(np.mean(fill_ms))
        achieved = bpe * nnz / (fill * 1e-3) / 1e9
        out_modes[name] = {
            "precision": desc + ", fp64 arithmetic",
            "bytes_per_entry": bpe,
            "value": nnz / (ms * 1e-3),
            "unit": "nonzeros/s",
            "ms_per_step": ms,
            "speedup_vs_fp64": ms_fp64 / ms,
            "fill_kernel_ms": fill,
            "fill_speedup_vs_fp64": fill_fp64_ms / fill,
            "fill_speedup_ceiling": BYTES_PER_ENTRY / bpe,
            "fill_roofline": {"achieved": achieved, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                              "frac": achieved / HBM_PEAK_GBS},
            "max_rel_entry_error_vs_fp64": _max_rel_errors(gm, g64),
        }
    return out_modes


def other_workload(name: str, steps: int = 10, warmup: int = 3):
    """Assembly throughput of another configuration at its full size: the timed graph replays,
    the fill kernel kernel by kernel (its HBM roofline), and its chunk size."""
    import numpy as np

    import fem_2d_amd as F

    w = build_workload(name)
    ctx = F.Context(0)
    dd = F.DeviceDomain(w.domain, ctx)
    step = dd.assembler(w.glq, w.basis, F.CurlCurl, F.L2Inner)

    for _ in range(warmup):
        out = step()
    ctx.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        out = step()
    ctx.synchronize()
    ms = (time.perf_counter() - t0) * 1e3 / steps
    nnz = int(out.nnz)
    total = []
    for _ in range(steps):
        step()
        total.append(ctx.last_timing()["total_ms"])
    ctx.set_graphs(False)
    step()
    fill, describe = [], []
    for _ in range(steps):
        step()
        t = ctx.last_timing()
        fill.append(t["fill_kernel_ms"])
        describe.append(t["count_kernel_ms"])
    ctx.set_graphs(True)
    t = ctx.last_timing()
    fill_ms = float(np.mean(fill))
    dev_ms = float(np.mean(total))
    achieved = BYTES_PER_ENTRY * nnz / (fill_ms * 1e-3) / 1e9
    ctx.close()
    return {"value": nnz / (ms * 1e-3), "unit": "nonzeros/s", "ms_per_step": ms, "n_dofs": int(out.n),
            "nnz_upper": nnz, "glq": list(w.glq), "basis": w.basis.__name__, "large_groups": int(t["n_large"]),
            "fill_chunk": int(t["fill_chunk"]), "fill_placement": FILL_PLACEMENT[int(t["fill_lib_lds"])],
            "device_ms": {"total": dev_ms, "describe_kernel": float(np.mean(describe)), "fill_kernel": fill_ms},
            "roofline": {"kernel": "k_fill_flat", "bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBS,
                         "unit": "GB/s", "frac": achieved / HBM_PEAK_GBS,
                         "algorithmic_bytes_per_launch": BYTES_PER_ENTRY * nnz},
            "assembly_roofline_frac": BYTES_PER_ENTRY * nnz / (dev_ms * 1e-3) / 1e9 / HBM_PEAK_GBS}


def sparse_eigensolve(w):
    """The sparse shift-invert eigensolve (the slepc_solve_gep stand-in) on the workload's
    device-resident GEP near the TE10 cutoff: one call (ordering, block factorisation, iteration);
    beside it, the GPU call and the oracle's ARPACK shift-invert (scipy, host) on the 19 296-DoF
    hp-irregular test GEP."""
    import numpy as np

    import fem_2d_amd as F
    from oracle import eigen as OE
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import cases

    ctx = F.Context(0)
    dd = F.DeviceDomain(w.domain, ctx)
    dev = dd.assemble(w.glq, w.basis)
    t0 = time.perf_counter()
    pair = F.solve_gep_sparse(dev, 10.0, ctx=ctx)
    ms = (time.perf_counter() - t0) * 1e3
    st = ctx.last_eigen_stats()
    out = {"solver": "block-tridiagonal level-set ordering; block Cholesky of A + tau B (rocSOLVER potrf/trtri, "
                     "rocBLAS trsm/syrk; applied by column-dot kernels over the inverse factors and their "
                     "transposes) preconditioning GMRES inside a residual-correction shift-invert iteration; FP64",
           w.name: {"n": int(dev.n), "ms": ms, "eigenvalue": pair.value,
                    "rel_err_vs_te10": abs(pair.value - np.pi ** 2) / np.pi ** 2,
                    "residual": st["residual"], "blocks": st["blocks"], "max_block": st["max_block"],
                    "factor_gb": st["factor_bytes"] / 1e9, "symbolic_ms": st["symbolic_ms"],
                    "factor_ms": st["factor_ms"], "iterate_ms": st["iterate_ms"],
                    "outer_iterations": st["iterations"], "gmres_steps": st["inner_iterations"]}}
    dom, glq = cases.small_hp_irregular()
    dds = F.DeviceDomain(dom, ctx)
    devs = dds.assemble(glq, F.KOLShapeFn)
    F.solve_gep_sparse(devs, 5.0, ctx=ctx)
    devs = dds.assemble(glq, F.KOLShapeFn)
    t0 = time.perf_counter()
    p = F.solve_gep_sparse(devs, 5.0, ctx=ctx)
    gpu_ms = (time.perf_counter() - t0) * 1e3
    A, B = dds.download(dds.assemble(glq, F.KOLShapeFn)).to_scipy()
    t0 = time.perf_counter()
    lam, _ = OE.sparse_solve_gep(A, B, 5.0)
    cpu_ms = (time.perf_counter() - t0) * 1e3
    out["small_hp_irregular"] = {"n": int(A.shape[0]), "gpu_ms": gpu_ms, "eigenvalue": p.value,
                                 "cpu_baseline": {"ms": cpu_ms, "eigenvalue": lam, "cores": 1,
                                                  "kind": "ARPACK shift-invert Lanczos (scipy eigsh, SuperLU)"}}
    ctx.close()
    return out


def host_boundary(w, nnz: int, calls: int = 3):
    """The drop-in entry point with host arrays on both sides: view upload, assembly and the
    CSR download into host memory (PCIe-inclusive)."""
    import ctypes as C

    import fem_2d_amd as F
    from fem_2d_amd import _native as N

    lib = N.load()
    ctx = F.Context(0)
    view = w.domain.view()

    def call():
        out = N.GepCsr()
        F.errors.check(lib.fem2d_galerkin_sample_gep_hcurl(ctx._h, C.byref(view), w.basis.code, F.CurlCurl.code,
                                                           F.L2Inner.code, w.glq[0], w.glq[1], 0, C.byref(out)))
        lib.fem2d_gep_csr_free(C.byref(out))

    call()
    t0 = time.perf_counter()
    for _ in range(calls):
        call()
    dt = (time.perf_counter() - t0) / calls
    ctx.close()
    return {"value": nnz / dt, "unit": "nonzeros/s", "ms_per_call": dt * 1e3,
            "entry_point": "fem2d_galerkin_sample_gep_hcurl (host view in, host CSR out)"}


def domain_build(w, calls: int = 7):
    """Domain construction from the workload's Mesh (Domain::from_mesh, domain.rs:69-159), three
    ways, all giving the same Domain: on the GPU straight into HBM (fem2d_device_domain_from_mesh:
    host flattening of the Mesh, one upload, the kernels, the Domain's derived device fields), and
    on the host data-parallel and sequentially (the reference's construction order; neither
    includes the later upload of the view, ``domain_upload_ms``). Median over `calls` builds, after
    one untimed build of each; each timed build includes freeing the previous one."""
    import fem_2d_amd as F

    mesh = w.domain.mesh
    ctx = F.Context(0)
    out = {}
    for name, build in (("device", lambda: F.DeviceDomain.from_mesh(mesh, F.ContinuityCondition.HCurl, ctx=ctx)),
                        ("parallel", lambda: F.Domain.from_mesh(mesh, F.ContinuityCondition.HCurl)),
                        ("serial", lambda: F.Domain.from_mesh_serial(mesh, F.ContinuityCondition.HCurl))):
        d = build()
        n = d.n_dofs if name == "device" else d.num_dofs
        ts = []
        for _ in range(calls):
            t0 = time.perf_counter()
            del d
            d = build()
            ts.append(time.perf_counter() - t0)
        del d
        out[name + "_ms"] = float(sorted(ts)[len(ts) // 2]) * 1e3
    ctx.close()
    out["n_dofs"] = n
    out["threads"] = min(16, os.cpu_count() or 1)
    out["speedup"] = out["serial_ms"] / out["parallel_ms"]
    out["device_speedup_vs_serial"] = out["serial_ms"] / out["device_ms"]
    out["dofs_per_s"] = n / (out["parallel_ms"] * 1e-3)
    out["device_dofs_per_s"] = n / (out["device_ms"] * 1e-3)
    return out


def petsc_writer(w, calls: int = 2):
    """GEP::print_to_petsc_binary_files (linalg.rs:44-52) from the device-resident GEP of the
    workload: both full symmetric AIJ files (transpose, big-endian words on the device, then the
    file writes) into a temporary directory; the oracle's numpy writer is timed on the host on
    the leading rows' submatrix (about 2 M stored entries)."""
    import shutil
    import tempfile

    import numpy as np

    import fem_2d_amd as F

    ctx = F.Context(0)
    dd = F.DeviceDomain(w.domain, ctx)
    dev = dd.assemble(w.glq)
    tmp = tempfile.mkdtemp(prefix="fem2d_petsc_")
    try:
        os.makedirs(os.path.join(tmp, "tmp"))
        dd.print_to_petsc_binary_files(dev, tmp, "bench")
        t0 = time.perf_counter()
        for _ in range(calls):
            dd.print_to_petsc_binary_files(dev, tmp, "bench")
        ms = (time.perf_counter() - t0) * 1e3 / calls
        nbytes = sum(os.path.getsize(os.path.join(tmp, "tmp", f"bench_{m}.dat")) for m in ("a", "b"))
        g = dd.download(dev)
    finally:
        shutil.rmtree(tmp, ignore_errors=True)
    ctx.close()
    full = 2 * g.nnz - int(np.count_nonzero(g.rows() == g.col))
    out = {"ms_per_call": ms, "file_bytes": nbytes, "GBs": nbytes / (ms * 1e-3) / 1e9,
           "full_entries": full, "entries_per_s": 2 * full / (ms * 1e-3)}
    from oracle import petsc as OP

    rows = g.rows()
    k = int(np.searchsorted(g.row_ptr, 2_000_000))
    sel = (rows < k) & (g.col < k)
    t0 = time.perf_counter()
    OP.aij_binary_bytes(k, rows[sel], g.col[sel], g.a_val[sel])
    OP.aij_binary_bytes(k, rows[sel], g.col[sel], g.b_val[sel])
    cpu_s = time.perf_counter() - t0
    n_sel = int(np.count_nonzero(sel))
    cpu_full = 2 * n_sel - int(np.count_nonzero(rows[sel] == g.col[sel]))
    out["cpu_baseline"] = {"entries_per_s": 2 * cpu_full / cpu_s, "s": cpu_s, "cores": 1, "kind": "port",
                           "sample": f"oracle numpy writer, both matrices of the leading {k} rows' submatrix "
                                     f"({n_sel} stored entries), bytes in memory (no file writes)"}
    return out


def eigensolve(calls: int = 3):
    """Dense eigensolves after the assembly, device-resident GEP in, eigenpair out (rocSOLVER after
    the library's CSR-to-dense kernel): the symmetric-definite solve near the TE10 cutoff on the
    1096-DoF waveguide and the 4496-DoF precision-study matrices, nalgebra_solve_gep on the reference's
    624-DoF problem; the CPU baseline is LAPACK dsygvd (scipy, the oracle's dense solve) on the
    1096-DoF matrices."""
    import numpy as np
    from threadpoolctl import threadpool_limits

    import fem_2d_amd as F
    from fem_2d_amd import workloads as W
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import cases

    ctx = F.Context(0)
    out = {"solver": "dense symmetric-definite: shift-invert inverse iteration on the rocSOLVER dgetrf factors of the "
                     "diagonally scaled A - target B, solved with their inverses (rocBLAS trsm, up to 2048 DoFs) or "
                     "dgetrs, refined against the unfactored matrix (dsygvd when inconclusive); nalgebra: "
                     "dpotrf+dpotri+dgemm+dsyevd; FP64"}

    def timed(fn):
        fn()
        t0 = time.perf_counter()
        for _ in range(calls):
            r = fn()
        return r, (time.perf_counter() - t0) * 1e3 / calls

    for name, w in (("waveguide_1096", W.waveguide_small()), ("precision_study_4496", W.precision_study())):
        dd = F.DeviceDomain(w.domain, ctx)
        dev = dd.assemble(w.glq)
        pair, ms = timed(lambda: F.solve_gep_dense(dev, 10.0, ctx=ctx))
        out[name] = {"n": int(dev.n), "ms": ms, "eigenvalue": pair.value,
                     "rel_err_vs_te10": abs(pair.value - np.pi ** 2) / np.pi ** 2}
        # slepc_solve_gep: the dense solve up to SLEPC_DENSE_LIMIT DoFs, the sparse one beyond
        pair, ms = timed(lambda: F.slepc_solve_gep(dev, 10.0, ctx=ctx))
        out[name]["slepc_solve_gep"] = {"ms": ms, "path": "dense" if dev.n <= F.linalg.SLEPC_DENSE_LIMIT
                                        else "sparse", "rel_err_vs_te10": abs(pair.value - np.pi ** 2) / np.pi ** 2}
        if name == "waveguide_1096":
            from oracle import eigen as OE

            A, B = dd.download(dev).to_dense()
            with threadpool_limits(16):
                t0 = time.perf_counter()
                lam, _ = OE.dense_solve_gep(A, B, 10.0)
                cpu_ms = (time.perf_counter() - t0) * 1e3
            out["cpu_baseline"] = {"ms": cpu_ms, "n": int(dev.n), "threads": min(16, os.cpu_count() or 1),
                                   "kind": "LAPACK dsygvd (scipy)", "eigenvalue": lam,
                                   "speedup": cpu_ms / ms}
    dom, glq = cases.slepc_problem()
    dev = F.DeviceDomain(dom, ctx).assemble(glq)
    pair, ms = timed(lambda: F.nalgebra_solve_gep(dev, 2.64, ctx=ctx))
    out["nalgebra_624"] = {"n": int(dev.n), "ms": ms, "eigenvalue": pair.value}
    pair, ms = timed(lambda: F.solve_gep_dense(dev, 1.475, ctx=ctx))
    out["slepc_problem_624"] = {"n": int(dev.n), "ms": ms, "eigenvalue": pair.value,
                                "abs_err_vs_reference": abs(pair.value - 1.4745880937)}
    ctx.close()
    return out


def fields(w, calls: int = 5, density: int = 8):
    """UniformFieldSpace::xy_fields on the workload's Domain (device-resident Domain, solution and
    field buffers; density x density points per leaf Elem), with the oracle's single-threaded
    restatement timed on the host beside it."""
    import ctypes as C

    import numpy as np

    import fem_2d_amd as F
    from fem_2d_amd import _native as N

    lib = N.load()
    ctx = F.Context(0)
    dd = F.DeviceDomain(w.domain, ctx)
    n_leaves = C.c_int64()
    F.errors.check(lib.fem2d_device_domain_num_leaves(dd._h, C.byref(n_leaves)))
    total = n_leaves.value * density * density
    sol = np.random.default_rng(5).standard_normal(w.domain.num_dofs)
    bufs = [C.c_void_p() for _ in range(3)]
    for b, nbytes in zip(bufs, (8 * sol.size, 8 * total, 8 * total)):
        F.errors.check(lib.fem2d_device_malloc(ctx._h, nbytes, C.byref(b)))
    F.errors.check(lib.fem2d_memcpy_to_device(ctx._h, bufs[0], sol.ctypes.data, 8 * sol.size))

    def call():
        F.errors.check(lib.fem2d_device_xy_fields(ctx._h, dd._h, w.basis.code, density, density, bufs[0], sol.size,
                                                  bufs[1], bufs[2]))

    call()
    t0 = time.perf_counter()
    for _ in range(calls):
        call()
    ms = (time.perf_counter() - t0) * 1e3 / calls
    for b in bufs:
        lib.fem2d_device_free(ctx._h, b)
    ctx.close()
    out = {"leaves": n_leaves.value, "density": density, "points": total, "ms_per_call": ms,
           "points_per_s": total / (ms * 1e-3), "output_GBs": 16 * total / (ms * 1e-3) / 1e9}
    import oracle

    t0 = time.perf_counter()
    rc, _, _ = oracle.xy_fields(w.domain.view(), w.basis.code, (density, density), sol)
    cpu_s = time.perf_counter() - t0
    out["cpu_baseline"] = {"points_per_s": total / cpu_s, "s": cpu_s, "cores": 1, "kind": "port",
                           "sample": "oracle xy_fields over every leaf of the same Domain"}
    return out


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--workload", default="waveguide_64x32")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-host-boundary", action="store_true",
                    help="skip timing the host-array entry point (upload + assembly + download)")
    ap.add_argument("--cpu-seconds", type=float, default=12.0)
    ap.add_argument("--no-eigen", action="store_true", help="skip timing the dense eigensolves")
    ap.add_argument("--no-petsc", action="store_true", help="skip timing the PETSc binary writer")
    ap.add_argument("--no-fields", action="store_true", help="skip timing the field evaluation")
    ap.add_argument("--no-sparse-eigen", action="store_true",
                    help="skip timing the sparse eigensolve of the workload's GEP")
    ap.add_argument("--no-other-workloads", action="store_true",
                    help="skip the hp-irregular and 256-guide assembly measurements")
    ap.add_argument("--no-domain-build", action="store_true",
                    help="skip timing the host Domain construction (parallel and sequential builders)")
    ap.add_argument("--no-mixed", action="store_true",
                    help="skip the FP32-storage (mixed precision) assembly and its error check")
    ap.add_argument("--calibrate-copy", action="store_true",
                    help="run only a plain 1 GiB device copy (for scaling HBM byte counters)")
    args = ap.parse_args()

    if args.calibrate_copy:
        import torch

        n = 1 << 27  # 2^27 doubles = 1 GiB
        src = torch.ones(n, dtype=torch.float64, device="cuda")
        dst = torch.empty_like(src)
        for _ in range(3):
            dst.copy_(src)
        torch.cuda.synchronize()
        print(json.dumps({"copy_bytes_read": n * 8, "copy_bytes_written": n * 8, "launches": 3}), flush=True)
        return

    if args.gpus != 1:
        print(f"bench.py measures one GPU only (asked for {args.gpus}); the assembly shards by base Elem "
              "tree across GPUs by design but no multi-GPU path is built.", file=sys.stderr)
        sys.exit(2)

    import numpy as np

    import fem_2d_amd as F

    w = build_workload(args.workload)
    ctx = F.Context(0)
    # the Domain's upload (host view to HBM, and the device kernels that derive its per-Elem,
    # per-spec and per-DoF fields), once per Domain, outside the timed assemblies: timed on a
    # second upload (the first loads the kernels) and reported beside them
    warm = F.DeviceDomain(w.domain, ctx)
    del warm
    ctx.synchronize()
    t_up = time.perf_counter()
    dd = F.DeviceDomain(w.domain, ctx)
    ctx.synchronize()
    upload_ms = (time.perf_counter() - t_up) * 1e3

    # one foreign call per step (fem2d_assemble_device with its arguments bound once)
    step = dd.assembler(w.glq, w.basis, F.CurlCurl, F.L2Inner)

    for _ in range(args.warmup):
        out = step()
    # every assembly synchronises its stream before returning; the timed region is
    # also bracketed by device-wide synchronisation. Assemblies replay the
    # recorded HIP graphs of the pipeline (the library's default).
    ctx.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        out = step()
    ctx.synchronize()
    t1 = time.perf_counter()
    ms_per_step = (t1 - t0) * 1000.0 / args.steps
    nnz = int(out.nnz)
    n = int(out.n)
    t_last = ctx.last_timing()
    # device time of a graph replay (events around the graph), outside the timed region
    total_ms = []
    for _ in range(args.steps):
        step()
        total_ms.append(ctx.last_timing()["total_ms"])

    # Per-kernel durations: the same steps launched kernel by kernel, with HIP
    # events recorded on the assembly stream right before and after the fill
    # kernel (and the describe kernel).
    ctx.set_graphs(False)
    step()
    fill_ms, count_ms = [], []
    for _ in range(args.steps):
        step()
        t = ctx.last_timing()
        fill_ms.append(t["fill_kernel_ms"])
        count_ms.append(t["count_kernel_ms"])
    ctx.set_graphs(True)
    fill_avg = float(np.mean(fill_ms))
    mixed = None if args.no_mixed else mixed_precision(dd, w, args, nnz, ms_per_step, fill_avg)
    dev_total = float(np.mean(total_ms))

    # element pairs visited by the reference's loops (pattern-independent work count)
    a = w.domain.arrays()
    nbs = np.diff(a["bs_offsets"])
    parent = a["parent"]
    pairs = int(np.sum(nbs * (nbs + 1) // 2))
    # ancestor-descendant pairs: sum over elems of |own specs| * |specs of every ancestor|
    anc_specs = np.zeros(len(parent), dtype=np.int64)
    for e in range(len(parent)):
        p = parent[e]
        s = 0
        while p >= 0:
            s += nbs[p]
            p = parent[p]
        anc_specs[e] = s
    pairs += int(np.sum(nbs * anc_specs))

    achieved = BYTES_PER_ENTRY * nnz / (fill_avg * 1e-3) / 1e9
    line = {
        "metric": METRIC,
        "value": nnz / (ms_per_step * 1e-3),
        "unit": "nonzeros/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms_per_step,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic",
        "config": {
            "workload": w.name,
            "n_elems": int(a["n_elems"]),
            "n_dofs": n,
            "nnz_upper": nnz,
            "element_pairs": pairs,
            "glq": list(w.glq),
            "basis": w.basis.__name__,
            "precision": "fp64",
            "large_groups": int(t_last["n_large"]),
            "fill_chunk": int(t_last["fill_chunk"]),
            "fill_placement": FILL_PLACEMENT[int(t_last["fill_lib_lds"])],
        },
        "element_pairs_per_s": pairs / (ms_per_step * 1e-3),
        "domain_upload_ms": upload_ms,
        "device_ms": {"total": dev_total, "describe_kernel": float(np.mean(count_ms)),
                      "fill_kernel": fill_avg},
        # the whole assembly (every launch of the recorded graph) against the same output bytes
        "assembly_roofline": {"achieved": BYTES_PER_ENTRY * nnz / (dev_total * 1e-3) / 1e9, "peak": HBM_PEAK_GBS,
                              "unit": "GB/s",
                              "frac": BYTES_PER_ENTRY * nnz / (dev_total * 1e-3) / 1e9 / HBM_PEAK_GBS},
        "roofline": {
            "kernel": "k_fill_flat",
            "bound": "hbm",
            "achieved": achieved,
            "peak": HBM_PEAK_GBS,
            "unit": "GB/s",
            "frac": achieved / HBM_PEAK_GBS,
            "traffic": None,
            "algorithmic_bytes_per_launch": BYTES_PER_ENTRY * nnz,
        },
    }
    line["roofline"]["traffic"] = profiled_traffic(w.name)
    if mixed is not None:
        line["mixed_precision"] = mixed
    if not args.no_host_boundary:
        line["host_boundary"] = host_boundary(w, nnz)
    if not args.no_domain_build:
        line["domain_build"] = domain_build(w)
    if not args.no_eigen:
        line["eigensolve"] = eigensolve()
    if not args.no_petsc:
        line["petsc_writer"] = petsc_writer(w)
    if not args.no_fields:
        line["fields"] = fields(w)
    if not args.no_sparse_eigen:
        line["sparse_eigensolve"] = sparse_eigensolve(w)
    if not args.no_other_workloads and w.name == "waveguide_64x32":
        line["other_workloads"] = {name: other_workload(name) for name in ("hp_irregular", "many_waveguides")}
    if not args.no_cpu_baseline:
        line["cpu_baseline"] = cpu_baseline(w, pairs, nnz, args.cpu_seconds)
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
