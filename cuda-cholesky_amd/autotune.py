#!/usr/bin/env python3
"""Measure the tunable schedule parameters of the library on this GPU.

* Outer block size of the blocked factorisations: for every precision (D:
  cuDpotrf, Z: cuZpotrf, S: cuSpotrf, B: the BF16 factor of cuDsposvx) and
  every order in the sweep, each candidate block size is set with
  cuLAPACKSetBlockSize and the factorisation timed (median of a few runs, the
  candidates interleaved, fresh input each time).  The winner for each order
  covers all n up to it.
* Tile choice of each GEMM kernel family: a launch takes the family's larger
  tile when it has at least `min_tiles` of them.  Each candidate threshold is
  set through $CUCHOLESKY_TILE_MIN_<family> (read by the library on every
  launch) and a factorisation that uses the family is timed at several orders;
  the threshold with the least total time wins, among those that cost no
  product of PRODUCTS more than 3 % over the library's present threshold (the
  products use the same threshold; those fill the chip with whole rounds of the
  larger tile, where it is at its best).  Families: D (double tile kernel, 128
  vs 64: cuDpotrf), Z (complex, 64 vs 32: cuZpotrf), S (FP32 kernel, 128 vs 64:
  cuSpotrf), H and W (16-bit kernel, 128 vs 64 and 256 vs 128: the FP16-product
  factor of cuDsposvx).  A threshold above any launch's tile count means "always
  the smaller tile".
* Workgroup cap of the factorisation's late trailing updates: a trailing
  update of order t <= t_max runs on at most `workgroups` workgroups, each
  taking several tiles, so that the look-ahead chain (diagonal blocks and
  panel products on the other stream) finds free room on the CUs.  Each
  candidate (t_max, workgroups) is set through
  $CUCHOLESKY_TRAILING_CAP_<precision> and the factorisation timed
  (median of a few runs, candidates interleaved, since the differences are
  about 1-2 %).

The table goes to tuning.txt beside the library (or --out), where the library
reads it at first use:

    potrf_nb <precision> <n_max> <nb>
    gemm_tile <family> <min_tiles>
    trailing_cap <precision> <t_max> <workgroups>

    python cuda-cholesky_amd/autotune.py [--quick] [--only nb|tiles|cap] [--out PATH]
"""
import argparse
import importlib.util
import os
import sys
import time

HERE = os.path.dirname(os.path.abspath(__file__))

SWEEP = {
    # precision: (orders, candidate block sizes)
    "D": ([1024, 2048, 4096, 6144, 8192, 12288, 16384, 32768], [256, 384, 512, 768, 1024, 1536]),
    "Z": ([1024, 2048, 4096, 8192], [128, 192, 256, 384, 512, 768]),
    "S": ([2048, 4096, 6144, 8192, 16384, 32768], [384, 512, 768, 1024, 1536]),
    "B": ([4096, 8192, 16384, 32768], [384, 512, 768, 1024]),
}
QUICK = {
    "D": ([4096, 16384], [256, 384, 512]),
    "Z": ([4096], [128, 256]),
    "S": ([8192], [384, 768]),
    "B": ([8192], [384, 768]),
}


def package():
    name = "cuda_cholesky_amd"
    if name in sys.modules:
        return sys.modules[name]
    spec = importlib.util.spec_from_file_location(name, os.path.join(HERE, "__init__.py"))
    mod = importlib.util.module_from_spec(spec)
    sys.modules[name] = mod
    spec.loader.exec_module(mod)
    return mod


def spd(torch, n, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    if dtype == torch.complex128:
        H = torch.complex(torch.randn(n, n, generator=g, device="cuda", dtype=torch.float64),
                          torch.randn(n, n, generator=g, device="cuda", dtype=torch.float64))
        A = H @ H.conj().T / n
    else:
        G = torch.randn(n, n, generator=g, device="cuda", dtype=torch.float64)
        A = G @ G.T / n
    A.diagonal().add_(1.0)
    return A.to(dtype) if dtype != torch.complex128 else A


def time_one(torch, pkg, h, prec, n, A0, B):
    A = A0.clone()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    if prec == "D":
        st, info = pkg.cuDpotrf(h, pkg.Lower, n, pkg.ptr(A), n)
    elif prec == "Z":
        st, info = pkg.cuZpotrf(h, pkg.Upper, n, pkg.ptr(A), n)
    elif prec == "S":
        st, info = pkg.cuSpotrf(h, pkg.Lower, n, pkg.ptr(A), n)
    else:  # the solve with BF16 (B) or FP16 (H) products
        X = torch.zeros_like(B)
        st, _, used, info = pkg.cuDsposvx(h, pkg.Lower, n, B.shape[0], pkg.ptr(A), n, pkg.ptr(B), n,
                                          pkg.ptr(X), n, prec, "I")
    torch.cuda.synchronize()
    dt = time.perf_counter() - t0
    if st != 0 or info != 0:
        raise RuntimeError(f"{prec} n={n}: status {st} info {info}")
    return dt


def medians(torch, pkg, h, prec, n, A0, B, cands, choose, reps):
    """Median time per candidate; choose(c) makes c the one that runs.  One
    untimed run each (workspace, warm-up), then reps rounds of all in turn."""
    times = {c: [] for c in cands}
    for r in range(reps + 1):
        for c in cands:
            choose(c)
            t = time_one(torch, pkg, h, prec, n, A0, B)
            if r > 0:
                times[c].append(t)
    return {c: sorted(v)[len(v) // 2] for c, v in times.items()}


def tune_nb(torch, pkg, h, sweep, reps):
    """potrf_nb lines."""
    lines = []
    for prec, (orders, cands) in sweep.items():
        dtype = {"D": torch.float64, "Z": torch.complex128, "S": torch.float32, "B": torch.float64}[prec]
        for i, n in enumerate(orders):
            A0 = spd(torch, n, dtype, seed=n)
            B = torch.randn(4, n, device="cuda", dtype=torch.float64) if prec == "B" else None

            def choose(nb):
                assert pkg.cuLAPACKSetBlockSize(h, prec, nb) == 0

            times = medians(torch, pkg, h, prec, n, A0, B, [c for c in cands if c <= n], choose, reps)
            choose(0)
            best = min(times, key=times.get)
            n_max = n if i + 1 < len(orders) else 1 << 40
            detail = " ".join(f"{nb}:{t * 1e3:.3f}ms" for nb, t in times.items())
            lines.append(f"potrf_nb {prec} {n_max} {best}   # n={n} {detail}")
            print(lines[-1], flush=True)
            del A0, B
            torch.cuda.empty_cache()
    return lines


def use_measured(pkg, h, routine, n, lines):
    """Order n takes the block size and the families the tile thresholds that
    `lines` (the sweeps just run) give them; without any, the library's own table
    decides."""
    for ln in lines:
        if ln.startswith("gemm_tile "):
            os.environ[f"CUCHOLESKY_TILE_MIN_{ln.split()[1]}"] = ln.split()[2]
    prec = "B" if routine == "H" else routine
    fields = [ln.split() for ln in lines if ln.startswith(f"potrf_nb {prec} ")]
    nb = next((int(f[3]) for f in fields if n <= int(f[2])), 0)
    assert pkg.cuLAPACKSetBlockSize(h, prec, nb) == 0


# family: (routine, orders, candidate thresholds); 1 << 30: never the larger tile
TILE_SWEEP = {
    "D": ("D", [4096, 8192, 16384], [120, 240, 480, 960, 1920, 1 << 30]),
    "Z": ("Z", [2048, 4096, 8192], [120, 240, 480, 960, 1440, 1920, 2880, 1 << 30]),
    "S": ("S", [4096, 8192, 16384], [60, 120, 240, 480, 1 << 30]),
    "H": ("H", [8192, 16384], [120, 240, 480, 1 << 30]),
    "W": ("H", [16384, 32768], [128, 256, 512, 1024, 1 << 30]),
}
TILE_QUICK = {
    "D": ("D", [8192], [120, 240, 1 << 30]),
    "W": ("H", [16384], [256, 512, 1 << 30]),
}


# products (m, n, k) of exactly one and two rounds of two workgroups per CU
PRODUCTS = {"D": [(8192, 1024, 4096), (4096, 4096, 1024)], "Z": [(2048, 1024, 1024), (2048, 2048, 1024)]}


def time_product(torch, pkg, hb, fam, m, n, k):
    dtype = torch.float64 if fam == "D" else torch.complex128
    A, B, D = (torch.randn(s, device="cuda", dtype=dtype) for s in (m * k, k * n, m * n))
    gemm = pkg.cuDgemm2 if fam == "D" else pkg.cuZgemm2
    stream = torch.cuda.current_stream().cuda_stream
    best = float("inf")
    for _ in range(5):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(10):
            assert gemm(hb, pkg.NoTrans, pkg.NoTrans, m, n, k, 1.0, pkg.ptr(A), m, pkg.ptr(B), k, 0.0, 0, m,
                        pkg.ptr(D), m, stream) == 0
        torch.cuda.synchronize()
        best = min(best, (time.perf_counter() - t0) / 10)
    return best


def tune_tiles(torch, pkg, h, sweep, reps, measured):
    """gemm_tile lines."""
    lines = []
    for fam, (routine, orders, cands) in sweep.items():
        dtype = {"D": torch.float64, "Z": torch.complex128, "S": torch.float32, "H": torch.float64}[routine]
        total = {c: 0.0 for c in cands}
        detail = []
        for n in orders:
            A0 = spd(torch, n, dtype, seed=n)
            B = torch.randn(4, n, device="cuda", dtype=torch.float64) if routine == "H" else None
            var = f"CUCHOLESKY_TILE_MIN_{fam}"
            use_measured(pkg, h, routine, n, measured)

            def choose(c):
                os.environ[var] = str(c)

            times = medians(torch, pkg, h, routine, n, A0, B, cands, choose, reps)
            os.environ.pop(var, None)
            row = []
            for c, t in times.items():
                total[c] += t
                row.append(f"{'never' if c >= 1 << 30 else c}:{t * 1e3:.2f}ms")
            detail.append(f"n={n} " + " ".join(row))
            del A0, B
            torch.cuda.empty_cache()
        for m, w, k in PRODUCTS.get(fam, []):
            with pkg.BLASHandle() as hb:
                limit = 1.03 * time_product(torch, pkg, hb, fam, m, w, k)
                row = []
                for c in cands:
                    choose(c)
                    t = time_product(torch, pkg, hb, fam, m, w, k)
                    row.append(f"{'never' if c >= 1 << 30 else c}:{t * 1e3:.3f}ms")
                    if t > limit:
                        total.pop(c, None)
                os.environ.pop(var, None)
            detail.append(f"{m}x{w}x{k} " + " ".join(row))
        best = min(total, key=total.get)
        lines.append(f"gemm_tile {fam} {best}   # {'; '.join(detail)}")
        print(lines[-1], flush=True)
    return lines


# precision: (order, candidate (t_max, workgroups) pairs; (0, 0) = no cap)
CAP_SWEEP = {
    "D": (16384, [(0, 0), (8192, 384), (8192, 448), (12288, 448), (16384, 448), (16384, 480)]),
    "Z": (8192, [(0, 0), (8192, 384), (8192, 448)]),
}
CAP_QUICK = {"D": (16384, [(0, 0), (12288, 448)])}


def tune_cap(torch, pkg, h, sweep, reps, measured):
    """trailing_cap lines: per precision, the candidate with the least median
    time."""
    lines = []
    for prec, (n, cands) in sweep.items():
        dtype = {"D": torch.float64, "Z": torch.complex128}[prec]
        A0 = spd(torch, n, dtype, seed=n)
        var = f"CUCHOLESKY_TRAILING_CAP_{prec}"
        use_measured(pkg, h, prec, n, measured)

        def choose(c):
            os.environ[var] = f"{c[0]}:{c[1]}"

        med = medians(torch, pkg, h, prec, n, A0, None, cands, choose, reps)
        os.environ.pop(var, None)
        best = min(med, key=med.get)
        detail = " ".join(f"{c[0]}:{c[1]}:{t * 1e3:.2f}ms" for c, t in med.items())
        if best[1] > 0:
            lines.append(f"trailing_cap {prec} {best[0]} {best[1]}   # n={n} median {detail}")
        else:
            lines.append(f"# trailing_cap {prec}: no cap   # n={n} median {detail}")
        print(lines[-1], flush=True)
        del A0
        torch.cuda.empty_cache()
    return lines


def main():
    ap = argparse.ArgumentParser(description=__doc__, formatter_class=argparse.RawDescriptionHelpFormatter)
    ap.add_argument("--quick", action="store_true", help="a reduced sweep (a minute or two)")
    ap.add_argument("--reps", type=int, default=5)
    ap.add_argument("--out", default=os.path.join(HERE, "tuning.txt"))
    ap.add_argument("--only", choices=["nb", "tiles", "cap"], help="run one of the sweeps")
    args = ap.parse_args()
    import torch
    pkg = package()
    pkg.lib()
    h = pkg.LAPACKHandle()
    sweep = QUICK if args.quick else SWEEP
    lines = ["# schedule parameters measured by autotune.py on " + torch.cuda.get_device_name(0),
             "# potrf_nb <precision> <n_max> <nb>   (milliseconds per candidate in the trailing comment)",
             "# gemm_tile <family> <min_tiles>   (milliseconds per order and candidate in the trailing comment)",
             "# trailing_cap <precision> <t_max> <workgroups>   (median milliseconds per candidate in the trailing comment)"]
    if args.only in (None, "nb"):
        lines += tune_nb(torch, pkg, h, sweep, args.reps)
    if args.only in (None, "tiles"):
        lines += tune_tiles(torch, pkg, h, TILE_QUICK if args.quick else TILE_SWEEP, args.reps, lines)
    if args.only in (None, "cap"):
        lines += tune_cap(torch, pkg, h, CAP_QUICK if args.quick else CAP_SWEEP, args.reps + 4, lines)
    h.close()
    if args.only is not None and os.path.exists(args.out):
        # keep the entries of the sweeps that did not run
        ran = {"nb": "potrf_nb", "tiles": "gemm_tile", "cap": "trailing_cap"}[args.only]
        with open(args.out) as f:
            lines += [ln.rstrip("\n") for ln in f
                      if not ln.startswith("#") and not ln.startswith(ran) and ln.strip()]
    with open(args.out, "w") as f:
        f.write("\n".join(lines) + "\n")
    print(f"wrote {args.out}", flush=True)


if __name__ == "__main__":
    main()
