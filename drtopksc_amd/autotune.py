"""Autotuner of the batched form: picks alpha and the delegate-pass tile per
(ceil log2 n, ceil log2 k) cell and writes the table drtopk_batch_plan takes.

    python -m drtopksc_amd.autotune --out drtopksc_amd/tuning/mi355x.json

For every key type (uint32 uniform, float32 N(0,1): the two row kinds of the batched workload,
whose keys spread differently over the radix digits) and every cell in the batched workload's
range (n 2^12..2^22, k 1..4096) it builds a batch of `rows` rows of that type whose n and k fall
in that cell, times drtopk_select_batched (HIP events on the launch stream, median of `reps`)
for each candidate, checks that every candidate returns the same outputs, and keeps the fastest.
Candidates: alpha in policy-2 .. policy+2 (the planner lowers invalid ones), tiles of 2^13 or
2^15 keys.  Rows of one cell share a batch, so a cell's time is its throughput when batched with its
own kind.

The result is JSON: {"device": ..., "cells": [[dtype, log2n, log2k, alpha, digit_bits, tile_log2], ...]};
drtopksc_amd.tuning_from_table() turns it into a drtopk_tuning, and

    python -m drtopksc_amd.autotune --emit-c drtopksc_amd/tuning/mi355x.json

writes csrc/tuning_table.inc, the library's built-in table (drtopk_tuning_default).

The single-vector table (alpha DRTOPK_ALPHA_TUNED of drtopk_select) is tuned and emitted with

    python -m drtopksc_amd.autotune --single          # -> tuning/mi355x_single.json
    python -m drtopksc_amd.autotune --emit-c-single drtopksc_amd/tuning/mi355x_single.json
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time


DIGIT_BITS = 8  # of every cell: no kernel of the batched form depends on it


def policy_alpha(n: int, k: int) -> int:
    """The reference's alpha policy (baseline+filter+beta+shuffle/main.cu:83-89)."""
    ln = n.bit_length() - 1
    lk = (k - 1).bit_length()
    return max(0, (ln + 3 - lk) // 2)


def cell_rows(ln: int, lk: int, rows: int, rng, dtype: int):
    """Rows with ceil(log2 n) == ln and ceil(log2 k) == lk (k <= n / 8 when possible), all of
    one key type (0 uint32 uniform, 1 float32 N(0,1))."""
    import numpy as np
    lo_n = (1 << (ln - 1)) + 1
    hi_n = 1 << ln
    out = []
    for i in range(rows):
        n = int(rng.integers(lo_n, hi_n + 1))
        lo_k = 1 if lk == 0 else (1 << (lk - 1)) + 1
        hi_k = 1 << lk
        k = int(rng.integers(lo_k, hi_k + 1))
        out.append((n, min(k, n), dtype))
    return out


def time_batch(dt, torch, rows, buf, keys_len, out_len, tuning, reps):
    b = dt.Batch(rows, keys_len, out_len, tuning=tuning)
    out = b.alloc_out()
    st = torch.cuda.current_stream()
    b.run(buf, out=out, stream=st)
    torch.cuda.synchronize()
    ts = []
    for _ in range(reps):
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record(st)
        b.run(buf, out=out, stream=st)
        e1.record(st)
        e1.synchronize()
        ts.append(e0.elapsed_time(e1))
    ts.sort()
    return ts[len(ts) // 2], out


def emit_c(json_path: str, inc_path: str) -> None:
    """Write the cells of a tuning JSON as the C include compiled into libdrtopk.so."""
    cells = json.load(open(json_path))["cells"]
    lines = ["// Generated by drtopksc_amd/autotune.py --emit-c from " + os.path.basename(json_path) + ".",
             "// {key type (0 uint32, 1 float32), ceil log2 n, ceil log2 k, alpha, digit bits, tile log2} per measured cell.",
             "static const unsigned char kTunedCells[][6] = {"]
    for c in cells:
        lines.append("    {" + ", ".join(str(int(x)) for x in c) + "},")
    lines.append("};")
    with open(inc_path, "w") as f:
        f.write("\n".join(lines) + "\n")


SINGLE_JSON = os.path.join(os.path.dirname(os.path.abspath(__file__)), "tuning", "mi355x_single.json")
SINGLE_INC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "csrc", "single_tuning.inc")


def single_candidates(dt, n: int, k: int):
    """(alpha, beta, params) to time for one cell of the single-vector table, the reference policy first.  All
    name their alpha: a call that leaves it to the library takes a pipeline that the table does not steer."""
    pol = min(policy_alpha(n, k), n.bit_length() - 1)
    out = [(pol, 2 if 0 < pol <= 5 else 1, dt.params(alpha=pol))]
    for a in range(max(1, pol - 2), min(n.bit_length() - 1, pol + 2) + 1):
        for b in ((1, 2, 3, 4) if a <= 5 else (1,)):
            fl = dt.FLAGS_DEFAULT if b > 1 else (dt.FLAG_FILTER | dt.FLAG_SHUFFLE)
            if (a, b) != out[0][:2]:
                out.append((a, b, dt.params(alpha=a, beta=max(b, 2), flags=fl)))
    return out


def tune_single(lns, kmax_log2: int, reps: int, margin: float, out_path: str) -> int:
    """The single-vector table (DRTOPK_ALPHA_TUNED), which the general pipeline follows: for n = 2^ln
    uniform uint32 keys and every k = 2^lk, time drtopk_select (keys + indices out, HIP events, median of `reps`) for alpha in
    policy-2 .. policy+2 and, at alpha <= 5, beta 1 (one delegate) .. 4; every candidate must
    return the reference policy's outputs.  A cell keeps the fastest candidate when it beats the
    policy by more than `margin`, else the policy."""
    import torch

    import drtopksc_amd as dt
    cells, report = [], []
    t_start = time.time()
    st = torch.cuda.current_stream()
    for ln in lns:
        n = 1 << ln
        g = torch.Generator(device="cuda")
        g.manual_seed(ln)
        dev = torch.randint(-2 ** 31, 2 ** 31 - 1, (n,), dtype=torch.int32, device="cuda", generator=g)
        kth = torch.empty(1, dtype=torch.int32, device="cuda")
        okeys = torch.empty(1 << min(kmax_log2, ln), dtype=torch.int32, device="cuda")
        oidx = torch.empty(1 << min(kmax_log2, ln), dtype=torch.int64, device="cuda")
        ws = torch.empty(256, dtype=torch.uint8, device="cuda")
        for lk in range(0, min(kmax_log2, ln - 4) + 1):
            k = 1 << lk
            res = {}
            ref = None
            for a, b, p in single_candidates(dt, n, k):
                try:
                    need = dt.workspace_size(n, k, dt.ALGO_RADIX, dt.U32, p)
                except dt.DrTopKError:
                    continue  # not a valid (alpha, beta) for this (n, k)
                if ws.numel() < need:
                    del ws
                    torch.cuda.empty_cache()
                    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
                o = (kth, okeys[:k], oidx[:k])
                dt.select(dev, k, p=p, workspace=ws, out=o, stats=True)
                got = [x.clone() for x in o]
                if ref is None:
                    ref = got
                elif not all(torch.equal(x, y) for x, y in zip(got, ref)):
                    raise RuntimeError(f"n 2^{ln} k 2^{lk} alpha {a} beta {b}: outputs differ")
                ts = []
                for _ in range(reps):
                    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                    e0.record(st)
                    dt.select(dev, k, p=p, workspace=ws, out=o, stream=st)
                    e1.record(st)
                    e1.synchronize()
                    ts.append(e0.elapsed_time(e1))
                ts.sort()
                res[a, b] = ts[len(ts) // 2]
            pol_key = next(iter(res))  # the policy was timed first
            best = min(res.items(), key=lambda kv: kv[1])
            pick = best[0] if best[1] < res[pol_key] * (1.0 - margin) else pol_key
            cells.append([ln, lk, pick[0], pick[1]])
            report.append({"log2n": ln, "log2k": lk, "policy": list(pol_key), "policy_ms": round(res[pol_key], 4),
                           "best": list(best[0]), "best_ms": round(best[1], 4), "pick": list(pick)})
            print(f"[autotune-single] n 2^{ln} k 2^{lk}: policy {pol_key} {res[pol_key]:.4f} ms, best {best[0]} "
                  f"{best[1]:.4f} ms -> {pick}", flush=True)
        del dev, ws
        torch.cuda.empty_cache()
    props = torch.cuda.get_device_properties(0)
    with open(out_path, "w") as f:
        json.dump({"device": getattr(props, "gcnArchName", props.name), "reps": reps, "margin": margin,
                   "seconds": round(time.time() - t_start, 1), "single": cells, "report": report}, f, indent=1)
    print(f"[autotune-single] wrote {out_path} ({len(cells)} cells)", flush=True)
    return 0


def emit_c_single(json_path: str, inc_path: str) -> None:
    """Write the single-vector cells that differ from the reference policy as the C include."""
    cells = json.load(open(json_path))["single"]
    lines = ["// Generated by drtopksc_amd/autotune.py --emit-c-single from " + os.path.basename(json_path) + ".",
             "// {floor log2 n, ceil log2 k, alpha, beta} where the measured choice differs from the",
             "// reference policy (beta 1: one delegate per subrange; 2..4: the beta path).",
             "static const unsigned char kSingleTuned[][4] = {"]
    kept = 0
    for ln, lk, a, b in cells:
        n, k = 1 << ln, 1 << lk
        pa = policy_alpha(n, k)
        pb = 2 if pa <= 5 else 1
        if (a, b) != (pa, pb):
            lines.append(f"    {{{ln}, {lk}, {a}, {b}}},")
            kept += 1
    if kept == 0:
        lines.append("    {0, 0, 0, 0},  // no cell differs")
    lines.append("};")
    with open(inc_path, "w") as f:
        f.write("\n".join(lines) + "\n")


def main(argv=None):
    ap = argparse.ArgumentParser()
    ap.add_argument("--out", default=os.path.join(os.path.dirname(os.path.abspath(__file__)), "tuning",
                                                  "mi355x.json"))
    ap.add_argument("--rows", type=int, default=96)
    ap.add_argument("--reps", type=int, default=5)
    ap.add_argument("--ln", default="12-22")
    ap.add_argument("--lk", default="0-12")
    ap.add_argument("--emit-c", metavar="JSON", help="only write csrc/tuning_table.inc from a tuning JSON")
    ap.add_argument("--single", action="store_true", help="tune the single-vector table (DRTOPK_ALPHA_TUNED)")
    ap.add_argument("--single-ln", default="16-30", help="log2 n of the single-vector table: a-b or a,b,...")
    ap.add_argument("--single-kmax", type=int, default=24)
    ap.add_argument("--margin", type=float, default=0.02)
    ap.add_argument("--emit-c-single", metavar="JSON", help="only write csrc/single_tuning.inc from a JSON")
    args = ap.parse_args(argv)
    if args.emit_c_single:
        emit_c_single(args.emit_c_single, SINGLE_INC)
        return 0
    if args.single:
        out = args.out if args.out != ap.get_default("out") else SINGLE_JSON
        if "-" in args.single_ln:
            lo, hi = (int(x) for x in args.single_ln.split("-"))
            lns = list(range(lo, hi + 1))
        else:
            lns = [int(x) for x in args.single_ln.split(",")]
        return tune_single(lns, args.single_kmax, args.reps, args.margin, out)
    if args.emit_c:
        emit_c(args.emit_c, os.path.join(os.path.dirname(os.path.abspath(__file__)), "csrc", "tuning_table.inc"))
        return 0
    import numpy as np
    import torch

    import drtopksc_amd as dt
    from drtopksc_amd.workloads import pack

    lns = range(int(args.ln.split("-")[0]), int(args.ln.split("-")[1]) + 1)
    lks = range(int(args.lk.split("-")[0]), int(args.lk.split("-")[1]) + 1)
    rng = np.random.default_rng(1234)
    cells = []
    report = []
    t_start = time.time()
    for dtype in (0, 1):
        for ln in lns:
            for lk in lks:
                if (1 << lk) > (1 << ln) // 8 and lk > 0:
                    continue
                rows_nk = cell_rows(ln, lk, args.rows, rng, dtype)
                rows, keys_len, out_len = pack(rows_nk)
                g = torch.Generator(device="cuda")
                g.manual_seed(ln * 64 + lk)
                if dtype == 0:
                    buf = torch.randint(-2 ** 31, 2 ** 31 - 1, (keys_len,), dtype=torch.int32, device="cuda", generator=g)
                else:
                    buf = torch.randn(keys_len, device="cuda", generator=g).view(torch.int32)
                n_mid = 1 << ln
                k_mid = 1 << lk
                a0 = policy_alpha(n_mid, k_mid)
                best = None
                ref = None
                for a in range(max(0, a0 - 2), a0 + 3):
                    for tl in (13, 15):
                        if a > tl:
                            continue
                        t = dt.tuning_default()
                        t.alpha[dtype][ln][lk] = a
                        t.digit_bits[dtype][ln][lk] = DIGIT_BITS
                        t.tile_log2[dtype][ln][lk] = tl
                        ms, out = time_batch(dt, torch, rows, buf, keys_len, out_len, t, args.reps)
                        if ref is None:
                            ref = [o.clone() for o in out]
                        elif not all(torch.equal(x, y) for x, y in zip(out, ref)):
                            raise RuntimeError(f"cell ({dtype},{ln},{lk}) alpha {a} tile {tl}: outputs differ")
                        if best is None or ms < best[0]:
                            best = (ms, a, DIGIT_BITS, tl)
                cells.append([dtype, ln, lk, best[1], best[2], best[3]])
                report.append({"dtype": dtype, "log2n": ln, "log2k": lk, "policy_alpha": a0, "alpha": best[1],
                               "digit_bits": best[2], "tile_log2": best[3], "ms": round(best[0], 4), "rows": len(rows)})
                print(f"[autotune] {'float32' if dtype else 'uint32'} n~2^{ln} k~2^{lk}: alpha {best[1]} (policy {a0}), "
                      f"{best[2]}-bit digits, tile 2^{best[3]}, {best[0]:.4f} ms for {len(rows)} rows", flush=True)
                del buf
    os.makedirs(os.path.dirname(args.out), exist_ok=True)
    props = torch.cuda.get_device_properties(0)
    with open(args.out, "w") as f:
        json.dump({"device": getattr(props, "gcnArchName", props.name), "rows_per_cell": args.rows,
                   "reps": args.reps, "seconds": round(time.time() - t_start, 1), "cells": cells,
                   "report": report}, f, indent=1)
    print(f"[autotune] wrote {args.out} ({len(cells)} cells)", flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
