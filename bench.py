#!/usr/bin/env python3
"""Headline benchmark: boards/s of the B=4096 16-bit forward on one MI355X.

One "step" is one batched forward of 4096 synthetic positions through the
default-architecture policy/value CNN (inputs and packed weights already in
HBM).  Prints ONE JSON line.  Alongside the headline it reports the fused
kernel's MFMA roofline fraction (HIP-event timing of the kernel launches), the
G=8 grouped-history rate, the other arithmetic modes with their agreement with
the fp32 kernel, the HBM-bound tail kernels, and a CPU baseline (the PyTorch
oracle on the host cores, bounded sample).
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
if str(ROOT) not in sys.path:
    sys.path.insert(0, str(ROOT))

CONV_FLOP_PER_BOARD = 269_554_368        # dense conv count, 2 * 134,777,184 MAC
MFMA_PEAK_TFLOPS = 2500.0                # MI355X dense bf16 / fp16
HBM_PEAK_GBS = 8000.0
# HBM bytes per B=4096 launch of the fused kernel: rocprofv3 --pmc FETCH_SIZE and WRITE_SIZE (one
# run each), scaled by what the same counters read for a 256 MiB copy (x2.00 and x1.00); the
# figures are in profiles/cases_kernel_trace.md (bf16f6: profiles/fused_forward_bf16f6_b4096.md).
TRAFFIC_BYTES = {"bf16c": 51.1e6, "bf16f6": 33.7e6, "bf16": 33.2e6}
# The cascade: every board with plain bf16 layer boundaries, then the boards whose decision is
# closer than the rounding noise again with the low parts of activations (fp6) and weights (bf16)
# carried.  The fastest bf16-MFMA mode that meets the >= 99 % argmax gate, and it meets it with
# margin (99.9 %); its time depends on how many boards go twice, which the line reports.
HEADLINE = "bf16c"


def _lib_names():
    from connect6_amd import _lib
    return _lib.PREC_BY_NAME


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=50)
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--batch", type=int, default=4096)
    ap.add_argument("--precision", default=HEADLINE, choices=["bf16c", "bf16f6w", "bf16f6", "bf16", "fp16", "fp32"])
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-extras", action="store_true", help="headline + roofline only")
    ap.add_argument("--calibrate-copy", action="store_true",
                    help="also launch one plain 256 MiB device copy (reference for rocprof byte counters)")
    args = ap.parse_args()
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py measures one GPU: the forward shards by board with no exchange step, "
              "and this build runs and reports a single MI355X only (use --gpus 1).", file=sys.stderr)
        return 2

    import torch

    import connect6_amd as c6
    from connect6_amd.synthetic import gen_boards, gen_uniform

    dev = torch.device("cuda:0")
    c6.load()
    B, K, W = args.batch, args.steps, args.warmup
    torch.manual_seed(1234)
    model = c6.PolicyValueNet().to(dev).eval()       # reference init (connect6/model.py:83-94)
    x_host, legal_host = gen_boards(B, 200, 2025)
    x = x_host.to(dev)
    legal = legal_host.to(dev)

    def run_mode(prec: str, steps: int, warmup: int):
        """(seconds per step by wall clock, seconds per launch by HIP events)"""
        model.precision = prec
        with torch.inference_mode():
            for _ in range(warmup):
                model.forward_masked(x, fill=float("-inf"))
            torch.cuda.synchronize()
            evs = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True))
                   for _ in range(steps)]
            t0 = time.perf_counter()
            for a, b in evs:
                a.record()                         # same stream the kernel is launched on
                model.forward_masked(x, fill=float("-inf"))
                b.record()
            torch.cuda.synchronize()
            wall = (time.perf_counter() - t0) / steps
        kernel = sum(a.elapsed_time(b) for a, b in evs) / steps * 1e-3
        return wall, kernel

    if args.calibrate_copy:
        src = torch.ones(64 * 1024 * 1024, dtype=torch.float32, device=dev)   # 256 MiB
        dst = src + 1.0          # one elementwise kernel: reads 256 MiB, writes 256 MiB
        torch.cuda.synchronize()
        del src, dst

    wall, kern = run_mode(args.precision, K, W)
    value = B / wall
    achieved = B * CONV_FLOP_PER_BOARD / kern / 1e12
    kernel_name = {"fp32": "half_forward_kernel<fp32>", "bf16": "duo_forward_kernel<bf16>",
                   "fp16": "duo_forward_kernel<fp16>"}.get(args.precision, f"fused_pipe_kernel<{args.precision}>")
    cascade = None
    if args.precision == "bf16c":
        # HIP events bracket the whole step: the bf16 kernel over all boards, then the kernel
        # that carries the low parts over the listed ones.  The first pass alone is timed with
        # threshold 0 (no board listed; the second kernel still starts and finds nothing).
        kernel_name = "duo_forward_kernel<bf16> over all boards + second_pass_kernel<bf16f6w> over the listed boards"
        twice = int(model.cascade_stats["second_pass"].item())
        model.cascade_threshold = 0.0
        _, first = run_mode("bf16c", max(5, K // 2), 3)
        model.cascade_threshold = None
        cascade = {"threshold": c6.CASCADE_THRESHOLD, "boards_evaluated_twice": twice, "fraction": twice / B,
                   "first_pass_ms": first * 1e3, "second_pass_ms": (kern - first) * 1e3}
    out = {
        "metric": "boards/sec B=4096 bf16 forward + % MFMA peak; G=8 grouped-history boards/sec",
        "value": value,
        "unit": "boards/s",
        "n_gpus": 1,
        "steps": K,
        "warmup": W,
        "ms_per_step": wall * 1e3,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic",
        "config": {
            "workload": f"configs[1]: default CNN, B={B}, stones 0..200, masked logits + value, "
                        f"reference init, seed 1234/2025",
            "precision_mode": args.precision,
            "batch": B,
        },
        "roofline": {
            "bound": "mfma",
            "achieved": achieved,
            "peak": MFMA_PEAK_TFLOPS,
            "unit": "TFLOP/s",
            "frac": achieved / MFMA_PEAK_TFLOPS,
            "traffic": TRAFFIC_BYTES.get(args.precision),
            "traffic_unit": "bytes per launch",
            "kernel": kernel_name,
            "kernel_ms": kern * 1e3,
            "flop_per_board": CONV_FLOP_PER_BOARD,
        },
    }
    if cascade is not None:
        out["roofline"]["cascade"] = cascade
    # What this card sustains on back-to-back bf16 MFMAs alone (every CU, one wave per SIMD): the
    # published peak assumes the top shader clock, which the card's power management does not hold
    # under a dense matrix load with ordinary operand bits.  Reported beside the roofline, which
    # stays priced against the published peak.
    try:
        rnd = c6.probe_mfma_rate(60000, zero_operands=False)
        zer = c6.probe_mfma_rate(60000, zero_operands=True)
        out["roofline"]["sustained_mfma_only"] = {
            "random_operands": rnd, "zero_operands": zer,
            "frac_of_sustained": achieved / rnd["tflops"],
            "note": "v_mfma_f32_32x32x16_bf16 back to back on all CUs; TFLOP/s over the launch (HIP events), "
                    "mean shader clock from the cycle counter against the 100 MHz counter",
        }
    except c6.C6Error as exc:   # (the probe is an aid, not part of the measured path)
        out["roofline"]["sustained_mfma_only"] = {"error": str(exc)}

    if not args.no_extras:
        # ---- every arithmetic mode, with its agreement with the fp32 kernel ----
        model.precision = "fp32"
        with torch.inference_mode():
            l32, v32 = model.forward_masked(x, fill=float("-inf"))
        modes = {}
        for prec in ("bf16c", "bf16f6w", "bf16f6", "bf16", "fp16", "fp32"):
            w_, k_ = run_mode(prec, max(5, K // 2), 3)
            with torch.inference_mode():
                lg, vg = model.forward_masked(x, fill=float("-inf"))
            fin = torch.isfinite(l32)
            modes[prec] = {
                "boards_per_s": B / w_,
                "kernel_ms": k_ * 1e3,
                "mfma_frac_dense": B * CONV_FLOP_PER_BOARD / k_ / 1e12 / (157.3 if prec == "fp32" else MFMA_PEAK_TFLOPS),
                "rel_l2_logits_vs_fp32_kernel": float((lg[fin] - l32[fin]).norm() / l32[fin].norm()),
                "argmax_agreement_vs_fp32_kernel": float((lg.argmax(1) == l32.argmax(1)).float().mean()),
            }
        out["modes"] = modes

        # ---- grouped history: G=8 weight sets x 512 boards in one launch ----
        cfg = {"architecture_version": 4, "kernels": list(model.kernels), "channels": list(model.channels)}
        cps = []
        for i in range(8):
            torch.manual_seed(1234 + i)
            cps.append(c6.HistoricalCheckpoint(
                path=Path(f"model_update_{i + 1:08d}.pt"), update=i + 1,
                model_state=c6.PolicyValueNet().state_dict(), model_config=cfg,
                game_config={"board_size": 19, "win_length": 6}))
        # (a bf16 ensemble picks its own mode, as a caller's would: the cascade without a low part of
        # the weights, which parameters held in bf16 do not have; any other mode is passed on)
        ens_precision = None if args.precision in ("fp32", HEADLINE) else args.precision
        ens = c6.HistoricalPolicyEnsemble(cps, dev, dtype=torch.bfloat16, precision=ens_precision)
        xg = x.view(8, B // 8, 3, 19, 19).to(torch.bfloat16)

        def timed(fn, steps=max(5, K // 2), warmup=3):
            with torch.inference_mode():
                for _ in range(warmup):
                    fn()
                torch.cuda.synchronize()
                t0 = time.perf_counter()
                for _ in range(steps):
                    fn()
                torch.cuda.synchronize()
            return (time.perf_counter() - t0) / steps

        tg = timed(lambda: ens.forward_grouped(xg))
        out["grouped_g8"] = {
            "boards_per_s": B / tg, "ms": tg * 1e3, "ratio_to_single": (B / tg) / value,
            "workload": f"configs[2]: 8 weight sets x {B // 8} boards, one launch, bf16 in/out",
            "precision_mode": {v: k for k, v in _lib_names().items()}[ens._prec],
        }

        # production shape of the history path (configs/train.yaml of the reference: up to 128
        # frozen models sharing 512 tables): weight traffic per board is 32x the G=8 case
        cps128 = [cps[i % 8] for i in range(128)]
        ens128 = c6.HistoricalPolicyEnsemble(cps128, dev, dtype=torch.bfloat16, precision=ens_precision)
        xg128 = x[:512].view(128, 4, 3, 19, 19).to(torch.bfloat16)
        ens128.conv_weights, ens128.conv_biases, ens128.policy_weight, ens128.policy_bias   # (stack: host work + H2D)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        ens128._packed_weights()                 # 128 weight sets into kernel layout: two launches
        torch.cuda.synchronize()
        pack128 = time.perf_counter() - t0
        tg128 = timed(lambda: ens128.forward_grouped(xg128))
        out["grouped_g128x4"] = {"boards_per_s": 512 / tg128, "ms": tg128 * 1e3,
                                 "pack_128_weight_sets_ms": pack128 * 1e3}
        del ens128, cps128

        # ---- fused self-play step, configs[3]: B=16384, stones 0..300 ----
        model.precision = args.precision
        xs = gen_boards(16384, 300, 2025)[0].to(dev)
        us = gen_uniform(16384, 7).to(dev)
        ts = timed(lambda: model.selfplay_step(xs, us, 1.0), steps=10)
        out["selfplay_step_b16384"] = {"boards_per_s": 16384 / ts, "ms": ts * 1e3}

        # ---- the same step fed from int8 environment state (view + canonical input + gather in the loader) ----
        occ_ = (xs[:, 0] + xs[:, 1]) > 0
        boards8 = (xs[:, 0] - xs[:, 1]).to(torch.int8)
        player8 = torch.ones(16384, dtype=torch.int8, device=dev)
        left8 = torch.ones(16384, dtype=torch.int8, device=dev)
        tsb = timed(lambda: model.selfplay_step_boards(boards8, player8, left8, us, 1.0, view=5), steps=10)
        out["selfplay_step_from_int8_boards_b16384"] = {"boards_per_s": 16384 / tsb, "ms": tsb * 1e3}
        del occ_

        # ---- D4-averaged evaluation, configs[4]: 8192 base boards -> 65536 views ----
        xd = gen_boards(8192, 200, 2025)[0].to(dev)
        td = timed(lambda: c6.evaluate_d4(model, xd), steps=5, warmup=2)
        out["d4_eval_8192x8"] = {"base_boards_per_s": 8192 / td, "ms": td * 1e3}

        # ---- HBM-bound tail kernels: algorithmic bytes / kernel time (HIP events) ----
        def event_timed(fn, steps=20, warmup=3):
            with torch.inference_mode():
                for _ in range(warmup):
                    fn()
                torch.cuda.synchronize()
                e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                e0.record()
                for _ in range(steps):
                    fn()
                e1.record()
                torch.cuda.synchronize()
            return e0.elapsed_time(e1) * 1e-3 / steps

        nb, nd = 262144, 32768          # large enough that launch overhead does not show
        lg = torch.randn(nb, 361, device=dev)
        lgl = gen_boards(nb, 300, 5)[1].to(dev)
        un = gen_uniform(nb, 3).to(dev)
        xdd = gen_boards(nd, 200, 9)[0].to(dev)
        views = torch.randn(8, nd, 361, device=dev)
        vals = torch.randn(8, nd, device=dev)
        hbm = {}
        t = event_timed(lambda: c6.mask_logits(lg, lgl))
        hbm["mask_logits_f32"] = {"GBps": nb * 361 * (4 + 1 + 4) / t / 1e9, "boards": nb}
        t = event_timed(lambda: c6.sample_actions(lg, lgl, 1.0, un))
        hbm["softmax_sample"] = {"GBps": nb * (361 * 5 + 4 + 12) / t / 1e9, "boards": nb}
        t = event_timed(lambda: c6.d4_expand(xdd))
        hbm["d4_expand_f32"] = {"GBps": nd * 3 * 361 * 4 * 9 / t / 1e9, "boards": nd}
        t = event_timed(lambda: c6.d4_reduce(views, vals))
        hbm["d4_reduce"] = {"GBps": nd * (361 * 4 * 9 + 4 * 9) / t / 1e9, "boards": nd}
        # environment step (VectorConnect6.step) and canonical input on mid-game positions
        xe, le = gen_boards(nb, 200, 11)
        env = c6.VectorConnect6(nb, 19, 6, device=dev)
        env.boards.copy_((xe[:, 0] - xe[:, 1]).to(torch.int8))
        env.empty_count.copy_(le.sum(1).to(torch.int16))
        env.move_count.copy_((361 - le.sum(1)).to(torch.int16))
        acts = torch.rand(le.shape).masked_fill(~le, -1.0).argmax(1).to(dev)
        t = event_timed(lambda: env.step(acts))
        # per game: action 8 + state 6 + up to 40 neighbour squares in; stone 1 + state 6 + results 9 out
        hbm["env_step"] = {"GBps": nb * 70 / t / 1e9, "boards": nb, "games_per_s": nb / t}
        t = event_timed(lambda: env.network_input())
        hbm["canonical_input"] = {"GBps": nb * (361 + 2 + 3 * 361 * 4) / t / 1e9, "boards": nb}
        env16 = c6.VectorConnect6(16384, 19, 6, device=dev)
        env16.boards.copy_(env.boards[:16384])
        t16 = event_timed(lambda: env16.step(acts[:16384]))
        out["env_step_b16384"] = {"games_per_s": 16384 / t16, "us": t16 * 1e6}
        # one whole collector iteration (connect6/train.py:730-748, :791-799, :854-864 of the
        # reference): int8 state -> view -> forward -> mask -> sample -> map back -> step -> reset
        def collector_iteration():
            a_, _, _ = model.selfplay_step_boards(env16.boards, env16.current_player, env16.stones_left,
                                                  us, 1.0, view=5)
            step = env16.step(a_, view=5)
            env16.reset(torch.nonzero(step.done).flatten())
        env16.reset()
        tc = timed(collector_iteration, steps=20)
        out["collector_iteration_b16384"] = {"boards_per_s": 16384 / tc, "ms": tc * 1e3}
        del env, env16, xe, le, acts
        for v in hbm.values():
            v["frac_of_hbm_peak"] = v["GBps"] / HBM_PEAK_GBS
        out["hbm_kernels"] = hbm
        del lg, lgl, un, xdd, views, vals

    if not args.no_cpu_baseline:
        # The PyTorch fp32 oracle (the checker) on this box's host cores, configs[0] shape.
        from oracle import torch_ref as R

        threads = min(os.cpu_count() or 1, 16)
        torch.set_num_threads(threads)
        st = {k: v.detach().cpu().float() for k, v in model.state_dict().items()}
        xb = x_host[:256]
        with torch.inference_mode():
            for _ in range(2):
                R.forward(st, xb)
            times = []
            t_end = time.perf_counter() + 12.0
            while len(times) < 5 or (time.perf_counter() < t_end and len(times) < 40):
                t0 = time.perf_counter()
                R.forward(st, xb)
                times.append(time.perf_counter() - t0)
        times.sort()
        med = times[len(times) // 2]
        cpu_model = ""
        try:
            with open("/proc/cpuinfo") as fh:
                cpu_model = next((ln.split(":", 1)[1].strip() for ln in fh if ln.startswith("model name")), "")
        except OSError:
            pass
        out["cpu_baseline"] = {
            "value": 256 / med, "unit": "boards/s", "cores": threads, "kind": "port",
            "cpu_model": cpu_model, "os_cpu_count": os.cpu_count(),
            "sample": f"configs[0]: {len(times)} fp32 forwards of B=256 (same generator, same weights) "
                      f"with the PyTorch oracle, median",
        }
    print(json.dumps(out))
    return 0


if __name__ == "__main__":
    sys.exit(main())
