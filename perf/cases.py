"""The work a program that uses this package has it do, as cases to be timed.

Every case goes through the public entry points with the inputs that the callers of the reference
feed them: 0/1 planes with a constant third plane, int8 environment state, networks with the
reference's initialisation.  ``listed`` names the cases, ``draw`` takes further ones from the same
ranges, ``prepare`` builds what a program holds before the call, ``run`` is one pass.
"""
from __future__ import annotations

import math
from pathlib import Path

import torch

import connect6_amd as c6
from connect6_amd.synthetic import gen_boards, gen_uniform

PIX = 361
PARAMS = 374_082
FLOP_PER_BOARD = 269_692_992          # eight convolutions (dense count) and both heads
DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # One position at a time, parameters in fp32: a player waiting for the program's move.
        {"name": "move_fp32_b1", "path": "move", "dtype": "fp32", "batch": 1},
        # The same under autocast: the smallest call of the 16-bit path.
        {"name": "move_bf16_b1", "path": "move", "dtype": "bf16", "batch": 1},
        # Two checkpoints playing a match: the open games in which one of them is to move.
        {"name": "match_fp32_b53", "path": "move", "dtype": "fp32", "batch": 53},
        # The benchmark loop: a vector environment's network input, fp32 forward, legality mask.
        {"name": "envloop_fp32_b2048", "path": "envloop", "dtype": "fp32", "batch": 2048},
        # A ragged batch in half precision.
        {"name": "move_fp16_b777", "path": "move", "dtype": "fp16", "batch": 777},
        # One collector step: the current model's three quarters of 2048 environments, gathered
        # from the int8 state through one of the eight board symmetries, sampled in the same call.
        {"name": "collect_bf16_1536of2048", "path": "collect", "dtype": "bf16", "envs": 2048, "batch": 1536, "view": 5},
        # The ordinary large batch, logits masked in the call.
        {"name": "masked_bf16_b4096", "path": "masked", "dtype": "bf16", "batch": 4096},
        # Historical opponents as training runs them: many frozen networks with few tables each.
        {"name": "history_bf16_128x4", "path": "history", "dtype": "bf16", "models": 128, "tables": 4},
        # ... and as an evaluation runs them: few networks with many tables each.
        {"name": "history_bf16_8x512", "path": "history", "dtype": "bf16", "models": 8, "tables": 512},
        # Evaluation averaged over the eight board symmetries, the largest call.
        {"name": "d4_bf16_b8192", "path": "d4", "dtype": "bf16", "batch": 8192},
        # A small network on a small board, as a first experiment configures it.
        {"name": "arch_fp32_9x9_b1024", "path": "arch", "dtype": "fp32", "batch": 1024, "board": 9,
         "kernels": "5,3,3", "channels": "16,32,32", "models": 1},
        # What follows the logits in a rollout: draw, environment step, next network input.
        {"name": "rollout_n16384", "path": "rollout", "dtype": "fp32", "batch": 16384},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    path = rng.choice(["move", "move", "move", "envloop", "collect", "masked", "history", "history", "d4", "arch", "rollout"])
    if path == "move":
        return {"path": path, "dtype": rng.choice(["fp32", "bf16", "fp16"]), "batch": _log_int(rng, 2, 3000)}
    if path == "envloop":
        return {"path": path, "dtype": "fp32", "batch": _log_int(rng, 32, 3000)}
    if path == "collect":
        envs = _log_int(rng, 64, 16384)
        return {"path": path, "dtype": rng.choice(["bf16", "bf16", "fp16"]), "envs": envs,
                "batch": max(1, int(envs * rng.uniform(0.2, 1.0))), "view": rng.randrange(8)}
    if path == "masked":
        return {"path": path, "dtype": rng.choice(["bf16", "bf16", "fp16"]), "batch": _log_int(rng, 2, 16384)}
    if path == "history":
        models = _log_int(rng, 2, 128)
        return {"path": path, "dtype": rng.choice(["bf16", "bf16", "fp16"]), "models": models,
                "tables": _log_int(rng, 1, max(1, 6000 // models))}
    if path == "d4":
        return {"path": path, "dtype": "bf16", "batch": _log_int(rng, 2, 8000)}
    if path == "arch":
        board = rng.choice([5, 7, 9, 13, 15, 19])
        layers = rng.randint(2, 5)
        kernels = [rng.choice([3, 5, 7])] + [rng.choice([1, 3, 3, 3, 5]) for _ in range(layers - 1)]
        channels = [rng.choice([8, 16, 24, 32]) for _ in range(layers)]
        models = rng.choice([1, 1, 2, 4])
        case = {"path": path, "dtype": rng.choice(["fp32", "fp32", "bf16"]), "batch": models, "board": board,
                "kernels": ",".join(map(str, kernels)), "channels": ",".join(map(str, channels)), "models": models}
        most = max(1, min(1500, int(4e9 / _arch_flops(case))))
        case["batch"] = models * _log_int(rng, 1, max(1, most // models))
        return case
    return {"path": path, "dtype": "fp32", "batch": _log_int(rng, 16, 65536)}


def _arch(case):
    return [int(v) for v in case["kernels"].split(",")], [int(v) for v in case["channels"].split(",")]


def _arch_flops(case):
    """of one board"""
    kernels, channels = _arch(case)
    total, cin = 0, 3
    for k, c in zip(kernels, channels):
        total += k * k * cin * c
        cin = c
    return 2 * case["board"] ** 2 * (total + 2 * cin)


def _arch_params(case):
    kernels, channels = _arch(case)
    total, cin = 0, 3
    for k, c in zip(kernels, channels):
        total += (k * k * cin + 1) * c
        cin = c
    return total + 2 * (cin + 1)


# -- what a program holds before the call ----------------------------------------------------

def _network(seed, device, case=None):
    with torch.random.fork_rng(devices=[]):
        torch.manual_seed(seed)
        if case is None:
            net = c6.PolicyValueNet()
        else:
            kernels, channels = _arch(case)
            net = c6.build_model({"kernels": kernels, "channels": channels}, case["board"])
    return net.to(device).eval()


def _ensemble(case, seed, device):
    other = case["path"] == "arch"
    checkpoints = []
    for i in range(case["models"]):
        net = _network(seed * 1000 + i, "cpu", case if other else None)
        checkpoints.append(c6.HistoricalCheckpoint(
            path=Path(f"model_update_{i + 1:08d}.pt"), update=i + 1, model_state=net.state_dict(),
            model_config={"kernels": list(net.kernels), "channels": list(net.channels)},
            game_config={"board_size": net.board_size, "win_length": 6}))
    return c6.HistoricalPolicyEnsemble(checkpoints, device, dtype=DTYPES[case["dtype"]])


def _environment(batch, seed, device):
    """Mid-game positions as the vector environment holds them."""
    x, legal = gen_boards(batch, 200, seed)
    env = c6.VectorConnect6(batch, 19, 6, device=device)
    g = torch.Generator().manual_seed(seed + 1)
    player = torch.where(torch.rand(batch, generator=g) < 0.5, -1, 1).to(torch.int8)
    env.boards.copy_((x[:, 0] - x[:, 1]).to(torch.int8) * player.view(-1, 1, 1))
    env.current_player.copy_(player)
    env.stones_left.copy_(torch.where(x[:, 2, 0, 0] > 0, 1, 2).to(torch.int8))
    free = legal.sum(1)
    env.empty_count.copy_(free.to(torch.int16))
    env.move_count.copy_((PIX - free).to(torch.int16))
    return env, legal


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    path, s = case["path"], {"case": case}
    s["autocast"] = DTYPES[case["dtype"]] if case["dtype"] != "fp32" else None
    if path in ("move", "masked", "d4"):
        s["model"] = _network(seed, dev)
        x, legal = gen_boards(case["batch"], 200, seed)
        s["x"], s["legal"] = x.to(dev), legal.to(dev)
    elif path == "envloop":
        s["model"] = _network(seed, dev)
        s["env"], _ = _environment(case["batch"], seed, dev)
    elif path == "collect":
        s["model"] = _network(seed, dev)
        s["env"], _ = _environment(case["envs"], seed, dev)
        order = torch.randperm(case["envs"], generator=torch.Generator().manual_seed(seed + 2))
        s["index"] = order[: case["batch"]].sort().values.to(dev)
        s["u"] = gen_uniform(case["batch"], seed + 3).to(dev)
    elif path == "history":
        s["ensemble"] = _ensemble(case, seed, dev)
        x, _ = gen_boards(case["models"] * case["tables"], 200, seed)
        s["x"] = x.view(case["models"], case["tables"], 3, 19, 19).to(dev)
    elif path == "arch":
        board = case["board"]
        x, _ = gen_boards(case["batch"], board * board // 2, seed, board_size=board)
        s["x"] = x.to(dev)
        if case["models"] == 1:
            s["model"] = _network(seed, dev, case)
        else:
            s["ensemble"] = _ensemble(case, seed, dev)
            s["x"] = s["x"].view(case["models"], -1, 3, board, board)
    else:  # rollout
        s["env"], legal = _environment(case["batch"], seed, dev)
        s["legal"] = legal.to(dev)
        s["logits"] = torch.randn(case["batch"], PIX, generator=torch.Generator().manual_seed(seed + 2)).to(dev)
        s["u"] = gen_uniform(case["batch"], seed + 3).to(dev)
    return s


# -- one pass ----------------------------------------------------------------------------------

def run(s):
    with torch.inference_mode():
        if s["autocast"] is None:
            return _run(s)
        with torch.autocast("cuda", dtype=s["autocast"]):
            return _run(s)


def _run(s):
    path = s["case"]["path"]
    if path == "move":
        logits, value = s["model"](s["x"])
        return logits, value, c6.mask_logits(logits.float(), s["legal"])
    if path == "envloop":
        env = s["env"]
        logits, value = s["model"](env.network_input())
        return logits, value, c6.mask_logits(logits.float(), env.legal_mask())
    if path == "collect":
        env = s["env"]
        return s["model"].selfplay_step_boards(env.boards, env.current_player, env.stones_left, s["u"], 1.0,
                                               index=s["index"], view=s["case"]["view"])
    if path == "masked":
        return s["model"].forward_masked(s["x"], fill=float("-inf"))
    if path == "d4":
        return c6.evaluate_d4(s["model"], s["x"])
    if path == "history" or (path == "arch" and s["case"]["models"] > 1):
        return s["ensemble"].forward_grouped(s["x"])
    if path == "arch":
        return s["model"](s["x"])
    env = s["env"]
    actions, logprob = c6.sample_actions(s["logits"], s["legal"], 1.0, s["u"])
    step = env.step(actions)
    # (the same squares again in a further pass: the stones there are replaced, the counters go on)
    return (actions, logprob, step.reward, step.done, step.winner, step.transition_sign, step.game_lengths,
            env.boards, env.current_player, env.stones_left, env.empty_count, env.move_count, env.network_input())


# -- what a pass cannot do without -------------------------------------------------------------

def work(case):
    path, b = case["path"], case["batch"] if "batch" in case else case["models"] * case["tables"]
    size = 4 if case["dtype"] == "fp32" else 2      # bytes of a parameter as the arithmetic reads it
    planes, logits, value = 3 * PIX * 4, PIX * 4, 4
    if path == "move":       # ... and the masked copy: legality in, logits out
        return {"bytes": b * (planes + 2 * logits + value + PIX) + PARAMS * size, "flops": b * FLOP_PER_BOARD}
    if path == "envloop":    # int8 state in; logits, value and masked logits out
        return {"bytes": b * (PIX + 2 + 2 * logits + value) + PARAMS * size, "flops": b * FLOP_PER_BOARD}
    if path == "collect":    # int8 state, row and draw in; action, log-probability and value out
        return {"bytes": b * (PIX + 2 + 8 + 4 + 8 + 4 + value) + PARAMS * size, "flops": b * FLOP_PER_BOARD}
    if path == "masked":
        return {"bytes": b * (planes + logits + value) + PARAMS * size, "flops": b * FLOP_PER_BOARD}
    if path == "history":    # (policy only; logits in the ensemble's type)
        return {"bytes": b * (planes + PIX * size) + case["models"] * PARAMS * size,
                "flops": b * (FLOP_PER_BOARD - 2 * PIX * 96)}
    if path == "d4":         # every board eight times through the network
        return {"bytes": b * (planes + logits + value) + PARAMS * size, "flops": 8 * b * FLOP_PER_BOARD}
    if path == "arch":
        nn = case["board"] ** 2
        return {"bytes": b * nn * (3 * 4 + size) + case["models"] * _arch_params(case) * size,
                "flops": b * _arch_flops(case)}
    # rollout: logits, legality and draw in, action and log-probability out; the step's state and
    # results; the board in and its planes out
    return {"bytes": b * (PIX * 5 + 4 + 12 + 8 + 2 * 6 + 9 + PIX + 2 + planes), "flops": b * 20 * PIX}


def tolerance(case):
    if case["path"] == "rollout":
        # draws and rules: the same numbers; a draw on the edge of two squares may fall either way
        return {"rel": 1e-5, "differ": 1e-3}
    if case["dtype"] == "fp32":
        # 32-bit sums of up to 1587 products through eight layers; a value near zero is the rest
        # of a sum that cancels
        return {"rel": 3e-5, "max": 1e-3}
    # one rounding to the 16-bit type per layer boundary, its size relative to the logits; a draw
    # next to the edge of two squares falls either way, its log-probability with it
    return {"rel": 4e-3 if case["dtype"] == "fp16" else 2e-2, "max": 0.5, "differ": 0.01}
