"""Workloads for timing the library through its Python entry points.

`listed()` names the fixed cases, `draw(rng)` makes one more of the same ranges,
`prepare(case, seed)` puts the inputs on the GPU and makes the context or trainer a
program keeps, `run(state)` is one pass, `work(case)` the bytes and operations a pass
cannot do without, and `tolerance(case)` how far two correct evaluations may lie apart.

Kinds of work:

  chain       forward and backward of the per-thread graph, one problem per element
  accumulate  the same graph, its gradients added into shared slots (strategy "auto")
  train       one iteration of splatting: render, loss, gradients, Adam
  render      forward only, the depth order made anew for every image
  trainer     the training front-end: ten iterations with the loss of the last
  sgd         the least-squares fit, all steps on the device
"""
import math

import torch

from xyz_autodiff_cuda_amd import accumulate, chain, linreg, rng, splat, trainer

DEVICE = "cuda:0"
TRAINER_ITERATIONS = 10  # the training program reports its loss every tenth iteration
# Adam rates of the training cases, one per parameter row: centre (pixels), log-scale, angle, colour, opacity
LEARNING_RATES = (0.01, 0.01, 0.001, 0.001, 0.001, 0.002, 0.002, 0.002, 0.005)


def listed():
    return [
        # A handful of problems per call: what a caller with many small batches pays, launch and host path included.
        {"name": "chain_4099", "kind": "chain", "n": 4099},
        # A million independent problems, the size the host cores are compared on.
        {"name": "chain_1m", "kind": "chain", "n": 1_000_000},
        # The benchmark's batch: 64 Mi problems, 3.5 GB of arrays, far beyond the caches.
        {"name": "chain_64mi", "kind": "chain", "n": 64 * 1024 * 1024},
        # A few parameters shared by everybody: every slot is contended.
        {"name": "accumulate_16mi_64_zipf", "kind": "accumulate", "n": 16 * 1024 * 1024, "slots": 64, "law": "zipf"},
        # A large parameter table with a hot head and a long cold tail.
        {"name": "accumulate_16mi_262144_zipf", "kind": "accumulate", "n": 16 * 1024 * 1024, "slots": 262_144, "law": "zipf"},
        # No slot hotter than another, more slots than a compute unit's LDS holds (a scene's worth of Gaussians), odd length.
        {"name": "accumulate_1m_10k_uniform", "kind": "accumulate", "n": 1_000_003, "slots": 10_000, "law": "uniform"},
        # The training program with its default number of Gaussians, on a photograph-sized target with ragged edges.
        {"name": "trainer_1000_640x427", "kind": "trainer", "gaussians": 1000, "width": 640, "height": 427},
        # The small benchmark scene, trained without ever waiting for the device.
        {"name": "train_10k_512", "kind": "train", "gaussians": 10_000, "width": 512, "height": 512, "scale_lo": 1.0,
         "scale_hi": 20.0, "mode": "static", "loss": False},
        # A loop that keeps the defaults: depths checked, the loss read back every iteration; a ragged image.
        {"name": "train_50k_1277x719", "kind": "train", "gaussians": 50_021, "width": 1277, "height": 719, "scale_lo": 1.0,
         "scale_hi": 20.0, "mode": "checked", "loss": True},
        # The large benchmark scene, trained without waiting.
        {"name": "train_200k_2048", "kind": "train", "gaussians": 200_000, "width": 2048, "height": 2048, "scale_lo": 0.5,
         "scale_hi": 40.0, "mode": "static", "loss": False},
        # Rendering frames of a scene whose depths change from frame to frame.
        {"name": "render_100k_1920x1080", "kind": "render", "gaussians": 100_000, "width": 1920, "height": 1080,
         "scale_lo": 0.5, "scale_hi": 30.0, "mode": "every_step"},
        # The least-squares example's own sizes, a stretch of its ten thousand steps.
        {"name": "sgd_100k_8192", "kind": "sgd", "total": 100_000, "batch": 8192, "epochs": 200},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("chain", "accumulate", "train", "train", "render", "trainer", "sgd"))
    if kind == "chain":
        return {"kind": kind, "n": _log_uniform(rng, 4099, 64 * 1024 * 1024)}
    if kind == "accumulate":
        return {"kind": kind, "n": _log_uniform(rng, 1_000_003, 16 * 1024 * 1024), "slots": _log_uniform(rng, 64, 262_144),
                "law": rng.choice(("zipf", "uniform"))}
    if kind == "sgd":
        return {"kind": kind, "total": _log_uniform(rng, 10_000, 1_000_000), "batch": _log_uniform(rng, 256, 8192),
                "epochs": _log_uniform(rng, 20, 200)}
    # images from a thumbnail to the largest listed, with as many Gaussians per pixel as the listed scenes have
    width, height = _log_uniform(rng, 256, 2048), _log_uniform(rng, 256, 2048)
    density = math.exp(rng.uniform(math.log(0.004), math.log(0.047)))
    gaussians = max(1000, int(density * width * height))
    if kind == "trainer":
        return {"kind": kind, "gaussians": min(gaussians, 20_000), "width": min(width, 1024), "height": min(height, 1024)}
    case = {"kind": kind, "gaussians": gaussians, "width": width, "height": height, "scale_lo": round(rng.uniform(0.5, 1.5), 2),
            "scale_hi": round(rng.uniform(10.0, 40.0), 1), "mode": rng.choice(("checked", "static", "every_step"))}
    if kind == "train":
        case["loss"] = rng.random() < 0.5
    return case


def prepare(case, seed):
    kind = case["kind"]
    state = {"kind": kind}
    if kind in ("chain", "accumulate"):
        n = case["n"]
        inputs = [torch.empty(n, dtype=torch.float32, device=DEVICE) for _ in chain.INPUT_NAMES]
        state["inputs"] = rng.chain_inputs_(inputs, seed)
        if kind == "chain":
            state["outputs"] = [torch.empty(n, dtype=torch.float32, device=DEVICE) for _ in chain.OUTPUT_NAMES]
            return state
        slot = torch.empty(n, dtype=torch.int32, device=DEVICE)
        if case["law"] == "zipf":
            accumulate.zipf_(slot, seed, 10, case["slots"], 1.1)
        else:
            u = torch.empty(n, dtype=torch.float32, device=DEVICE)
            rng.uniform_(u, seed, 10, 0.0, 1.0)
            slot.copy_((u.double() * case["slots"]).to(torch.int32).clamp_(max=case["slots"] - 1))
        state["slot"] = slot
        state["grads"] = torch.empty(case["slots"], accumulate.WIDTH, dtype=torch.float32, device=DEVICE)
        return state
    if kind == "sgd":
        state["samples"] = [torch.from_numpy(a).to(DEVICE) for a in linreg.synthetic_data(case["total"], seed=seed)]
        state["params"] = torch.tensor(linreg.INITIAL_PARAMS, dtype=torch.float64, device=DEVICE)
        state["batch"], state["epochs"], state["seed"] = case["batch"], case["epochs"], seed
        return state
    G, W, H = case["gaussians"], case["width"], case["height"]
    if kind == "trainer":
        target = splat.synthetic_target(G, W, H, seed=seed + 1, scale_px=(2.0, 12.0)).cpu().numpy()
        config = trainer.TrainingConfig.defaults(num_gaussians=G, seed=seed, target_image_path="synthetic", lr_center=0.05,
                                                 lr_scale=0.001, lr_rotation=0.002, lr_color=0.003, lr_opacity=0.004)
        state["trainer"] = trainer.Trainer(config, target)
        return state
    scale = (case["scale_lo"], case["scale_hi"])
    state["params"], state["depth"] = splat.synthetic_scene(G, W, H, seed=seed, scale_px=scale)
    # room for the lists as the benchmark of the large scene asks for it; smaller scenes start from the default
    hint = 45 * G if G > 50_000 else 0
    state["context"] = splat.SplatContext(W, H, G, pair_capacity_hint=hint, device=DEVICE, depth_mode=case["mode"])
    state["image"] = torch.empty(H, W, 3, dtype=torch.float32, device=DEVICE)
    if kind == "train":
        state["target"] = splat.synthetic_target(G, W, H, seed=seed + 1, scale_px=scale)
        state["grads"] = torch.empty_like(state["params"])
        state["m"], state["v"] = torch.zeros_like(state["params"]), torch.zeros_like(state["params"])
        state["gate"] = state["context"].overflow_word()
        state["loss"], state["iteration"] = case["loss"], 0
    return state


def run(state):
    kind = state["kind"]
    if kind == "chain":
        return chain.forward_backward(state["inputs"], state["outputs"])
    if kind == "accumulate":
        return accumulate.accumulate_chain_gradients(state["inputs"], state["slot"], state["grads"].zero_())
    if kind == "sgd":
        x1, x2, y = state["samples"]
        history = linreg.sgd(x1, x2, y, state["params"], state["batch"], state["epochs"], seed=state["seed"], want_history=True)
        return {"params": state["params"], "history": history}
    if kind == "trainer":
        loss = state["trainer"].run(TRAINER_ITERATIONS)
        after = state["trainer"].state()
        return {"loss": loss, "params": after["params"], "m": after["m"], "v": after["v"]}
    context = state["context"]
    if kind == "render":
        return context.forward(state["params"], state["depth"], state["image"])
    image, grads, loss = context.step(state["params"], state["depth"], state["target"], state["image"], state["grads"],
                                      want_loss=state["loss"])
    state["iteration"] += 1
    # the update is withheld on the device when the lists of a step that did not wait were cut short
    splat.adam_step(state["params"], grads, state["m"], state["v"], LEARNING_RATES, state["iteration"],
                    hold_if_nonzero=state["gate"])
    out = {"image": image, "grads": grads, "params": state["params"], "m": state["m"], "v": state["v"]}
    if loss is not None:
        out["loss"] = loss
    return out


def _composited_per_pixel(G, W, H, lo, hi):
    """Gaussians a pixel composites: those whose 3-sigma ellipse covers it (scales log-uniform in lo..hi), at most the
    66 after which a pixel of such a scene has fallen below the transmittance it stops at (their mean -log(1 - alpha) is
    0.14, the stop is at 9.2)."""
    mean_scale = (hi - lo) / math.log(hi / lo)
    return min(66.0, G * 9.0 * math.pi * mean_scale ** 2 / (W * H))


def work(case):
    kind = case["kind"]
    if kind == "chain":
        return {"bytes": 52.0 * case["n"], "flops": 130.0 * case["n"]}
    if kind == "accumulate":
        return {"bytes": 28.0 * case["n"] + 24.0 * case["slots"], "flops": 136.0 * case["n"]}
    if kind == "sgd":
        draws = float(case["batch"]) * case["epochs"]
        return {"bytes": 24.0 * min(case["total"], draws) + 8.0 * case["epochs"] + 64.0, "flops": 30.0 * draws}
    G, pixels = case["gaussians"], case["width"] * case["height"]
    if kind == "trainer":
        scales, iterations = (math.e, math.e ** 2), TRAINER_ITERATIONS  # the trainer's own initial Gaussians
    else:
        scales, iterations = (case["scale_lo"], case["scale_hi"]), 1
    composited = _composited_per_pixel(G, case["width"], case["height"], *scales) * pixels
    # forward: falloff, alpha, three colours, transmittance (16 operations per pixel and Gaussian); backward about 40 more
    if kind == "render":
        return {"bytes": 40.0 * G + 12.0 * pixels, "flops": 16.0 * composited}
    # parameters and both moments read and written, gradients and depth; target read, image written
    return {"bytes": iterations * (292.0 * G + 24.0 * pixels), "flops": iterations * 56.0 * composited}


def tolerance(case):
    """Largest relative error (2-norm) of another correct evaluation: about four times what the path was seen to differ
    from a 64-bit evaluation, or from another 32-bit one with its sums in another order."""
    kind = case["kind"]
    if kind == "chain":
        return {"rel": 1e-4}  # 8.5e-6 from 64 bits, 3.8e-5 from another 32-bit evaluation: det = ac - b^2 cancels
    if kind == "accumulate":
        return {"rel": 1e-5}  # 2.0e-6 where a slot has a hundred terms
    if kind == "sgd":
        return {"rel": 1e-12}  # 64-bit sums of a batch, in any order
    if kind == "render":
        return {"rel": 1e-5}  # 7e-7, and now and then a pixel that stops one Gaussian earlier
    if kind == "trainer":
        return {"rel": 1e-4}  # ten Adam steps from zero moments: 8e-6 between two runs of the same thing
    # Gradients: 5.7e-6 where scales span a factor of 20, 1.1e-4 to 4.4e-4 where they span 80 (the condition of an inverse
    # covariance is the square of that, and the worst conditioned Gaussians have the largest gradients)
    return {"rel": 3e-5 * max(1.0, (case["scale_hi"] / case["scale_lo"] / 20.0) ** 2.5)}
