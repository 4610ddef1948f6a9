"""What a user of this framework runs and waits for, as cases to time.

A case is one call sequence through the public entry points: a policy's `forward()` on an observation (Pi0, Pi05, DM0, full depth,
seeded synthetic checkpoints in the converted layout), the observation transforms around it, and the whole control step
`ObservationTransforms.infer` from host camera frames to host actions.  `listed()` holds the benchmark configurations and the ends of
the range, `draw()` gives further cases of the same ranges.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("realtime-vla_amd"))      # of the tree this is run in, which need not be the one this file lies in

import synthetic as syn  # noqa: E402
from dm0_infer import DM0Inference  # noqa: E402
from obs_transforms import ObservationTransforms  # noqa: E402
from pi05_infer import Pi05Inference  # noqa: E402
from pi0_infer import Pi0Inference  # noqa: E402

VIEW_NAMES = ("base_0_rgb", "left_wrist_0_rgb", "right_wrist_0_rgb")
PI05_MAX_TOKENS = 200          # Pi05Inference's default allocation for prompts given as token ids


def listed():
    return [
        # one small wrist camera already at the model's size, Pi05 statistics with the 256-bin state: what is left is launches and host work
        {"name": "observe_1x224x224_pi05", "kind": "observe", "model": "pi05", "views": 1, "height": 224, "width": 224, "frames": "u8", "chunk": 50, "dims": 7},
        # the usual three VGA cameras, frames on the device (bench.py --transforms)
        {"name": "observe_3x480x640_pi0", "kind": "observe", "model": "pi0", "views": 3, "height": 480, "width": 640, "frames": "u8", "chunk": 50, "dims": 7},
        # two large cropped frames as dataset readers give them: float, channels first, odd sizes; two arms of seven joints
        {"name": "observe_2x717x1279_f32", "kind": "observe", "model": "pi0", "views": 2, "height": 717, "width": 1279, "frames": "f32_chw", "chunk": 63, "dims": 14},
        # the smallest forward in use: one camera, no prompt
        {"name": "pi0_1v_p0_c50", "kind": "pi0", "views": 1, "prompt": 0, "chunk": 50},
        # two cameras and a short prompt
        {"name": "pi0_2v_p20_c50", "kind": "pi0", "views": 2, "prompt": 20, "chunk": 50},
        # three cameras: the headline benchmark
        {"name": "pi0_3v_p20_c50", "kind": "pi0", "views": 3, "prompt": 20, "chunk": 50},
        # a long prompt: 968-token prefix
        {"name": "pi0_3v_p200_c50", "kind": "pi0", "views": 3, "prompt": 200, "chunk": 50},
        # the whole control step, host frames to host actions, with the long chunk and no prompt
        {"name": "infer_3v_480x640_p0_c63", "kind": "infer", "views": 3, "height": 480, "width": 640, "prompt": 0, "chunk": 63, "dims": 7},
        # Pi05 with a prompt of fixed embeddings: 20 text and 32 state tokens
        {"name": "pi05_3v_p52_c50", "kind": "pi05_embeds", "views": 3, "prompt": 52, "chunk": 50},
        # Pi05 with token ids that change per call, staged on the device; two cameras, odd lengths, a shorter chunk
        {"name": "pi05_2v_ids137_c33", "kind": "pi05_ids", "views": 2, "prompt": 137, "chunk": 33},
        # DM0 with one image and a short odd prompt
        {"name": "dm0_1i_l37", "kind": "dm0", "views": 1, "prompt": 37},
        # DM0 at its benchmark shape: the largest call
        {"name": "dm0_3i_l100", "kind": "dm0", "views": 3, "prompt": 100},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: the kinds in the proportions of the list, every size over its whole range, odd ones among them."""
    kind = rng.choice(["observe"] * 3 + ["pi0"] * 4 + ["infer", "pi05_embeds", "pi05_ids"] + ["dm0"] * 2)
    if kind == "observe":
        height = _log_int(rng, 120, 1080)
        width = max(120, min(1920, int(height * rng.uniform(0.75, 1.78))))
        return {"kind": kind, "model": rng.choice(["pi0", "pi05"]), "views": rng.randint(1, 3), "height": height, "width": width,
                "frames": rng.choice(["u8", "u8", "f32_chw"]), "chunk": rng.randint(16, 127), "dims": rng.choice([7, 8, 14, 32])}
    if kind == "dm0":
        return {"kind": kind, "views": rng.randint(1, 3), "prompt": _log_int(rng, 8, 100)}
    case = {"kind": kind, "views": rng.randint(1, 4 if kind == "pi0" else 3), "prompt": _log_int(rng, 1, 200), "chunk": rng.randint(16, 127)}
    if kind == "pi0" and rng.random() < 0.2:
        case["prompt"] = 0
    if kind == "infer":
        height = _log_int(rng, 240, 1080)
        case.update(height=height, width=max(240, min(1920, int(height * rng.uniform(1.0, 1.78)))), dims=rng.choice([7, 8, 14, 32]))
    return case


def _frames(case, seed, device):
    gen = torch.Generator(device=device).manual_seed(seed)
    shape = (case["views"], case["height"], case["width"], 3)
    if case.get("frames") == "f32_chw":
        return list(torch.rand(shape, device=device, generator=gen).permute(0, 3, 1, 2).contiguous())
    return list(torch.randint(0, 256, shape, dtype=torch.uint8, device=device, generator=gen))


def _norm_stats(model, dims, seed):
    rng = np.random.RandomState(seed % (1 << 31))
    groups = {}
    for group in ("state", "actions"):
        if model == "pi0":
            groups[group] = {"mean": rng.randn(dims).tolist(), "std": (rng.rand(dims) + 0.5).tolist()}
        else:
            groups[group] = {"q01": (-1.5 - rng.rand(dims)).tolist(), "q99": (1.5 + rng.rand(dims)).tolist()}
    return groups, rng.randn(dims)


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    kind = case["kind"]
    if kind == "observe":
        stats, joints = _norm_stats(case["model"], case["dims"], seed)
        gen = torch.Generator(device=dev).manual_seed(seed + 1)
        return {"kind": kind, "case": case,
                "transforms": ObservationTransforms(case["model"], stats, state_len=case["dims"], action_dim=case["dims"]),
                "frames": _frames(case, seed, dev), "joints": joints,
                "actions": torch.randn(case["chunk"], 32, device=dev, generator=gen).to(torch.bfloat16),
                # the policy's input buffers
                "images": torch.zeros(case["views"], 224, 224, 3, dtype=torch.bfloat16, device=dev),
                "state": torch.zeros(32, dtype=torch.bfloat16, device=dev)}
    views, prompt = case["views"], case["prompt"]
    if kind == "dm0":
        policy = DM0Inference(syn.dm0_checkpoint(seed, dev), num_images=views, max_lang_len=prompt)
        return {"kind": kind, "policy": policy, "inputs": syn.dm0_observation(seed, views, dev, max_lang_len=prompt)}
    images, state, noise = syn.observation(seed, views, case["chunk"], dev)
    if kind in ("pi0", "infer"):
        policy = Pi0Inference(syn.pi0_checkpoint(seed, prompt, dev, norms="random"), views, case["chunk"])
        if kind == "pi0":
            return {"kind": kind, "policy": policy, "inputs": (images, state, noise)}
        stats, joints = _norm_stats("pi0", case["dims"], seed)
        observation = {name: frame.numpy() for name, frame in zip(VIEW_NAMES, _frames(case, seed, torch.device("cpu")))}
        observation["state"] = joints
        return {"kind": kind, "policy": policy, "transforms": ObservationTransforms("pi0", stats, state_len=case["dims"], action_dim=case["dims"]),
                "observation": observation, "noise": noise}
    if kind == "pi05_embeds":
        state_tokens = min(32, prompt // 2)
        checkpoint = syn.pi05_checkpoint(seed, prompt - state_tokens, dev, state_tokens=state_tokens, norms="random")
        policy = Pi05Inference(checkpoint, views, case["chunk"], discrete_state_input=False)
        return {"kind": kind, "policy": policy, "inputs": (images, noise)}
    checkpoint = syn.pi05_checkpoint(seed, 0, dev, state_tokens=0, norms="random")
    del checkpoint["language_embeds"]
    checkpoint["embedding_weight"] = syn.normal_bf16(seed, "embedding_weight", (syn.VOCAB, 2048), 0.02, dev)
    policy = Pi05Inference(checkpoint, views, case["chunk"], max_tokenize_len=PI05_MAX_TOKENS, discrete_state_input=False)
    return {"kind": kind, "policy": policy, "inputs": (images, noise, syn.randint(seed, "prompt_ids", prompt, syn.VOCAB))}       # ids come from a host tokenizer


def run(state):
    kind = state["kind"]
    if kind == "observe":
        tr = state["transforms"]
        for frame, view in zip(state["frames"], state["images"]):
            tr.resize_pad_normalize_into(frame, view)
        pi05 = state["case"]["model"] == "pi05"
        joints, bins = tr._normalize_state(state["joints"], want_bins=pi05, out_bf16=state["state"])
        return {"images": state["images"], "state": state["state"], "joints": joints, "bins": bins,
                "actions": tr.postprocess_actions(state["actions"], state["joints"])}
    if kind == "infer":
        return state["transforms"].infer(state["policy"], state["observation"], state["noise"])
    if kind == "pi05_ids":
        return state["policy"].forward_ids(*state["inputs"])
    return state["policy"].forward(*state["inputs"])


def _transform_work(case):
    """Frames read once and 224 x 224 bf16 written per view; two taps per source pixel across and per intermediate pixel down."""
    h, w, n = case["height"], case["width"], case["views"]
    pixel = 12 if case.get("frames") == "f32_chw" else 3
    rows = max(1, int(h / max(h, w) * 224))
    cols = max(1, int(w / max(h, w) * 224))
    bytes_ = n * (h * w * pixel + 224 * 224 * 3 * 2) + case["chunk"] * (32 * 2 + case["dims"] * 8) + 1024
    return bytes_, n * 3 * (4 * h * max(w, cols) + 4 * max(h, rows) * cols + 3 * 224 * 224)


def work(case):
    kind = case["kind"]
    if kind == "observe":
        bytes_, flops = _transform_work(case)
        return {"bytes": bytes_, "flops": flops}
    n, prompt = case["views"], case["prompt"]
    steps = 10
    if kind == "dm0":
        rows, prefix, chunk = n * 2705, n * 169 + prompt, 50
        vit = 23 * (1024 * 3072 + 1024 * 1024 + 2 * 1024 * 4096)
        down = 9216 * 2048 + 18432 * 4096 + 4096 * 2048
        llm = 2048 * 4096 + 2048 * 2048 + 3 * 2048 * 6144
        expert = 28 * (1024 * 4096 + 2048 * 1024 + 3 * 1024 * 1536)
        keys = prefix + chunk
        flops = 2 * rows * (588 * 1024 + vit) + 23 * n * 16 * 4 * 2705 * 2705 * 64
        flops += 2 * n * (676 * 9216 * 2048 + 169 * 18432 * 4096 + 169 * 4096 * 2048)
        flops += 2 * prefix * (27 * llm + 2048 * 2048) + 27 * 16 * 2 * prefix * prefix * 128      # the last layer only fills its K / V
        flops += steps * (2 * chunk * expert + 28 * 16 * 4 * chunk * keys * 128)
        weights = 588 * 1024 + vit + down + 27 * llm + 2048 * 2048 + expert
        return {"bytes": 2 * weights + 2 * n * 3 * 728 * 728 + prompt * 4096, "flops": flops}
    alloc = PI05_MAX_TOKENS if kind == "pi05_ids" else prompt
    rows, prefix = 256 * n, 256 * n + prompt
    suffix = case["chunk"] + (0 if kind.startswith("pi05") else 1)
    keys = prefix + suffix
    vision = 27 * (1152 * 3456 + 1152 * 1152 + 2 * 1152 * 4304)
    llm = 2048 * 2560 + 2048 * 2048 + 3 * 2048 * 16384
    expert = 18 * (1024 * 2560 + 2048 * 1024 + 3 * 1024 * 4096)
    flops = 2 * rows * (588 * 1152 + vision + 1152 * 2048) + 27 * n * 16 * 4 * 256 * 256 * 72
    flops += 2 * prefix * (17 * llm + 2048 * 512) + 17 * 8 * 4 * prefix * prefix * 256            # the last layer only fills its K / V
    flops += steps * (2 * suffix * expert + 18 * 8 * 4 * suffix * keys * 256)
    weights = 588 * 1152 + vision + 1152 * 2048 + 17 * llm + 2048 * 512 + expert
    bytes_ = 2 * weights + n * 224 * 224 * 3 * 2 + alloc * 4096 + case["chunk"] * 32 * 4
    if kind == "infer":
        more = _transform_work(case)
        bytes_, flops = bytes_ + more[0], flops + more[1]
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    # the transforms reproduce 8-bit resampling and double-precision statistics bit for bit; a forward is bf16 storage with fp32
    # sums through up to 80 layers and ten integration steps
    return "exact" if case["kind"] == "observe" else {"rel": 1e-2}
