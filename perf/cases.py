"""The work that users of this framework have it do, as cases that can be timed and compared.

A case is one pass of one of the five benchmark networks (`rembrandt_amd.configs`) through the operator-level API: a
train step (forward, loss, backward, SGD with momentum), or a forward pass in the inference phase with fp32 or bf16
convolution operands.  What varies is what varies in use: the network, the batch (single images, micro-batches and the
ragged last batch of an epoch, full batches), and where a train step's frames come from (resident in device memory, or
u8 frames staged in host memory that are copied, cast, cropped and flipped on the way in).
"""
import math

import torch

from rembrandt_amd import configs
from rembrandt_amd.operator import SequentialOperatorWorker, SgdOpt

# Standard deviation of the initial filters and affine weights: about 1 / sqrt(fan-in) of the networks' wide layers, so
# that activations and deltas keep their scale through the depth (batch-normalised filters: KaimingFwd, by build_config).
INIT_STD = {"lenet": 0.05, "cifar10": 0.05, "alexnet": 0.02, "nin": 0.05, "resnet18": 0.05}
# Extent of the staged u8 frames: the ImageNet-shaped networks train on random crops of 256 x 256 frames.
RAW_EXTENT = {"lenet": 28, "cifar10": 32, "alexnet": 256, "nin": 256, "resnet18": 256}
NETS = sorted(INIT_STD)
BF16_NETS = ["alexnet", "nin"]   # the networks whose bf16 forward pass the benchmark quotes


def _case(name, net, mode, batch, frames="f32"):
    return {"name": name, "net": net, "mode": mode, "batch": batch, "frames": frames}


def listed():
    return [
        # one digit classified: the smallest call, a handful of dependent launches
        _case("lenet_infer_b1", "lenet", "infer", 1),
        # one image classified by the largest model: every affine weight is read once for it
        _case("alexnet_infer_b1", "alexnet", "infer", 1),
        # a small, odd group of requests through the batch-normalised network
        _case("resnet18_infer_b9", "resnet18", "infer", 9),
        # bf16 serving, an ordinary group of requests and a full batch
        _case("alexnet_infer_bf16_b37", "alexnet", "infer_bf16", 37),
        _case("nin_infer_bf16_b128", "nin", "infer_bf16", 128),
        # training at the configurations' own batch sizes
        _case("lenet_train_b64", "lenet", "train", 64),
        _case("cifar10_train_b128", "cifar10", "train", 128),
        _case("nin_train_b128", "nin", "train", 128),
        _case("alexnet_train_b256", "alexnet", "train", 256),
        _case("resnet18_train_b256", "resnet18", "train", 256),
        # a micro-batch of a larger minibatch
        _case("resnet18_train_b24", "resnet18", "train", 24),
        # an epoch's ragged last batch as a training loop hands it over: u8 frames from host memory, cropped and flipped
        _case("alexnet_train_u8_b50", "alexnet", "train", 50, "u8"),
    ]


def draw(rng):
    """One more case: half of them train steps of 8 to 256 samples (one in four fed from host frames), the others
    inference on 1 to 128 images."""
    mode = rng.choice(["train", "train", "infer", "infer_bf16"])
    net = rng.choice(BF16_NETS if mode == "infer_bf16" else NETS)
    lo, hi = (8, 256) if mode == "train" else (1, 128)
    batch = min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))
    frames = "u8" if mode == "train" and rng.random() < 0.25 else "f32"
    return {"net": net, "mode": mode, "batch": batch, "frames": frames}


class _DeviceArray:
    """An operator's device buffer, for torch.as_tensor; keeps the worker that owns it."""

    def __init__(self, worker, ptr, count):
        self.worker = worker
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": "<f4", "data": (ptr, False), "version": 2}


def _view(worker, idx, which):
    ptr, count = worker.device_ptr(idx, which)
    return torch.as_tensor(_DeviceArray(worker, ptr, count), device="cuda")


def _parameter_buffers(layers):
    """(operator, buffer) of everything a train step updates that a user keeps: parameters and momentum."""
    out = []
    for i, l in enumerate(layers):
        if l[0] in ("conv2d", "affine"):
            out += [(i, "weights"), (i, "bias"), (i, "acc_grad_weights"), (i, "acc_grad_bias")]
        units = {"bnorm_conv2d": 1, "stack_res_conv2d": 2, "proj_stack_res_conv2d": 3}.get(l[0], 0)
        out += [(i, "u%d.%s" % (u, b)) for u in range(units) for b in ("weights", "acc_grad_weights")]
        out += [(i, "u0.acc_bn_scale_grad")] * (units > 0)
    return out


def prepare(case, seed):
    net = configs.NETWORKS[case["net"]]()
    dims, layers, categories = net
    batch, train = case["batch"], case["mode"] == "train"
    gen = torch.Generator(device="cuda").manual_seed(seed)
    cfg = configs.build_config(net, init_std=INIT_STD[case["net"]])
    if case["frames"] == "u8":
        raw = RAW_EXTENT[case["net"]]
        cfg.data3d((raw, raw, dims[2]), normalize=True)
        if raw != dims[0]:
            cfg.crop(dims[0], dims[1])
        if case["net"] != "lenet":
            cfg.flip_x()
    worker = SequentialOperatorWorker(cfg, batch, "Backward" if train else "Forward", shared_seed=(seed, seed + 1),
                                      bf16_forward=case["mode"] == "infer_bf16")
    worker.init_params()
    if case["frames"] == "u8":
        frames = torch.randint(0, 256, (batch, dims[2], raw, raw), generator=gen, device="cuda", dtype=torch.uint8)
        worker.load_frames_u8(frames.cpu().numpy())
    else:
        frames = torch.randn((batch, dims[2], dims[1], dims[0]), generator=gen, device="cuda")
        worker.load_frames_f32(frames.cpu().numpy())
    state = {"worker": worker, "batch": batch, "mode": case["mode"], "frames": case["frames"]}
    # the logits (the last operator's activations) and the probabilities made of them
    state["outputs"] = {"logits": _view(worker, len(layers) - 1, "out_act"), "probs": _view(worker, len(layers), "out_act")}
    if train:
        labels = torch.randint(0, categories, (batch,), generator=gen, device="cuda")
        worker.stage_batch(labels.tolist(), 1.0 / batch)
        state["sgd"] = SgdOpt(batch, 0.001, ("Update", 0.9), 5e-4)
        state["sgd"].begin(worker)
        del state["outputs"]["logits"]   # a train step's caller sees the loss, the hits and the updated parameters
        state["outputs"]["updated"] = [_view(worker, i, b) for i, b in _parameter_buffers(layers)]
    return state


def run(state):
    worker, batch = state["worker"], state["batch"]
    if state["mode"] != "train":
        worker.forward(batch, training=False)
        return state["outputs"]
    if state["frames"] == "u8":   # the staged frames and labels go to the device every step
        worker.reload_frames(batch)
        worker.load_labels(batch)
        worker.load_weights(batch)
    loss, correct = state["sgd"].train_batch(worker, batch, fused=True)
    return {"loss": loss, "correct": correct, **state["outputs"]}


def work(case):
    """FLOPs of the convolutions and affine layers in their direct form; bytes: the frames, and the parameters read once
    (a train step also reads their momentum and writes both)."""
    net = configs.NETWORKS[case["net"]]()
    dims, layers, categories = net
    train = case["mode"] == "train"
    batch, frame = case["batch"], dims[0] * dims[1] * dims[2]
    if case["frames"] == "u8":
        frame = RAW_EXTENT[case["net"]] ** 2 * dims[2] / 4
    params = configs.build_config(net).params_len()
    return {"bytes": 4.0 * (batch * (frame + (1 if train else 2) * categories) + params * (4 if train else 1)),
            "flops": float(configs.train_flops(net, batch, forward_only=not train))}


def tolerance(case):
    """About four times what the path differs by from itself with its sums in another order (direct instead of Winograd
    convolutions, separate instead of fused epilogues and classifier tail; another batch around the same images).

    fp32 inference: 1.2e-6, 5e-6 at the worst value.  bf16 inference: 7e-4 and 6e-3 against the same roundings with sums
    in 64 bits, where a sum a hair off now and then rounds to the next bf16 value.  Train steps: 2e-3 to 7e-3 in the
    deep networks and 3e-7 or as much in the shallow ones, because the gradients are discontinuous: a max-pool window or
    a ReLU on the edge goes the other way in one sample of some millions, and moves that sample's whole share of a
    filter's gradient (0.1 to 0.4 of a typical value where few samples add up)."""
    if case["mode"] == "train":
        return {"rel": 0.025, "max": 0.99}
    return {"rel": 3e-3, "max": 2e-2} if case["mode"] == "infer_bf16" else {"rel": 1e-5, "max": 1e-4}
