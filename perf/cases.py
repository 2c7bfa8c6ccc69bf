"""The work that a user of the library has it do, as cases to be timed.

A case is one call of the mixture-of-experts layer for one batch, through the
entry points of gpt_oss_amd.abi.  What varies is what varies in use:

  entry    "forward": router and layer in one call, the result overwrites `out`;
           "block":   the FFN block in place on the bf16 residual stream (RMS
                      norm in front, residual add behind);
           "experts": the caller runs the router itself, clears its sum and has
                      the layer added to it, as the runner behind the C++ shim
                      does (ids of a token are distinct, which the shim says);
  weights  "bf16" or "mxfp4" expert matrices;
  experts  8, 32 or 128, always top-4;
  hidden, inter  2880 x 2880 as the 20B and 120B shapes have, or smaller ones;
  tokens   1 (one user) to 7168 (a long prompt);
  zipf     exponent of the experts' popularity, 0 for even routing;
  done     share of the rows that are inactive (finished sequences, pos < 0).
"""
import math

import numpy as np
import torch

from gpt_oss_amd import abi, synth

TOPK = 4
LIMIT = 7.0


def _case(name, entry, weights, tokens, experts=32, hidden=2880, inter=2880, zipf=0.0, done=0.0):
    return {"name": name, "entry": entry, "weights": weights, "tokens": tokens, "experts": experts,
            "hidden": hidden, "inter": inter, "zipf": zipf, "done": done}


def listed():
    return [
        # a test-sized model: launches and latency are all there is
        _case("small_64", "forward", "bf16", 64, experts=8, hidden=256, inter=256),
        # decode for one user
        _case("decode_1_mxfp4", "forward", "mxfp4", 1),
        # decode for a few users, the 120B shape, as part of a transformer block
        _case("decode_6_mxfp4_e128", "block", "mxfp4", 6, experts=128),
        # decode batches of a small server
        _case("decode_24_bf16", "experts", "bf16", 24),
        _case("decode_64_mxfp4", "forward", "mxfp4", 64),
        # decode batches of a busy server, some sequences finished
        _case("decode_200_mxfp4_e128", "block", "mxfp4", 200, experts=128, done=0.1),
        _case("decode_896_bf16", "experts", "bf16", 896, done=0.25),
        # short prompts with uneven routing
        _case("prefill_512_bf16_zipf", "forward", "bf16", 512, zipf=1.2),
        # long prompts: even and uneven routing, both weight formats, both expert counts
        _case("prefill_4096_bf16", "forward", "bf16", 4096),
        _case("prefill_4096_mxfp4", "block", "mxfp4", 4096),
        _case("prefill_7168_bf16_zipf", "forward", "bf16", 7168, zipf=1.2),
        _case("prefill_6144_bf16_e128", "forward", "bf16", 6144, experts=128),
    ]


def draw(rng):
    experts = rng.choice((8, 32, 32, 128))
    most = 6144 if experts == 128 else 7168
    tokens = min(most, int(round(math.exp(rng.uniform(0.0, math.log(most))))))
    hidden = inter = 2880
    if rng.random() < 0.3:
        hidden, inter = (32 * int(round(math.exp(rng.uniform(math.log(8), math.log(90))))) for _ in range(2))
    c = _case("", rng.choice(("forward", "forward", "block", "experts")), rng.choice(("bf16", "mxfp4")), tokens,
              experts, hidden, inter, rng.choice((0.0, 0.0, 0.6, 1.2)),
              round(rng.uniform(0.05, 0.5), 2) if tokens > 8 and rng.random() < 0.3 else 0.0)
    del c["name"]
    return c


def _pinned(t):
    """A device tensor as a numpy array in page-locked host memory, from where the upload is quick."""
    return torch.empty(t.shape, dtype=t.dtype, pin_memory=True).copy_(t).numpy()


def _upload(moe, case, gen):
    """Random weights of a trained layer's scale: N(0, 0.02), or MXFP4 codes with
    block scales of 2^-9 to 2^-6, which spread as far; router bias N(0, 0.1), or
    bent so that the experts' popularity follows Zipf's law."""
    E, H, IM = case["experts"], case["hidden"], case["inter"]

    def normal(*shape, std=0.02):
        return torch.randn(shape, generator=gen, device="cuda").mul_(std)

    wr, br = normal(E, H), normal(E, std=0.1)
    if case["zipf"]:
        # logits spread by about 0.02 * sqrt(H): 0.65 of that per unit of log popularity
        lift = 0.65 * 0.02 * math.sqrt(H) * np.log(synth.zipf_popularity(E, case["zipf"]))
        br += torch.from_numpy(lift.astype(np.float32)).cuda()
    wr, br, b1, b2 = (_pinned(t) for t in (wr, br, normal(E, 2 * IM), normal(E, H)))
    if case["weights"] == "bf16":
        moe.upload_layer(0, wr, br, _pinned(normal(E, 2 * IM, H)), b1, _pinned(normal(E, H, IM)), b2)
    else:
        def codes(rows, cols):
            b = torch.randint(0, 256, (E, rows, cols // 32, 16), generator=gen, device="cuda", dtype=torch.uint8)
            s = torch.randint(118, 122, (E, rows, cols // 32), generator=gen, device="cuda", dtype=torch.uint8)
            return _pinned(b), _pinned(s)

        moe.upload_layer_mxfp4(0, wr, br, *codes(2 * IM, H), b1, *codes(H, IM), b2)


def prepare(case, seed):
    """Layer, batch and buffers of a user's program: the weights uploaded, the
    rows RMS-normalised bf16 (for "block" the residual stream, whose rows differ in size)."""
    T, E, H = case["tokens"], case["experts"], case["hidden"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    moe = abi.Moe(H, case["inter"], E, max_tokens=1024 if T <= 1024 else 8192, swiglu_limit=LIMIT)
    _upload(moe, case, gen)
    x = torch.randn((T, H), generator=gen, device="cuda")
    x /= x.square().mean(dim=1, keepdim=True).add(1e-5).sqrt()
    state = {"moe": moe, "entry": case["entry"], "tokens": T, "pos": None}
    if case["done"]:
        pos = torch.randint(0, 1000, (T,), generator=gen, device="cuda", dtype=torch.int32)
        # exactly the stated share (work() counts on it), at random places
        pos[torch.randperm(T, generator=gen, device="cuda")[:int(T * case["done"])]] = -1
        state["pos"] = pos
    if case["entry"] == "block":
        x *= torch.rand((T, 1), generator=gen, device="cuda") * 3.5 + 0.5
        moe.upload_norm(0, _pinned(1.0 + 0.1 * torch.randn(H, generator=gen, device="cuda")))
        state["stream"] = torch.empty((T, H), device="cuda", dtype=torch.bfloat16)
    else:
        state["out"] = torch.zeros((T, H), device="cuda")
    if case["entry"] == "experts":
        moe.set_distinct_ids(True)
        state["topk_i"] = torch.empty((T, TOPK), device="cuda", dtype=torch.int32)
        state["topk_v"] = torch.empty((T, TOPK), device="cuda")
    state["x"] = x.to(torch.bfloat16)
    torch.cuda.synchronize()
    return state


def _ptr(t):
    return None if t is None else t.data_ptr()


def run(state):
    moe, T, x, pos = state["moe"], state["tokens"], state["x"], _ptr(state["pos"])
    stream = torch.cuda.current_stream().cuda_stream
    if state["entry"] == "block":
        # the residual stream as the layers in front of the block leave it
        s = state["stream"]
        s.copy_(x)
        moe.block_forward(0, _ptr(s), pos, T, stream=stream)
        return s
    out = state["out"]
    if state["entry"] == "forward":
        moe.forward(0, _ptr(x), pos, T, _ptr(out), stream=stream)
        return out
    ti, tv = state["topk_i"], state["topk_v"]
    moe.router(0, _ptr(x), pos, T, None, _ptr(ti), _ptr(tv), stream=stream)
    out.zero_()
    moe.experts(0, _ptr(x), pos, _ptr(ti), _ptr(tv), T, _ptr(out), accumulate=True, stream=stream)
    return {"out": out, "topk_i": ti, "topk_v": tv}


def _experts_reached(case, rows):
    """How many experts a batch names, in expectation (a token takes four of them, by popularity)."""
    share = np.minimum(1.0, TOPK * synth.zipf_popularity(case["experts"], case["zipf"]))
    return float((1.0 - (1.0 - share) ** rows).sum())


def work(case):
    T, E, H, IM = case["tokens"], case["experts"], case["hidden"], case["inter"]
    rows = T - int(T * case["done"])
    w = 2.0 if case["weights"] == "bf16" else 0.5 + 1.0 / 32
    weights = _experts_reached(case, rows) * (3.0 * H * IM * w + (2 * IM + H) * 4)
    stream = rows * H * (2 + (2 if case["entry"] == "block" else 4)) + E * H * 2
    return {"bytes": weights + stream, "flops": rows * (TOPK * 6.0 * H * IM + 2.0 * E * H)}


def tolerance(case):
    """The activation between the two products is rounded to bf16: sums taken in
    another order move a few of those roundings, and one moved rounding weighs the
    more the fewer rows are looked at.  Against the same layer in 64 bits, rounded
    at the same place, the fp32 result was off by at most 1.4e-4 (one value: 1.3e-3)
    over 30 sets of inputs at 1, 8 and 24 rows; the block's result is a bf16 stream,
    of which a few values land one step away (3.5e-4, 7.6e-3).  Four times that.
    Expert ids are defined bit for bit."""
    return {"rel": 1.4e-3, "max": 3e-2} if case["entry"] == "block" else {"rel": 5.5e-4, "max": 5.5e-3}
