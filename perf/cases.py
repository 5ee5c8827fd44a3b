"""Timing cases of the feed-forward block, the generalized linear layer and the block-sparse projections.

A case is a dict of plain values:

  call      "train": forward + backward of LeanFFN, returning the output, the input's gradient and every parameter's
            "infer": forward alone under no_grad in eval mode
            "linear": forward + backward of a stand-alone GeneralizedLinear (attention projections)
  dtype     "fp32" / "bf16" / "fp16": parameters and compute in that type; "autocast": fp32 parameters, bf16 compute
  stream    type of the block's input and output, the residual stream: "fp32", or "same" as the parameters
  batch, seq, hidden, inter, gated, act, dropout, post_ln
  layout    "" for dense projections, else the block-sparse layout descriptor of both of them
  rank      low-rank term of block-sparse projections; adapter of a "linear" case (out features = "inter" there)
"""
import torch

import lean_transformer_amd as lt

DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16, "autocast": torch.float32}


def _case(name, call, dtype, batch, seq, hidden, inter, **more):
    case = dict(name=name, call=call, dtype=dtype, stream="fp32", batch=batch, seq=seq, hidden=hidden, inter=inter,
                gated=True, act="gelu_fused", dropout=0.0, post_ln=False, layout="", rank=0)
    case.update(more)
    return case


def listed():
    return [
        # one step of token-by-token generation, eight sequences, on a layer of the small GPT the tests train
        _case("decode_small", "infer", "bf16", 8, 1, 768, 3072, stream="same"),
        # the same for one sequence on the widest benchmark layer: every weight is read for one token
        _case("decode_large", "infer", "bf16", 1, 1, 4096, 16384, stream="same"),
        # a prompt entering a mid-sized layer (benchmark configuration 2's) before generation starts
        _case("prefill", "infer", "bf16", 1, 512, 2048, 8192, gated=False, stream="same"),
        # a unit-test-sized training step: ragged rows, post-LayerNorm, nothing but launches and latency
        _case("train_tiny_fp32", "train", "fp32", 3, 33, 96, 160, post_ln=True, act="gelu"),
        # benchmark configuration 1: fp32 training
        _case("train_fp32", "train", "fp32", 8, 512, 768, 3072),
        # benchmark configuration 2: plain GELU, dropout
        _case("train_gelu_dropout", "train", "bf16", 4, 2048, 2048, 8192, gated=False, dropout=0.1),
        # benchmark configuration 3, the headline: wide GeGLU layer
        _case("train_wide", "train", "bf16", 2, 2048, 4096, 16384),
        # one layer of the GPT train step (configuration 5): mixed precision over fp32 parameters, many tokens, narrow layer
        _case("train_gpt_layer", "train", "autocast", 16, 1024, 768, 3072),
        # float16 parameters, sizes off every tile grid (hidden 1600), a batch that is not a multiple of anything
        _case("train_ragged_fp16", "train", "fp16", 3, 1111, 1600, 6400, act="silu", gated=False),
        # benchmark configuration 4: PixelFly projections, stretched butterfly, rank-128 term
        _case("train_sparse", "train", "bf16", 2, 2048, 4096, 16384, layout="pixelfly(block_size=64, stretch=True)", rank=128),
        # the reference's default layout (tiled butterfly) on a quarter-width layer
        _case("train_sparse_tiled", "train", "bf16", 4, 1000, 1024, 4096, layout="pixelfly(block_size=64)", rank=64),
        # fused query / key / value projection of the GPT's attention, with a per-layer low-rank adapter
        _case("linear_qkv", "linear", "autocast", 16, 1024, 768, 2304, rank=16),
    ]


def _log(rng, lo, hi):
    return lo * (hi / lo) ** rng.random()


def _width(rng, lo, hi, step):
    return max(step, int(round(_log(rng, lo, hi) / step)) * step)


def draw(rng):
    """One more case of the same ranges: token counts are any integer, widths are multiples of 64 (three in four) or of 8;
    training flops stay below the widest listed case's."""
    family = rng.choice(["decode", "prefill", "train", "train", "train", "tiny", "sparse", "linear"])
    step = 64 if rng.random() < 0.75 else 8
    half = rng.choice(["bf16", "bf16", "fp16"])
    if family in ("decode", "prefill"):
        hidden = _width(rng, 512, 4096, step)
        tokens = int(_log(rng, 1, 64.99)) if family == "decode" else int(_log(rng, 65, 2048))
        case = _case("", "infer", rng.choice([half, half, "fp32"]), tokens if family == "decode" else 1,
                     1 if family == "decode" else tokens, hidden, 4 * hidden, gated=rng.random() < 0.5,
                     act=rng.choice(["gelu_fused", "gelu_fused", "silu", "gelu"]), stream=rng.choice(["same", "fp32"]))
        if case["dtype"] == "fp32" and tokens * hidden * hidden > 2e9:
            case["dtype"] = half  # (fp32 prompts on the narrower layers only)
    elif family == "train":
        dtype = rng.choice([half, half, "autocast", "fp32"])
        gated = rng.random() < 0.5
        most = 2.5e11 if dtype == "fp32" else 4.0e12  # flops of a pass
        hidden = _width(rng, 512, 2048 if dtype == "fp32" else 4096, step)
        tokens = int(min(_log(rng, 128, 16384), most / (6.0 * hidden * 4 * hidden * (3 if gated else 2))))
        case = _case("", "train", dtype, 1, tokens, hidden, 4 * hidden, gated=gated,
                     act=rng.choice(["gelu_fused", "gelu_fused", "gelu_fused", "silu"]), dropout=rng.choice([0.0, 0.0, 0.1]),
                     post_ln=rng.random() < 0.15)
    elif family == "tiny":
        hidden = 8 * rng.randint(4, 32)
        case = _case("", "train", rng.choice(["fp32", "fp32", "bf16"]), rng.randint(1, 4), rng.randint(1, 64), hidden,
                     8 * rng.randint(4, 64), gated=rng.random() < 0.5, post_ln=rng.random() < 0.5)
    elif family == "sparse":
        hidden = rng.choice([512, 1024, 2048, 4096])
        case = _case("", "train", half, 1, int(_log(rng, 256, 4096)), hidden, 4 * hidden, gated=rng.random() < 0.75,
                     layout=f"pixelfly(block_size=64, stretch={rng.random() < 0.5})", rank=rng.choice([0, 64, 128]))
    else:
        hidden = _width(rng, 256, 2048, 64)
        case = _case("", "linear", rng.choice(["autocast", half, "fp32"]), 1, int(_log(rng, 64, 16384)), hidden,
                     rng.choice([1, 3]) * hidden, rank=rng.choice([0, 8, 16, 64]))
        if case["dtype"] == "fp32":
            case["seq"] = min(case["seq"], 4096)
    del case["name"]
    return case


def prepare(case, seed):
    """The module, its input and the upstream gradient, all on the GPU and all made from the seed"""
    device = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=device).manual_seed(seed)
    hidden, inter = case["hidden"], case["inter"]
    dtype = DTYPES[case["dtype"]]
    io = dtype if case["stream"] == "same" else torch.float32

    with device:  # parameters are created on the GPU
        if case["call"] == "linear":
            module = lt.GeneralizedLinear(lt.GeneralizedMatrix(hidden, inter), case["rank"])
            io = dtype
        else:
            up_width = 2 * inter if case["gated"] else inter
            projections = {}
            if case["layout"]:
                projections = dict(
                    i2h_proj=lt.GeneralizedLinear(lt.GeneralizedMatrix(hidden, up_width, case["layout"], case["rank"])),
                    h2o_proj=lt.GeneralizedLinear(lt.GeneralizedMatrix(inter, hidden, case["layout"], case["rank"])))
            module = lt.LeanFFN(hidden, inter, activation=lt.ACT2FN[case["act"]], gated=case["gated"], layer_norm_eps=1e-5,
                                dropout=case["dropout"], post_layer_norm=case["post_ln"], **projections)
    module = module.to(device=device, dtype=dtype).train(case["call"] != "infer")
    with torch.no_grad():
        for name, p in module.named_parameters():
            p.normal_(std=0.02, generator=gen)
            if name.endswith("layer_norm.weight"):
                p.add_(1.0)
    rows = (case["batch"], case["seq"])
    x = torch.randn(*rows, hidden, device=device, generator=gen).to(io)
    state = dict(call=case["call"], module=module, autocast=case["dtype"] == "autocast", x=x)
    if case["call"] != "infer":
        out_dtype = io if case["call"] != "linear" else torch.bfloat16 if state["autocast"] else dtype
        state["x"] = x.requires_grad_(True)
        state["wrt"] = [state["x"], *module.parameters()]
        state["dy"] = torch.randn(*rows, hidden if case["call"] == "train" else inter, device=device,
                                  generator=gen).to(out_dtype)
    torch.cuda.manual_seed(seed)  # the stream dropout draws from
    return state


def run(state):
    if state["call"] == "infer":
        with torch.no_grad():
            return state["module"](state["x"])
    if state["autocast"]:
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = state["module"](state["x"])
    else:
        y = state["module"](state["x"])
    return [y.detach(), *torch.autograd.grad(y, state["wrt"], state["dy"])]


def _active_share(case):
    """share of a projection's weights that a block-sparse layout keeps"""
    if not case["layout"]:
        return 1.0
    blocks = case["hidden"] // 64
    return (blocks.bit_length() - 1 + 1) / blocks


def work(case):
    tokens, hidden, inter, rank = case["batch"] * case["seq"], case["hidden"], case["inter"], case["rank"]
    size = {"fp32": 4, "autocast": 4}.get(case["dtype"], 2)
    if case["call"] == "linear":
        weights = hidden * inter + rank * (hidden + inter)
        moved = tokens * (2 * hidden + 2 * inter)  # x, dx, y, dy
        io = size
    else:
        up = 2 * inter if case["gated"] else inter
        weights = _active_share(case) * hidden * (up + inter) + rank * (2 * hidden + up + inter)
        moved = tokens * hidden * (2 if case["call"] == "infer" else 4)
        io = 4 if case["stream"] == "fp32" else size
    passes = 1 if case["call"] == "infer" else 3
    return {"bytes": weights * size * (1 if passes == 1 else 2) + moved * io, "flops": 2.0 * passes * tokens * weights}


def tolerance(case):
    # Largest 2-norm error of any output against the same computation in float64 from the same (rounded) parameters, over
    # these cases and ten drawn ones: 1.0e-6 in fp32, 5.4e-4 in fp16, 5.4e-3 in bf16.  The bars are three to five times that.
    if case["dtype"] == "fp32":
        return {"rel": 5e-6}
    return {"rel": 2e-3} if case["dtype"] == "fp16" else {"rel": 1.5e-2}
