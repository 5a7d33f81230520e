"""The work that programs have the norm / activation / embedding layers do, as timed cases.

Eight kinds of pass, each a call sequence out of a Stable Diffusion pipeline (convolutions and
matrix products between the calls belong to the application: their results are inputs here):

  tick         what a sampler step does outside the UNet: sinusoidal timestep embedding, the two
               time-embedding Linear layers, the DDIM update of the latent
  projections  the 22 per-ResBlock SiLU -> Linear projections of the time embedding
  text         the 12 layers of the text encoder: LayerNorm, residual adds, GELU / quick_GELU
  step         every norm / activation / embedding / add launch of one UNet step, recorded once as
               a HIP graph and replayed, as a sampler loop does
  resblock     the norms of one ResBlock and its skip add, called eagerly
  transformer  the norms of one SpatialTransformer block, GEGLU, the adds and the permute back
  attention    the row softmax of the self- and cross-attention scores of one block
  decoder      the norms of one ResBlock of the image decoder and its skip add

Latents of a 512-pixel image are 64 x 64; the UNet halves them three times, so their sides are
multiples of eight and the deeper levels get odd sizes (576 x 448 pixels: 72 x 56, ..., 9 x 7).
"""
import importlib
import math

import torch

msd = importlib.import_module("mobile-stable-diffusion_amd")

DTYPES = {"f16": torch.float16, "f32": torch.float32}

# (channels in, channels out, level, followed by a SpatialTransformer) of the UNet's 22 ResBlocks in
# execution order; level l works on latents of 1 / 2^l of the side
RESBLOCKS = (
    [(320, 320, 0, True)] * 2 + [(320, 640, 1, True), (640, 640, 1, True), (640, 1280, 2, True), (1280, 1280, 2, True)] +
    [(1280, 1280, 3, False)] * 2 + [(1280, 1280, 3, True), (1280, 1280, 3, False)] + [(2560, 1280, 3, False)] * 3 +
    [(2560, 1280, 2, True)] * 2 + [(1920, 1280, 2, True)] +
    [(1920, 640, 1, True), (1280, 640, 1, True), (960, 640, 1, True)] +
    [(960, 320, 0, True), (640, 320, 0, True), (640, 320, 0, True)]
)
HEADS, TEXT_TOKENS, TEXT_LAYERS = 8, 77, 12
EMBED = 1280  # channels of the time embedding


# ----------------------------------------------------------------------------------------
# the cases
# ----------------------------------------------------------------------------------------
def listed():
    return [
        # one prompt with classifier-free guidance: the smallest calls there are, one after the other
        {"name": "tick_b2_f32", "kind": "tick", "batch": 2, "h": 64, "w": 64, "dtype": "f32"},
        # prompt and empty prompt through the text encoder, once per image; fp32 as it is shipped
        {"name": "text_b2_f32", "kind": "text", "batch": 2, "dim": 768, "act": "gelu", "dtype": "f32"},
        # once per sampler step, all weights read once
        {"name": "projections_b2_f16", "kind": "projections", "batch": 2, "dtype": "f16"},
        # the interactive case: one 512 x 512 image with guidance, a graph replay per sampler step
        {"name": "step_512x512_b2_f16", "kind": "step", "batch": 2, "h": 64, "w": 64, "dtype": "f16"},
        # another aspect ratio: 72 x 56 latents, 9 x 7 at the deepest level
        {"name": "step_576x448_b2_f16", "kind": "step", "batch": 2, "h": 72, "w": 56, "dtype": "f16"},
        # the reference's own form: one sample at a time, fp32
        {"name": "step_512x512_b1_f32", "kind": "step", "batch": 1, "h": 64, "w": 64, "dtype": "f32"},
        # serving: eight images with guidance through the widest level
        {"name": "resblock_320_64x64_b16_f16", "kind": "resblock", "batch": 16, "cin": 320, "cout": 320,
         "h": 64, "w": 64, "inplace": True, "dtype": "f16"},
        # one image, eager calls
        {"name": "transformer_640_32x32_b2_f16", "kind": "transformer", "batch": 2, "dim": 640, "h": 32, "w": 32,
         "dtype": "f16"},
        # serving: eight images with guidance
        {"name": "transformer_320_64x64_b16_f16", "kind": "transformer", "batch": 16, "dim": 320, "h": 64, "w": 64,
         "dtype": "f16"},
        # the first level's attention scores, one image with guidance
        {"name": "attention_64x64_b2_f16", "kind": "attention", "batch": 2, "h": 64, "w": 64, "stable": False,
         "dtype": "f16"},
        # the same for a 768 x 768 image: 9216 keys per row, the largest tensors of the path
        {"name": "attention_96x96_b2_f16", "kind": "attention", "batch": 2, "h": 96, "w": 96, "stable": False,
         "dtype": "f16"},
        # the decoder's last level: one 512 x 512 image at full resolution
        {"name": "decoder_128_512x512_b1_f32", "kind": "decoder", "batch": 1, "channels": 128, "h": 512, "w": 512,
         "dtype": "f32"},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _draw(rng):
    kind = rng.choice(["tick", "projections", "text", "step", "step", "resblock", "resblock", "transformer",
                       "transformer", "attention", "attention", "decoder"])
    half = "f16" if rng.random() < 0.7 else "f32"
    # image sides from 256 to 768 pixels in steps of 64: latents from 4 x 4 blocks of eight to 12 x 12
    h8, w8 = rng.randint(4, 12), rng.randint(4, 12)
    if kind == "tick":
        return {"kind": kind, "batch": rng.randint(1, 8), "h": 8 * h8, "w": 8 * w8, "dtype": rng.choice(["f16", "f32"])}
    if kind == "projections":
        return {"kind": kind, "batch": rng.randint(1, 8), "dtype": half}
    if kind == "text":
        return {"kind": kind, "batch": _log_int(rng, 1, 16), "dim": rng.choice([768, 1024]),
                "act": rng.choice(["gelu", "quick_gelu"]), "dtype": rng.choice(["f16", "f32"])}
    if kind == "step":
        return {"kind": kind, "batch": _log_int(rng, 1, 8), "h": 8 * h8, "w": 8 * w8, "dtype": half}
    if kind == "decoder":
        channels, scale = rng.choice([(512, 1), (512, 2), (256, 4), (128, 8)])
        return {"kind": kind, "batch": rng.randint(1, 3), "channels": channels, "h": 8 * h8 * scale, "w": 8 * w8 * scale,
                "dtype": rng.choice(["f16", "f32"])}
    level = rng.randint(0, 3)
    batch, h, w = _log_int(rng, 1, 32), (8 >> level) * h8, (8 >> level) * w8
    if kind == "resblock":
        cin, cout = rng.choice(sorted({(i, o) for i, o, l, _ in RESBLOCKS if l == level}))
        return {"kind": kind, "batch": batch, "cin": cin, "cout": cout, "h": h, "w": w,
                "inplace": cin == cout and rng.random() < 0.7, "dtype": half}
    if kind == "transformer":
        return {"kind": kind, "batch": batch, "dim": (320, 640, 1280, 1280)[level], "h": h, "w": w, "dtype": half}
    return {"kind": kind, "batch": _log_int(rng, 1, 8), "h": h, "w": w, "stable": rng.random() < 0.5, "dtype": half}


def draw(rng):
    most = max(work(c)["bytes"] for c in listed())
    while True:
        case = _draw(rng)
        if work(case)["bytes"] <= most:
            return case


# ----------------------------------------------------------------------------------------
# what each pass cannot do without
# ----------------------------------------------------------------------------------------
def _size(case):
    return 2 if case["dtype"] == "f16" else 4


def _transformer_work(batch, dim, hw):
    """(elements moved, flops) of one SpatialTransformer's calls."""
    n = batch * dim * hw
    # tokens norm: read, write; first LayerNorm: read, write; two fused adds: two read, two written
    # each; GEGLU: 8 n in, 4 n out; feed-forward add: 2 in, 1 out; permute: 1 + 1; outer add: 2 + 1
    return (2 + 2 + 8 + 12 + 3 + 2 + 3) * n, (10 * 4 + 20 * 4 + 2) * n


def _tick_work(batch, latent, elt):
    weights = EMBED * 320 + EMBED * EMBED
    return weights * elt + 2 * EMBED * 4 + 3 * latent * elt, 2 * batch * weights + 5 * latent


def _projection_work(batch, elt):
    rows = sum(cout for _, cout, _, _ in RESBLOCKS)
    return rows * EMBED * elt + batch * (EMBED + rows) * elt + 4 * rows, 2 * batch * rows * EMBED


def work(case):
    elt, b, kind = _size(case), case["batch"], case["kind"]
    if kind == "tick":
        nbytes, flops = _tick_work(b, b * 4 * case["h"] * case["w"], elt)
    elif kind == "projections":
        nbytes, flops = _projection_work(b, elt)
    elif kind == "text":
        n = b * TEXT_TOKENS * case["dim"]
        # per layer: LayerNorm 2, fused add + LayerNorm 4, activation 4 n in and out, add 3; last norm 2
        nbytes, flops = (TEXT_LAYERS * (2 + 4 + 8 + 3) + 2) * n * elt, TEXT_LAYERS * (10 * 2 + 16 * 4 + 1) * n
    elif kind == "step":
        nbytes, flops = 0, 0
        for cin, cout, level, transformer in RESBLOCKS:
            hw = (case["h"] >> level) * (case["w"] >> level)
            nbytes += b * hw * (2 * cin + 2 * cout + 3 * cout) * elt
            flops += b * hw * (14 * cin + 16 * cout)
            if transformer:
                moved, done = _transformer_work(b, cout, hw)
                nbytes, flops = nbytes + moved * elt, flops + done
        last = b * 320 * case["h"] * case["w"]
        nbytes, flops = nbytes + 2 * last * elt, flops + 14 * last
        for more, done in (_tick_work(b, b * 4 * case["h"] * case["w"], elt), _projection_work(b, elt)):
            nbytes, flops = nbytes + more, flops + done
    elif kind == "resblock":
        hw = case["h"] * case["w"]
        nbytes, flops = b * hw * (2 * case["cin"] + 5 * case["cout"]) * elt, b * hw * (14 * case["cin"] + 16 * case["cout"])
    elif kind == "transformer":
        moved, flops = _transformer_work(b, case["dim"], case["h"] * case["w"])
        nbytes = moved * elt
    elif kind == "attention":
        hw = case["h"] * case["w"]
        n = b * HEADS * hw * (hw + TEXT_TOKENS)
        nbytes, flops = 2 * n * elt, 4 * n
    else:  # decoder
        n = b * case["channels"] * case["h"] * case["w"]
        nbytes, flops = 7 * n * elt, 29 * n
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # float16 results are float32 arithmetic rounded once: another summation order flips a last bit
    # (2^-11 of the value) here and there; against sums in 64 bits 1e-5 to 2e-5 in all, 3e-3 (a last
    # bit of a first result and what the second norm makes of it) at most.  float32: 7e-8 to 1.5e-7
    # in all, 1.2e-6 at most.
    if case["dtype"] == "f16":
        return {"rel": 8e-5, "max": 1.2e-2}
    return {"rel": 6e-7, "max": 5e-6}


# ----------------------------------------------------------------------------------------
# inputs and passes
# ----------------------------------------------------------------------------------------
class _Inputs:
    """Tensors made on the GPU from one seed."""

    def __init__(self, seed, dtype):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.dtype = dtype

    def normal(self, *shape, sigma=1.0, mean=0.0):
        return torch.empty(shape, dtype=self.dtype, device="cuda").normal_(mean, sigma, generator=self.gen)

    def affine(self, channels):
        weight = torch.empty(channels, device="cuda").normal_(1.0, 0.1, generator=self.gen)
        return weight, torch.empty(channels, device="cuda").normal_(0.0, 0.1, generator=self.gen)

    def linear(self, n, k):
        weight = self.normal(n, k, sigma=k ** -0.5)
        return weight, torch.empty(n, device="cuda").normal_(0.0, 0.1, generator=self.gen)


class _Tick:
    def __init__(self, case, inp):
        b = case["batch"]
        self.dtype = inp.dtype
        self.t = torch.randint(0, 1000, (b,), device="cuda", generator=inp.gen)
        self.fc1, self.fc2 = inp.linear(EMBED, 320), inp.linear(EMBED, EMBED)
        self.latent, self.noise = (inp.normal(b, 4, case["h"], case["w"]) for _ in range(2))
        _, alphas, previous, sigma = msd.ddim_schedule(50)
        self.coefficients = alphas[25], previous[25], sigma[25]

    def embedding(self):
        temb = msd.timestep_embedding(self.t, 320, dtype=self.dtype)
        hidden = msd.linear_rows(temb, *self.fc1, act_out=msd.ACT_SILU)
        return msd.linear_rows(hidden, *self.fc2)

    def run(self):
        emb = self.embedding()
        return emb, msd.ddim_update(self.latent, self.noise, *self.coefficients)


class _Projections:
    def __init__(self, case, inp):
        self.emb = inp.normal(case["batch"], EMBED)
        layers = [inp.linear(cout, EMBED) for _, cout, _, _ in RESBLOCKS]
        self.weights, self.biases = [w for w, _ in layers], [b for _, b in layers]

    def run(self):
        return msd.linear_rows_grouped(self.emb, self.weights, self.biases, act_in=msd.ACT_SILU)


class _Text:
    def __init__(self, case, inp):
        shape = (case["batch"], TEXT_TOKENS, case["dim"])
        self.x = inp.normal(*shape)
        self.layers = [(inp.affine(case["dim"]), inp.affine(case["dim"]), inp.normal(*shape), inp.normal(*shape[:2], 4 * shape[2]),
                        inp.normal(*shape)) for _ in range(TEXT_LAYERS)]
        self.last = inp.affine(case["dim"])
        self.act = msd.gelu if case["act"] == "gelu" else msd.quick_gelu

    def run(self):
        x, outs = self.x, []
        for norm1, norm2, attended, hidden, fed in self.layers:
            outs.append(msd.layernorm(x, *norm1))
            x, normed = msd.add_layernorm(attended, x, *norm2)
            outs += [normed, self.act(hidden)]
            x = msd.elemwise_add(fed, x)
        return outs + [msd.layernorm(x, *self.last)]


class _ResBlock:
    """In-norm, embedding add + out-norm, skip add.  `inplace`: the out-norm works on the buffer the
    in-norm filled (the convolution between them keeps it there), as the blocks of equal width do."""

    def __init__(self, case, inp, out=None):
        b, cin, cout, h, w = (case[k] for k in ("batch", "cin", "cout", "h", "w"))
        self.x = inp.normal(b, cin, h, w, sigma=2.0)
        self.hidden = None if case["inplace"] else inp.normal(b, cout, h, w)
        self.emb = inp.normal(b, cout)
        self.skip, self.conv = (inp.normal(b, cout, h, w) for _ in range(2))
        self.norm1, self.norm2 = inp.affine(cin), inp.affine(cout)
        out = out or (lambda like: None)
        self.out1, self.out3 = out(self.x), out(self.conv)
        self.out2 = None if case["inplace"] else out(self.hidden)

    def run(self, emb=None):
        first = msd.groupnorm(self.x, *self.norm1, 32, fuse_silu=True, out=self.out1)
        hidden, out = (first, first) if self.hidden is None else (self.hidden, self.out2)
        second = msd.chunk_add_groupnorm(hidden, self.emb if emb is None else emb, *self.norm2, 32, fuse_silu=True, out=out)
        return first, second, msd.elemwise_add(self.conv, self.skip, out=self.out3)


class _Transformer:
    def __init__(self, case, inp, out=None):
        b, dim, h, w = (case[k] for k in ("batch", "dim", "h", "w"))
        self.x = inp.normal(b, dim, h, w, sigma=2.0)
        self.attended1, self.attended2, self.fed = (inp.normal(b, h * w, dim) for _ in range(3))
        self.projected = inp.normal(b, h * w, 8 * dim)
        self.norm, self.norms = inp.affine(dim), [inp.affine(dim) for _ in range(3)]
        out = out or (lambda like: None)
        self.outs = [out(self.fed) for _ in range(6)] + [out(self.projected[..., :4 * dim]), out(self.x)]

    def run(self):
        o = self.outs
        tokens = msd.groupnorm_tokens(self.x, *self.norm, 32)
        normed1 = msd.layernorm(tokens, *self.norms[0], out=o[0])
        x1, normed2 = msd.add_layernorm(self.attended1, tokens, *self.norms[1], sum_out=o[1], out=o[2])
        x2, normed3 = msd.add_layernorm(self.attended2, x1, *self.norms[2], sum_out=o[3], out=o[4])
        gated = msd.geglu(self.projected, out=o[6])
        x3 = msd.elemwise_add(self.fed, x2, out=o[5])
        image = msd.permute_0_2_1(x3)
        return tokens, normed1, x1, normed2, x2, normed3, gated, x3, image, msd.elemwise_add(image.view_as(self.x), self.x, out=o[7])


class _Arena:
    """One block of memory that all outputs of a step are cut from; None until it is made."""

    def __init__(self, dtype):
        self.dtype, self.shapes, self.block = dtype, [], None

    def reserve(self, like):
        self.shapes.append(tuple(like.shape))
        return len(self.shapes) - 1

    def make(self):
        starts, end = [], 0
        for shape in self.shapes:
            starts.append(end)
            end += -(-math.prod(shape) // 128) * 128
        self.block = torch.zeros(end, dtype=self.dtype, device="cuda")
        return [self.block[s:s + math.prod(shape)].view(shape) for s, shape in zip(starts, self.shapes)]


class _Step:
    """A whole UNet step, recorded once and replayed."""

    def __init__(self, case, inp):
        arena = _Arena(inp.dtype)
        self.tick, self.projections, self.blocks = _Tick(case, inp), _Projections(case, inp), []
        for cin, cout, level, transformer in RESBLOCKS:
            size = {"batch": case["batch"], "h": case["h"] >> level, "w": case["w"] >> level}
            res = _ResBlock(dict(size, cin=cin, cout=cout, inplace=cin == cout), inp, arena.reserve)
            self.blocks.append((res, _Transformer(dict(size, dim=cout), inp, arena.reserve) if transformer else None))
        self.x, self.norm = inp.normal(case["batch"], 320, case["h"], case["w"], sigma=2.0), inp.affine(320)
        last = arena.reserve(self.x)
        views = arena.make()
        for res, transformer in self.blocks:
            res.out1, res.out3 = views[res.out1], views[res.out3]
            res.out2 = None if res.out2 is None else views[res.out2]
            if transformer:
                transformer.outs = [views[i] for i in transformer.outs]
        self.last, self.arena = views[last], arena
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            msd.init()
            self.launch()  # kernels are loaded before they are recorded
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph, stream=stream):
            self.recorded = self.launch()
        torch.cuda.current_stream().wait_stream(stream)

    def launch(self):
        emb = self.tick.embedding()
        self.projections.emb = emb
        projected, outs = self.projections.run(), [emb]
        for (res, transformer), rows in zip(self.blocks, projected):
            res.run(rows)
            if transformer:
                done = transformer.run()
                outs += [done[0], done[8]]  # tokens and image; the rest is in the arena
        msd.groupnorm(self.x, *self.norm, 32, fuse_silu=True, out=self.last)
        tick = self.tick
        return outs + projected + [msd.ddim_update(tick.latent, tick.noise, *tick.coefficients), self.arena.block]

    def run(self):
        self.graph.replay()
        return self.recorded


class _Attention:
    def __init__(self, case, inp):
        b, hw = case["batch"] * HEADS, case["h"] * case["w"]
        self.own, self.text = inp.normal(b, hw, hw, sigma=1.5), inp.normal(b, hw, TEXT_TOKENS, sigma=1.5)
        self.out = torch.empty_like(self.own), torch.empty_like(self.text)
        self.stable = case["stable"]

    def run(self):
        return msd.softmax(self.own, self.stable, out=self.out[0]), msd.softmax(self.text, self.stable, out=self.out[1])


class _Decoder:
    def __init__(self, case, inp):
        shape = tuple(case[k] for k in ("batch", "channels", "h", "w"))
        self.x, self.conv = inp.normal(*shape, sigma=2.0), inp.normal(*shape)
        self.norm1, self.norm2 = inp.affine(shape[1]), inp.affine(shape[1])

    def run(self):
        first = msd.groupnorm(self.x, *self.norm1, 32, eps=1e-6, fuse_silu=True)
        second = msd.groupnorm(first, *self.norm2, 32, eps=1e-6, fuse_silu=True, out=first)
        return second, msd.elemwise_add(self.conv, self.x)


_KINDS = {"tick": _Tick, "projections": _Projections, "text": _Text, "step": _Step, "resblock": _ResBlock,
          "transformer": _Transformer, "attention": _Attention, "decoder": _Decoder}


def prepare(case, seed):
    return _KINDS[case["kind"]](case, _Inputs(seed, DTYPES[case["dtype"]]))


def run(state):
    return state.run()
