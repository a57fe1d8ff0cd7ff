"""The work a user of this framework has it do, as measurable cases: the device-resident core (inference and training),
the allocation-free serving call, the layer stack and its nn.Module, the host-streaming module and the fp32 C API, from
one step of one sequence to a training step of a four-layer stack.

A case is a dict of plain values.  `call` names the public entry point, T / B / I / H (/ L) are sequence length, batch
rows, input features, hidden units (layers), `dtype` the element type of the caller's sequences ("f16" or "f32"; the
arithmetic is fp16 with fp32 accumulation either way), `state` whether initial states are handed over, `every` the
checkpoint interval of the host-streaming call.
"""
import ctypes
import math

import torch

import flashlstm_poc_amd as fl


def listed():
    return [
        # one step of one sequence in a serving loop that carries its own state: latency and launches only
        dict(name="serve_step", call="serve", T=1, B=1, I=128, H=256, dtype="f16", state=True),
        # scoring a batch of sequences, no gradients kept
        dict(name="infer_batch64", call="infer", T=512, B=64, I=1024, H=1024, dtype="f16", state=True),
        # inference of a layer whose weights do not fit on the chip
        dict(name="infer_wide4096", call="infer", T=64, B=32, I=1024, H=4096, dtype="f16", state=False),
        # a small model trained on fp32 tensors
        dict(name="train_small_f32", call="train", T=64, B=8, I=128, H=256, dtype="f32", state=False),
        # sizes that are a multiple of nothing, fp32 tensors
        dict(name="train_ragged_f32", call="train", T=200, B=70, I=65, H=257, dtype="f32", state=True),
        # between the two sizes the recurrence kernels were laid out for, a batch that is no power of two
        dict(name="train_mid1536", call="train", T=256, B=48, I=512, H=1536, dtype="f16", state=True),
        # the headline training step
        dict(name="train_batch256", call="train", T=1024, B=256, I=1024, H=1024, dtype="f16", state=True),
        # the latency-bound training step: few rows, many steps, wide
        dict(name="train_latency2048", call="train", T=2048, B=16, I=2048, H=2048, dtype="f16", state=False),
        # a two-layer module in an autograd training loop, parameters repacked every step as an optimizer changes them
        dict(name="module_2layers", call="module", T=100, B=20, I=256, H=650, L=2, dtype="f16", state=True),
        # a training step of the four-layer stack with a mean-squared-error loss (the benchmark's stack at a quarter
        # of its length, so that several fit the card)
        dict(name="stack_4layers", call="stack", T=1024, B=128, I=512, H=2048, L=4, dtype="f16", state=False),
        # sequences that live in pinned host memory, forward and backward (the streaming module's own test scale)
        dict(name="stream_host", call="stream", T=2048, B=32, I=1024, H=1024, dtype="f16", state=True, every=8),
        # the fp32 C API, forward, at the size of its own benchmark
        dict(name="capi_forward_f32", call="capi", T=2048, B=32, I=1024, H=1024, dtype="f32", state=True),
    ]


def _flops(case):
    T, B, I, H, L = case["T"], case["B"], case["I"], case["H"], case.get("L", 1)
    forward = sum(8.0 * T * B * H * ((I if l == 0 else H) + H) for l in range(L))
    if case["call"] in ("serve", "infer", "capi"):
        return forward
    whole = 3.0 * forward
    if case["call"] == "stack":   # the bottom layer's input gradient is not asked for
        whole -= 8.0 * T * B * H * I
    return whole


def _between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: sizes over the whole range (by their logarithm), half of them round numbers and half of them not."""
    call = rng.choice(["serve", "infer", "infer", "infer", "train", "train", "train", "train", "module", "stack", "stream", "capi"])
    T, B = _between(rng, 8, 2048), _between(rng, 1, 512)
    I, H = _between(rng, 16, 2048), _between(rng, 32, 4096)
    L = rng.randint(2, 4) if call in ("module", "stack") else 1
    if call == "serve":
        T, B = _between(rng, 1, 16), _between(rng, 1, 32)
    if rng.random() < 0.5:
        I, H = max(32, I // 32 * 32), max(32, H // 32 * 32)
        B = B if B < 8 else B // 8 * 8
    case = dict(call=call, T=T, B=B, I=I, H=H, dtype="f16", state=rng.random() < 0.5)
    if call == "capi" or (call in ("infer", "train") and rng.random() < 0.3):
        case["dtype"] = "f32"
    if L > 1:
        case["L"] = L
    if call == "stream":
        case["every"] = rng.choice([1, 8, 50])
        case["B"] = min(B, 128)
    # no dearer than the listed ones: a bound on the products and one on the steps of the recurrences
    most_steps = (2048 if H <= 2048 else 256) // L
    case["T"] = max(1, min(case["T"], most_steps))
    while _flops(case) > 2e13:
        case["T"] = max(1, case["T"] // 2)
        case["B"] = case["B"] if case["T"] > 8 else max(1, case["B"] // 2)
    return case


class _CApi:
    """A handle of the fp32 C API (include/flashlstm/lstm_api.h) with its weights packed."""

    class Buffers(ctypes.Structure):
        _fields_ = [("impl", ctypes.c_void_p)]

    ACC32, GRAPH = 0, 1

    def __init__(self, case, w_ih, w_hh):
        sz, vp, i32 = ctypes.c_size_t, ctypes.c_void_p, ctypes.c_int
        self.lib, self.buf = fl.load_library(), self.Buffers()
        handle = ctypes.POINTER(self.Buffers)
        self.lib.lstm_create_buffers.argtypes = [i32, sz, sz, sz, sz, i32, handle]
        self.lib.lstm_set_execution_mode.argtypes = [handle, i32]
        self.lib.lstm_pack_weights.argtypes = [i32, vp, vp, sz, sz, handle]
        self.lib.lstm_forward.argtypes = [vp] * 8 + [sz] * 4 + [handle, i32]
        self.lib.lstm_destroy_buffers.argtypes = [handle]
        self.sizes = (case["T"], case["B"], case["I"], case["H"])
        self.check(self.lib.lstm_create_buffers(self.ACC32, *self.sizes, 64, ctypes.byref(self.buf)))
        self.check(self.lib.lstm_set_execution_mode(ctypes.byref(self.buf), self.GRAPH))
        torch.cuda.current_stream().synchronize()   # the handle has a stream of its own
        self.check(self.lib.lstm_pack_weights(self.ACC32, w_ih.data_ptr(), w_hh.data_ptr(), case["I"], case["H"],
                                              ctypes.byref(self.buf)))

    @staticmethod
    def check(rc):
        if rc != 0:
            raise RuntimeError(f"the C API returned {rc}")

    def forward(self, x, b_ih, b_hh, h0, c0, y, hy, cy):
        ptr = lambda t: None if t is None else t.data_ptr()
        self.check(self.lib.lstm_forward(*[ptr(t) for t in (x, b_ih, b_hh, h0, c0, y, hy, cy)], *self.sizes,
                                         ctypes.byref(self.buf), self.ACC32))

    def __del__(self):
        self.lib.lstm_destroy_buffers(ctypes.byref(self.buf))


def prepare(case, seed):
    T, B, I, H, L, call = case["T"], case["B"], case["I"], case["H"], case.get("L", 1), case["call"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    dtype = torch.float32 if case["dtype"] == "f32" else torch.float16
    bound = 1.0 / math.sqrt(H)
    uniform = lambda *shape: (torch.rand(*shape, generator=g, device="cuda") * 2 - 1) * bound
    normal = lambda *shape: torch.randn(*shape, generator=g, device="cuda")
    weights = [(uniform(4 * H, I if l == 0 else H), uniform(4 * H, H), uniform(4 * H), uniform(4 * H)) for l in range(L)]
    s = dict(call=call, x=normal(T, B, I).to(dtype), h0=None, c0=None)
    state_shape = (L, B, H) if call in ("module", "stack") else (B, H)
    if case["state"]:
        s["h0"], s["c0"] = (normal(*state_shape) * 0.1).to(dtype), (normal(*state_shape) * 0.1).to(dtype)

    if call in ("serve", "infer", "train"):
        s["core"] = fl.LstmCore(B, I, H)
        s["core"].pack(*weights[0])
    if call in ("serve", "capi"):
        s["outputs"] = [torch.empty(*shape, device="cuda", dtype=dtype) for shape in ((T, B, H), (B, H), (B, H))]
    if call == "capi":
        s["core"], s["biases"] = _CApi(case, *weights[0][:2]), weights[0][2:]
    if call == "train":
        s["dy"] = normal(T, B, H).to(dtype)
    if call == "stack":
        s["core"], s["weights"] = fl.LstmStack(B, I, H, L), weights
        s["target"] = normal(T, B, H).to(dtype)
    if call == "module":
        s["core"] = fl.StackedLSTM(I, H, L)
        _set_parameters(s["core"], [t for layer in weights for t in layer])
        s["dy"] = normal(T, B, H).to(dtype)
        s["wanted"] = [s["x"].requires_grad_()] + list(s["core"].parameters())
    if call == "stream":
        fl.add_flashlstm_to_path()
        from flashlstm import StreamingLSTM
        s["core"], s["every"] = StreamingLSTM(I, H), case["every"]
        _set_parameters(s["core"], weights[0])
        s["x"] = _pinned(s["x"]).requires_grad_()
        s["dy"] = _pinned(normal(T, B, H).to(dtype))
        s["wanted"] = [s["x"]] + list(s["core"].parameters())
    return s


def _set_parameters(module, values):
    with torch.no_grad():
        for p, v in zip(module.parameters(), values):
            p.copy_(v)


def _pinned(t):
    host = torch.empty(t.shape, dtype=t.dtype, pin_memory=True)
    return host.copy_(t)


def run(s):
    call = s["call"]
    if call == "serve":
        s["core"].forward_static(s["x"], s["h0"], s["c0"], *s["outputs"])
        return s["outputs"]
    if call == "infer":
        return s["core"].forward(s["x"], s["h0"], s["c0"], save_for_backward=False)
    if call == "train":
        outputs = s["core"].forward(s["x"], s["h0"], s["c0"])
        return outputs, s["core"].backward(s["x"], s["dy"])
    if call == "stack":
        s["core"].pack(s["weights"])
        y, hys, cys = s["core"].forward(s["x"], s["h0"], s["c0"])
        _, grads, dh0s, dc0s = s["core"].backward_mse(y, s["target"], want_dx=False)
        return y, hys, cys, grads, dh0s, dc0s
    if call == "module":
        y, state = s["core"](s["x"], None if s["h0"] is None else (s["h0"], s["c0"]))
        return y.detach(), state[0].detach(), state[1].detach(), torch.autograd.grad(y, s["wanted"], s["dy"])
    if call == "stream":
        y, cache, state = s["core"](s["x"], s["h0"], s["c0"], recompute_interval=s["every"])
        return (y.detach(), cache.h, cache.c, state[0].detach(), state[1].detach(),
                torch.autograd.grad(y, s["wanted"], s["dy"]))
    if call == "capi":
        s["core"].forward(s["x"], *s["biases"], s["h0"], s["c0"], *s["outputs"])
        return s["outputs"]
    raise ValueError(f"unknown call {call!r}")


def work(case):
    """Bytes: the sequences, states and gradients that a caller hands over or gets, each once, and the weights once (fp16
    where the plan holds them packed, fp32 where the pass packs them or returns their gradients); no intermediate."""
    T, B, I, H, L, call = case["T"], case["B"], case["I"], case["H"], case.get("L", 1), case["call"]
    e = 4 if case["dtype"] == "f32" else 2
    n_weights = sum(4 * H * ((I if l == 0 else H) + H) for l in range(L))
    total = e * (T * B * (I + H) + 2 * L * B * H * (2 if case["state"] else 1)) + 16 * L * H
    total += n_weights * (2 if call in ("serve", "infer", "train", "capi") else 4)
    if call in ("train", "module", "stack", "stream"):
        total += e * T * B * H + 4 * (n_weights + 4 * L * H + 2 * L * B * H)
        total += e * T * B * I if call != "stack" else 0
    if call == "stream":
        total += 8 * -(-T // case["every"]) * B * H
    return {"bytes": float(total), "flops": _flops(case)}


def tolerance(case):
    """Activations, cached gates and gate gradients are rounded to fp16 (2^-11) between kernels and every sum is kept in
    fp32; through a whole sequence that leaves a few 1e-4 of relative error against fp32 arithmetic."""
    return {"rel": 2e-3}
