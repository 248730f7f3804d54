"""The work a user of the framework has it do, as measurable cases.

Every case goes through the public entry points of libpk_gpu.so (the ctypes
binding): single projections and feed-forward pairs on device pointers, the
host-pointer drop-in GEMM, attention, the convolution module's row
operations, the pre-encode and whole encoder passes.  Sizes are the 0.6 B
FastConformer's (d_model 1024, d_ff 4096, 8 heads of 128, 24 blocks), the
quantisation is the mixed model's: int4 feed-forward weights with one scale
per (row, 32 columns), int8 attention projections, fp32 pointwise
convolutions.

A case is a dict with "kind" and that kind's sizes:
  proj       one int8 projection of a short clip, default numerics, on a
             weight packed once at load time
  ffn        a feed-forward pair (up + bias + Swish, down + bias + half
             residual) on int4, int8 or fp32 weights; "fast" takes
             PK_GPU_NUMERICS_FAST with the workspace and weight copies a
             program that asks for that mode makes at load time
  dropin     the host-pointer int8 GEMM that replaces the reference's BLAS
             call: activations and result in host memory, weight registered
  attention  relative-position attention of one sequence
  rows       LayerNorm, GLU and depthwise convolution + Swish of one
             sequence
  pre        pre-encode: mel spectrogram to encoder input
  encoder    the 24 blocks over a chunked input, in one of the encoder's
             three numerics modes
"""
import ctypes
import importlib.util
import math
import os

import numpy as np
import torch

D, FF, HEADS, BLOCKS = 1024, 4096, 8, 24
CHUNK, OVERLAP = 400, 8          # output frames per chunk, context frames each side
PE_ROWS, PE_CENTER = 9999, 4999
MELS, SUB = 128, 256


def _binding():
    path = os.path.join(os.getcwd(), "parakeet-unified-en-0.6b-c_amd", "pk_gpu_ctypes.py")
    spec = importlib.util.spec_from_file_location("pk_gpu_ctypes", path)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


pk = _binding()
_ready = []


def _lib():
    if not _ready:
        pk.call("pk_gpu_init", 0)
        torch.cuda.set_device(0)
        _ready.append(pk.load())
    return _ready[0]


def _stream():
    return torch.cuda.current_stream().cuda_stream


def listed():
    return [
        # the fused QKV of a 2.5 s utterance: the smallest call, where launches and latency count
        {"name": "proj_clip", "kind": "proj", "m": 32, "n": 3072},
        # the feed-forward pair of 30 s of audio on the mixed model, bit-exact chains
        {"name": "ffn_i4_30s", "kind": "ffn", "bits": 4, "m": 375, "fast": False},
        # the same pair on the fp32 weight directory, 40 s of audio
        {"name": "ffn_f32_40s", "kind": "ffn", "bits": 32, "m": 500, "fast": False},
        # the pair over half of a 256 s batch for a program that accepts the 1e-3 contract
        {"name": "ffn_i4_batch_fast", "kind": "ffn", "bits": 4, "m": 1656, "fast": True},
        # the reference's own host code linked against the drop-in: one QKV call per 30 s
        {"name": "dropin_qkv_30s", "kind": "dropin", "m": 375, "n": 3072},
        # attention of one whole chunk (400 frames + 2 x 8 of context)
        {"name": "attention_chunk", "kind": "attention", "t": 416},
        # attention of 88 s with chunking off, an odd length
        {"name": "attention_unchunked", "kind": "attention", "t": 1101},
        # the row operations of the convolution module over 256 s unchunked
        {"name": "rows_256s", "kind": "rows", "t": 3200},
        # mel spectrogram of 256 s to encoder frames
        {"name": "pre_256s", "kind": "pre", "frames": 25600},
        # a 2.56 s clip through all blocks, short-utterance numerics
        {"name": "encoder_clip", "kind": "encoder", "t": 33, "mode": "default"},
        # 256 s of audio through all blocks, bit-exact: the headline workload
        {"name": "encoder_256s", "kind": "encoder", "t": 3200, "mode": "exact"},
        # the same under the 1e-3 contract
        {"name": "encoder_256s_fast", "kind": "encoder", "t": 3200, "mode": "fast"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("proj", "ffn", "ffn", "dropin", "attention", "attention", "rows", "pre", "encoder"))
    if kind == "proj":
        return {"kind": kind, "m": _log_int(rng, 1, 64), "n": rng.choice((1024, 3072))}
    if kind == "ffn":
        return {"kind": kind, "bits": rng.choice((4, 4, 8, 32)), "m": _log_int(rng, 65, 1656),
                "fast": rng.random() < 0.4}
    if kind == "dropin":
        return {"kind": kind, "m": _log_int(rng, 33, 500), "n": rng.choice((1024, 3072))}
    if kind == "attention":
        return {"kind": kind, "t": _log_int(rng, 24, 1200)}
    if kind == "rows":
        return {"kind": kind, "t": _log_int(rng, 33, 5000)}
    if kind == "pre":
        return {"kind": kind, "frames": _log_int(rng, 200, 25600)}
    mode = rng.choice(("default", "exact", "fast"))
    t = rng.randint(8, 64) if mode == "default" else _log_int(rng, 100, 3200)
    return {"kind": kind, "t": t, "mode": mode}


# ---- inputs ------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda:0")
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _normal(g, shape, sd=1.0, mean=0.0):
    return torch.randn(shape, generator=g, device="cuda:0") * sd + mean


class _W:
    """One weight matrix on the device in its on-disk format."""

    def __init__(self, g, bits, k, n, scale=0.01):
        self.bits, self.k, self.n, self.scale, self.scales = bits, k, n, scale, None
        if bits == 4:
            self.data = torch.randint(0, 256, (k, n // 2), generator=g, device="cuda:0", dtype=torch.uint8)
            self.scales = torch.rand((k, n // 32), generator=g, device="cuda:0") * 0.015 + 0.005
            self.ldb = n // 2
        elif bits == 8:
            self.data = torch.randint(-127, 128, (k, n), generator=g, device="cuda:0", dtype=torch.int8)
            self.ldb = n
        else:
            self.data = _normal(g, (k, n), 0.02)
            self.ldb = n

    def double(self):
        """The dequantised weight [k][n] in 64 bits."""
        if self.bits == 4:
            b = self.data.to(torch.int32)
            q = torch.stack((b & 15, b >> 4), dim=2).reshape(self.k, self.n)
            q = torch.where(q > 7, q - 16, q).double()
            return q * self.scales.double().repeat_interleave(32, dim=1)
        if self.bits == 8:
            return self.data.double() * float(np.float32(self.scale))
        return self.data.double()


def _gemm(lib, w, m, a, lda, c, ldc, bias, epi, s):
    if w.bits == 4:
        rc = lib.pk_gpu_gemm_i4_ex_dev(m, w.n, w.k, 1.0, a, lda, w.data.data_ptr(), w.scales.data_ptr(), w.ldb,
                                       0.0, c, ldc, bias, epi, s)
    elif w.bits == 8:
        rc = lib.pk_gpu_gemm_i8_ex_dev(m, w.n, w.k, 1.0, a, lda, w.data.data_ptr(), w.scale, w.ldb,
                                       0.0, c, ldc, bias, epi, s)
    else:
        rc = lib.pk_gpu_sgemm_ex_dev(m, w.n, w.k, 1.0, a, lda, w.data.data_ptr(), w.ldb, 0.0, c, ldc, bias, epi, s)
    if rc:
        pk.check("gemm", rc)


class _Proj:
    def __init__(self, case, seed):
        lib, g = _lib(), _gen(seed)
        self.m, self.n = case["m"], case["n"]
        self.x = _normal(g, (self.m, D))
        self.w = _W(g, 8, D, self.n)
        self.bias = _normal(g, (self.n,), 0.02)
        self.out = torch.empty((self.m, self.n), device="cuda:0")
        pk.check("pack", lib.pk_gpu_pack_weight_dev(8, D, self.n, self.w.data.data_ptr(), self.n, None, _stream()))

    def run(self):
        _gemm(_lib(), self.w, self.m, self.x.data_ptr(), D, self.out.data_ptr(), self.n, self.bias.data_ptr(),
              pk.EPI_NONE, _stream())
        return self.out

    def exact(self):
        return self.x.double() @ self.w.double() + self.bias.double()

    def __del__(self):
        if _ready and hasattr(self, "out"):
            _ready[0].pk_gpu_unpack_weight_dev(self.w.data.data_ptr())


class _Ffn:
    def __init__(self, case, seed):
        lib, g = _lib(), _gen(seed)
        self.m, self.fast = case["m"], case["fast"]
        bits = case["bits"]
        self.ln = _normal(g, (self.m, D))                    # the normalised input
        self.x = _normal(g, (self.m, D))                     # the residual stream
        self.up, self.down = _W(g, bits, D, FF, 0.002), _W(g, bits, FF, D, 0.002)
        self.b1, self.b2 = _normal(g, (FF,), 0.02), _normal(g, (D,), 0.02)
        self.h = torch.empty((self.m, FF), device="cuda:0")
        self.out = torch.empty((self.m, D), device="cuda:0")
        self.work = None
        if self.fast:
            self.work = torch.empty(pk.SPLIT_WORKSPACE_BYTES // 4, device="cuda:0")
            for w in (self.up, self.down):
                pk.check("presplit", lib.pk_gpu_presplit_weight_dev(
                    bits, w.k, w.n, w.data.data_ptr(), w.ldb,
                    w.scales.data_ptr() if bits == 4 else None, _stream()))

    def run(self):
        lib, s = _lib(), _stream()
        if self.fast:
            lib.pk_gpu_set_numerics(pk.NUMERICS_FAST)
            lib.pk_gpu_set_workspace(self.work.data_ptr(), pk.SPLIT_WORKSPACE_BYTES)
        self.out.copy_(self.x)                               # the residual, updated in place below
        _gemm(lib, self.up, self.m, self.ln.data_ptr(), D, self.h.data_ptr(), FF, self.b1.data_ptr(),
              pk.EPI_SWISH, s)
        _gemm(lib, self.down, self.m, self.h.data_ptr(), FF, self.out.data_ptr(), D, self.b2.data_ptr(),
              pk.EPI_HALF_RESIDUAL, s)
        if self.fast:
            lib.pk_gpu_set_workspace(None, 0)
            lib.pk_gpu_set_numerics(pk.NUMERICS_DEFAULT)
        return [self.h, self.out]

    def exact(self):
        h = self.ln.double() @ self.up.double() + self.b1.double()
        h = h * torch.sigmoid(h)
        return [h, self.x.double() + 0.5 * (h @ self.down.double() + self.b2.double())]

    def __del__(self):
        if _ready and getattr(self, "fast", False) and hasattr(self, "work"):
            for w in (self.up, self.down):
                _ready[0].pk_gpu_unsplit_weight_dev(w.data.data_ptr())


class _Dropin:
    def __init__(self, case, seed):
        lib, g = _lib(), _gen(seed)
        self.m, self.n = case["m"], case["n"]
        self.x = _normal(g, (self.m, D)).cpu().numpy()
        self.w = torch.randint(-127, 128, (D, self.n), generator=g, device="cuda:0", dtype=torch.int8).cpu().numpy()
        self.out = np.empty((self.m, self.n), np.float32)
        pk.check("register", lib.pk_gpu_register_weight(self.w.ctypes.data, self.w.nbytes))
        self.registered = True

    def run(self):
        pk.check("pk_gpu_gemm_i8", _lib().pk_gpu_gemm_i8(
            self.m, self.n, D, 1.0, self.x.ctypes.data, D, self.w.ctypes.data, 0.01, self.n, 0.0,
            self.out.ctypes.data, self.n))
        return self.out

    def exact(self):
        x, w = torch.from_numpy(self.x).cuda().double(), torch.from_numpy(self.w).cuda().double()
        return x @ (w * float(np.float32(0.01)))

    def __del__(self):
        if _ready and getattr(self, "registered", False):
            _ready[0].pk_gpu_unregister_weight(self.w.ctypes.data)


def _attend(qkv, p, pu, pv, t):
    """Relative-position attention of one sequence in the inputs' precision:
    qkv [t][3D], p [2t-1][D] (row m is relative position t-1-m)."""
    q, k, v = (qkv[:, i * D:(i + 1) * D].reshape(t, HEADS, 128).transpose(0, 1).contiguous() for i in range(3))
    ph = p.reshape(2 * t - 1, HEADS, 128).transpose(0, 1).contiguous()
    u, w = pu.reshape(HEADS, 1, 128), pv.reshape(HEADS, 1, 128)
    ac = torch.matmul(q + u, k.transpose(1, 2).contiguous())
    bd = torch.matmul(q + w, ph.transpose(1, 2).contiguous())
    idx = t - 1 - torch.arange(t, device=p.device)[:, None] + torch.arange(t, device=p.device)[None, :]
    bd = torch.gather(bd, 2, idx.expand(HEADS, t, t))
    a = torch.softmax((ac + bd) / math.sqrt(128.0), dim=2)
    return torch.matmul(a, v).transpose(0, 1).reshape(t, D)


class _Attention:
    def __init__(self, case, seed):
        lib, g = _lib(), _gen(seed)
        t = self.t = case["t"]
        self.qkv, self.p = _normal(g, (t, 3 * D)), _normal(g, (2 * t - 1, D))
        self.pu, self.pv = _normal(g, (D,), 0.1), _normal(g, (D,), 0.1)
        self.out = torch.empty((t, D), device="cuda:0")
        self.ws_floats = lib.pk_gpu_attention_ws_floats(t, HEADS)
        self.ws = torch.empty(max(4, self.ws_floats), device="cuda:0")

    def run(self):
        rc = _lib().pk_gpu_attention_ws_dev(self.qkv.data_ptr(), 3 * D, self.p.data_ptr(), D, self.pu.data_ptr(),
                                            self.pv.data_ptr(), self.out.data_ptr(), D, self.t, HEADS,
                                            self.ws.data_ptr(), self.ws_floats, _stream())
        if rc:
            pk.check("pk_gpu_attention_ws_dev", rc)
        return self.out

    def exact(self):
        return _attend(self.qkv.double(), self.p.double(), self.pu.double(), self.pv.double(), self.t)


def _depthwise(x, w, b):
    """x [t][D] over time with zero padding, w [D][9], then Swish."""
    y = torch.nn.functional.conv1d(x.t()[None], w.reshape(D, 1, 9), b, padding=4, groups=D)[0].t()
    return y * torch.sigmoid(y)


class _Rows:
    def __init__(self, case, seed):
        g = _gen(seed)
        _lib()
        t = self.t = case["t"]
        self.x, self.h = _normal(g, (t, D), 2.0, 0.3), _normal(g, (t, 2 * D))
        self.gamma, self.beta = _normal(g, (D,), 0.1, 1.0), _normal(g, (D,), 0.1)
        self.dw, self.db = _normal(g, (D, 9), 1.0 / 3.0), _normal(g, (D,), 0.02)
        self.ln, self.glu, self.out = (torch.empty((t, D), device="cuda:0") for _ in range(3))

    def run(self):
        lib, s, t = _lib(), _stream(), self.t
        rc = lib.pk_gpu_layer_norm_dev(self.x.data_ptr(), self.gamma.data_ptr(), self.beta.data_ptr(),
                                       self.ln.data_ptr(), t, D, s)
        rc = rc or lib.pk_gpu_glu_dev(self.h.data_ptr(), self.glu.data_ptr(), t, D, s)
        rc = rc or lib.pk_gpu_depthwise_dev(self.glu.data_ptr(), D, self.dw.data_ptr(), self.db.data_ptr(),
                                            self.out.data_ptr(), D, t, D, 9, 1, s)
        if rc:
            pk.check("rows", rc)
        return [self.ln, self.glu, self.out]

    def exact(self):
        ln = torch.nn.functional.layer_norm(self.x.double(), (D,), self.gamma.double(), self.beta.double(), 1e-5)
        h = self.h.double()
        glu = h[:, :D] * torch.sigmoid(h[:, D:])
        return [ln, glu, _depthwise(glu, self.dw.double(), self.db.double())]


# ---- the encoder -------------------------------------------------------------

_pe = []


def _pe_table():
    """Sinusoidal relative positions, row p = position PE_CENTER - p."""
    if not _pe:
        pos = (PE_CENTER - np.arange(PE_ROWS, dtype=np.float64))[:, None]
        div = np.exp(-(2.0 * np.arange(D // 2)) * np.log(10000.0) / D)[None, :]
        t = np.empty((PE_ROWS, D), np.float32)
        t[:, 0::2], t[:, 1::2] = np.sin(pos * div), np.cos(pos * div)
        _pe.append(t)
    return _pe[0]


class _Model:
    """Random parameters of `blocks` conformer blocks, on the host as a loaded
    model is; the attention projections' scales as a trained model's."""

    def __init__(self, g, blocks):
        self.keep, self.blocks, self.parts = [], (pk.BlockWeights * max(1, blocks))(), []
        for b in range(blocks):
            w, part = self.blocks[b], {}

            def put(field, t):
                part[field] = t.cpu().numpy()
                setattr(w, field, part[field].ctypes.data)

            def weight(field, x):
                part[field] = x
                x.data = x.data.cpu().numpy()
                x.scales = None if x.scales is None else x.scales.cpu().numpy()
                setattr(w, field, pk.Weight(x.data.ctypes.data, x.scale if x.bits == 8 else 0.0,
                                            None if x.scales is None else x.scales.ctypes.data, x.bits))

            for n in ("ff1", "sa", "conv", "ff2", "out"):
                put("norm_%s_w" % n, _normal(g, (D,), 0.02, 1.0))
                put("norm_%s_b" % n, _normal(g, (D,), 0.02))
            for n in ("ff1", "ff2"):
                weight(n + "_linear1_w", _W(g, 4, D, FF))
                put(n + "_linear1_b", _normal(g, (FF,), 0.02))
                weight(n + "_linear2_w", _W(g, 4, FF, D))
                put(n + "_linear2_b", _normal(g, (D,), 0.02))
            weight("linear_qkv_w", _W(g, 8, D, 3 * D, 0.00055))
            put("linear_qkv_b", _normal(g, (3 * D,), 0.02))
            weight("linear_pos_w", _W(g, 8, D, D, 0.0005))
            weight("linear_out_w", _W(g, 8, D, D, 0.0005))
            put("linear_out_b", _normal(g, (D,), 0.02))
            put("pos_bias_u", _normal(g, (D,), 0.02))
            put("pos_bias_v", _normal(g, (D,), 0.02))
            put("conv_pw1_w", _normal(g, (2 * D, D), 0.02))
            put("conv_pw1_b", _normal(g, (2 * D,), 0.02))
            put("conv_dw_w", _normal(g, (D, 9), 1.0 / 3.0))
            put("conv_dw_b", _normal(g, (D,), 0.02))
            put("conv_pw2_w", _normal(g, (D, D), 0.02))
            put("conv_pw2_b", _normal(g, (D,), 0.02))
            self.parts.append(part)


def _chunks(t):
    """Input rows [i0, i1) and output rows [o0, o1) of every chunk."""
    out = []
    for o0 in range(0, t, CHUNK):
        o1 = min(o0 + CHUNK, t)
        out.append((max(o0 - OVERLAP, 0), min(o1 + OVERLAP, t), o0, o1))
    return out


class _Encoder:
    def __init__(self, case, seed):
        lib, g = _lib(), _gen(seed)
        self.t = case["t"]
        self.x = _normal(g, (self.t, D))
        self.out = torch.empty_like(self.x)
        self.model = _Model(g, BLOCKS)
        self.h = ctypes.c_void_p()
        pe = _pe_table()
        pk.check("pk_gpu_encoder_create", lib.pk_gpu_encoder_create(
            ctypes.byref(self.h), ctypes.cast(self.model.blocks, ctypes.c_void_p), BLOCKS, pe.ctypes.data, PE_ROWS,
            PE_CENTER))
        mode = {"default": pk.NUMERICS_DEFAULT, "exact": pk.NUMERICS_EXACT, "fast": pk.NUMERICS_FAST}[case["mode"]]
        pk.check("pk_gpu_encoder_set_numerics", lib.pk_gpu_encoder_set_numerics(self.h, mode))

    def run(self):
        rc = _lib().pk_gpu_encoder_run_dev(self.h, self.x.data_ptr(), self.t, CHUNK, OVERLAP, self.out.data_ptr(),
                                           _stream())
        if rc:
            pk.check("pk_gpu_encoder_run_dev", rc)
        return self.out

    def exact(self):
        dev = lambda a: torch.from_numpy(a).cuda().double()  # noqa: E731
        pe = _pe_table()
        chunks = _chunks(self.t)
        xs = torch.cat([self.x[i0:i1] for i0, i1, _, _ in chunks]).double()
        for part in self.model.parts:
            def weight(name):
                w = part[name]
                d = _W.__new__(_W)
                d.bits, d.k, d.n, d.scale = w.bits, w.k, w.n, w.scale
                d.data = torch.from_numpy(w.data).cuda()
                d.scales = None if w.scales is None else torch.from_numpy(w.scales).cuda()
                return d.double()

            def norm(x, n):
                return torch.nn.functional.layer_norm(x, (D,), dev(part["norm_%s_w" % n]), dev(part["norm_%s_b" % n]),
                                                      1e-5)

            def ffn(x, n):
                h = norm(x, n) @ weight(n + "_linear1_w") + dev(part[n + "_linear1_b"])
                h = h * torch.sigmoid(h)
                return x + 0.5 * (h @ weight(n + "_linear2_w") + dev(part[n + "_linear2_b"]))

            xs = ffn(xs, "ff1")
            qkv = norm(xs, "sa") @ weight("linear_qkv_w") + dev(part["linear_qkv_b"])
            pos, pu, pv = weight("linear_pos_w"), dev(part["pos_bias_u"]), dev(part["pos_bias_v"])
            att, r = [], 0
            for i0, i1, _, _ in chunks:
                n = i1 - i0
                att.append(_attend(qkv[r:r + n], dev(pe[PE_CENTER - n + 1:PE_CENTER + n]) @ pos, pu, pv, n))
                r += n
            xs = xs + torch.cat(att) @ weight("linear_out_w") + dev(part["linear_out_b"])
            h = norm(xs, "conv") @ dev(part["conv_pw1_w"]).t() + dev(part["conv_pw1_b"])
            h = h[:, :D] * torch.sigmoid(h[:, D:])
            conv, r = [], 0
            for i0, i1, _, _ in chunks:
                n = i1 - i0
                conv.append(_depthwise(h[r:r + n], dev(part["conv_dw_w"]), dev(part["conv_dw_b"])))
                r += n
            xs = xs + torch.cat(conv) @ dev(part["conv_pw2_w"]).t() + dev(part["conv_pw2_b"])
            xs = norm(ffn(xs, "ff2"), "out")
        out, r = [], 0
        for i0, i1, o0, o1 in chunks:
            out.append(xs[r + o0 - i0:r + o1 - i0])
            r += i1 - i0
        return torch.cat(out)

    def __del__(self):
        if _ready and getattr(self, "h", None):
            torch.cuda.synchronize()
            _ready[0].pk_gpu_encoder_destroy(self.h)


class _Pre:
    """An encoder handle without blocks' work: the pre-encode alone (one block
    uploaded, as the handle needs at least one)."""

    def __init__(self, case, seed):
        lib, g = _lib(), _gen(seed)
        self.frames = case["frames"]
        self.mel = _normal(g, (MELS, self.frames), 2.0)
        self.model = _Model(g, 1)
        self.h = ctypes.c_void_p()
        pe = _pe_table()
        pk.check("pk_gpu_encoder_create", lib.pk_gpu_encoder_create(
            ctypes.byref(self.h), ctypes.cast(self.model.blocks, ctypes.c_void_p), 1, pe.ctypes.data, PE_ROWS,
            PE_CENTER))
        self.p, w = {}, pk.PreEncodeWeights()
        for name, shape, sd in (("conv0", (SUB, 9), 0.3), ("conv2", (SUB, 9), 0.3), ("conv3", (SUB, SUB), 1.0 / 16),
                                ("conv5", (SUB, 9), 0.3), ("conv6", (SUB, SUB), 1.0 / 16)):
            self.p[name + "_w"] = _normal(g, shape, sd).cpu().numpy()
            self.p[name + "_b"] = _normal(g, (SUB,), 0.02).cpu().numpy()
        self.out_w = torch.randint(-127, 128, (FF, D), generator=g, device="cuda:0", dtype=torch.int8).cpu().numpy()
        self.p["out_b"] = _normal(g, (D,), 0.02).cpu().numpy()
        for k, v in self.p.items():
            setattr(w, k, v.ctypes.data)
        self.scale = 0.01 / 64
        w.out_w = pk.Weight(self.out_w.ctypes.data, self.scale, None, 8)
        pk.check("pk_gpu_encoder_set_pre_encode", lib.pk_gpu_encoder_set_pre_encode(self.h, ctypes.byref(w)))
        self.tp = lib.pk_gpu_encoder_frames(self.frames)
        self.out = torch.empty((self.tp, D), device="cuda:0")

    def run(self):
        rc = _lib().pk_gpu_encoder_pre_encode_dev(self.h, self.mel.data_ptr(), self.frames, self.out.data_ptr(),
                                                  _stream())
        if rc:
            pk.check("pk_gpu_encoder_pre_encode_dev", rc)
        return self.out

    def exact(self):
        def conv(x, name, groups):                     # [H][W][C] in and out, by taps: plain sums in 64 bits
            w = torch.from_numpy(self.p[name + "_w"]).cuda().double()
            h, wd = (x.shape[0] - 1) // 2 + 1, (x.shape[1] - 1) // 2 + 1
            x = torch.nn.functional.pad(x, (0, 0, 1, 2, 1, 2))
            y = torch.from_numpy(self.p[name + "_b"]).cuda().double().expand(h, wd, SUB).clone()
            for k in range(9):
                y += x[k // 3:k // 3 + 2 * h:2, k % 3:k % 3 + 2 * wd:2] * w[:, k]
            return y

        def pointwise(x, name):
            w, b = (torch.from_numpy(self.p[name + s]).cuda().double() for s in ("_w", "_b"))
            return torch.relu(x.reshape(-1, SUB) @ w.t() + b).reshape(x.shape)

        out, step = [], 400                            # output frames at a time, from the mel rows they need
        mel = self.mel.t().double()
        for f0 in range(0, self.tp, step):
            f1 = min(f0 + step, self.tp)
            a = max(0, f0 - 2)                         # two frames of context, dropped below
            x = mel[8 * a:min(8 * f1 + 16, self.frames), :, None]
            x = torch.relu(conv(x, "conv0", 1))
            x = pointwise(conv(x, "conv2", SUB), "conv3")
            x = pointwise(conv(x, "conv5", SUB), "conv6")
            out.append(x[f0 - a:f1 - a].permute(0, 2, 1).reshape(f1 - f0, FF))
        w = torch.from_numpy(self.out_w).cuda().double() * float(np.float32(self.scale))
        return (torch.cat(out) @ w + torch.from_numpy(self.p["out_b"]).cuda().double()) * 32.0

    def __del__(self):
        if _ready and getattr(self, "h", None):
            torch.cuda.synchronize()
            _ready[0].pk_gpu_encoder_destroy(self.h)


_KINDS = {"proj": _Proj, "ffn": _Ffn, "dropin": _Dropin, "attention": _Attention, "rows": _Rows, "pre": _Pre,
          "encoder": _Encoder}


def prepare(case, seed):
    return _KINDS[case["kind"]](case, seed)


def run(state):
    return state.run()


def exact(case, seed):
    return prepare(case, seed).exact()


# ---- what a pass cannot do without --------------------------------------------

def _weight_bytes(bits, k, n):
    return {4: k * n // 2 + 4 * k * (n // 32), 8: k * n, 32: 4 * k * n}[bits]


def _attention_flops(t):
    return 6.0 * t * t * D                 # content scores, shifted position scores, scores x V


def work(case):
    kind = case["kind"]
    if kind == "proj":
        m, n = case["m"], case["n"]
        return {"bytes": D * n + 4 * (m * D + m * n + n), "flops": 2.0 * m * n * D}
    if kind == "ffn":
        m, b = case["m"], case["bits"]
        return {"bytes": _weight_bytes(b, D, FF) + _weight_bytes(b, FF, D) + 4 * (3 * m * D + m * FF + FF + D),
                "flops": 4.0 * m * D * FF}
    if kind == "dropin":
        m, n = case["m"], case["n"]
        return {"bytes": D * n + 4 * (m * D + m * n), "flops": 2.0 * m * n * D}
    if kind == "attention":
        t = case["t"]
        return {"bytes": 4 * (4 * t * D + (2 * t - 1) * D), "flops": _attention_flops(t)}
    if kind == "rows":
        t = case["t"]
        return {"bytes": 4 * t * D * (2 + 3 + 1), "flops": t * D * (8.0 + 4.0 + 20.0)}
    if kind == "pre":
        n = case["frames"]
        h = [n]
        for _ in range(3):
            h.append((h[-1] - 1) // 2 + 1)
        conv = 18.0 * SUB * (h[1] * 64 + h[2] * 32 + h[3] * 16)
        point = 2.0 * SUB * SUB * (h[2] * 32 + h[3] * 16)
        return {"bytes": 4 * (MELS * n + 3 * 9 * SUB + 2 * SUB * SUB + h[3] * D) + FF * D,
                "flops": conv + point + 2.0 * h[3] * FF * D}
    t = case["t"]
    rows = sum(i1 - i0 for i0, i1, _, _ in _chunks(t))
    gemm = 2.0 * rows * D * (4 * FF + 3 * D + D + 2 * D + D)
    att = sum(_attention_flops(i1 - i0) for i0, i1, _, _ in _chunks(t))
    weights = 2 * (_weight_bytes(4, D, FF) + _weight_bytes(4, FF, D)) + 4 * D * D + 4 * 3 * D * D
    longest = max(i1 - i0 for i0, i1, _, _ in _chunks(t))
    return {"bytes": BLOCKS * (weights + 4 * (2 * longest - 1) * D) + 8 * t * D, "flops": BLOCKS * (gemm + att)}


def tolerance(case):
    """Everything outside the tolerance modes is promised bit for bit.  The
    others: about four times their distance from the exact sums."""
    kind = case["kind"]
    if kind == "proj" or (kind == "dropin" and case["m"] <= 64):   # short clips: the small-M kernels
        return {"rel": 1e-5, "max": 1e-4}
    if kind == "ffn" and case["fast"]:
        return {"rel": 2e-5, "max": 2e-4}
    if kind == "encoder" and case["mode"] != "exact":
        return {"rel": 1.3e-4 if case["mode"] == "fast" else 6e-5, "max": 1e-3}
    return "exact"
