"""Performance cases: the work this library is used for, through its public
entry points, on synthetic data.

Six families, each over the range of sizes its users have:
  slws         pooled lookups in fused-rowwise tables (mi355x_frwq_slws)
  fc           RowwiseQuantizedFullyConnected (mi355x_rwq_fc_i8)
  conv         ChannelwiseQuantizedConvolution, plain or with the residual add
               behind it (mi355x_cwq_conv2d_i8 / _add_i8)
  elementwise  Quantize, RescaleQuantized, ElementAdd, Dequantize
  resnet50     requests to a resident int8 ResNet-50 (DeviceManager.run)
  dlrm         requests to a resident ranking net (DeviceManager.run)

The first four call the kernel library on device memory, the way a backend
with buffers of its own does; the last two take host arrays in and out, the way
a server drives a device manager: the network is loaded once and kept, a
request brings new inputs.
"""
import functools
import math

import numpy as np
import torch

from glow_amd import capi
from glow_amd import host as H
from glow_amd import workloads
from glow_amd.harness import dlrm
from glow_amd.harness import net as netlib
from glow_amd.harness import resnet50

TABLES = 26           # lookup tables of the ranking net
BOTTOM = (512, 256, 64)
TOP = (512, 256, 1)
DENSE = 13
MAX_FC_MACS = 8192 * 4096 * 4096
MAX_CONV_MACS = 16 * 10 ** 9
MAX_LOOKUPS = 2_600_000


def listed():
    return [
        # One request's pooled lookup: a handful of bags from a 4-bit table, where
        # the call itself is most of the time.
        dict(name="slws_request", op="slws", rows=100_000, cols=64, kind=capi.FUSED_U4_F16,
             bags=32, mean_len=20, idx64=False, weighted=False),
        # The pooled lookup of bench.py's headline: 4M x 128 bytes, 4096 bags.
        dict(name="slws_batch", op="slws", rows=4_000_000, cols=128, kind=capi.FUSED_U8_F32,
             bags=4096, mean_len=40, idx64=True, weighted=True),
        # A large offline batch over rows of a width no power of two divides.
        dict(name="slws_bulk_cols100", op="slws", rows=1_000_000, cols=100,
             kind=capi.FUSED_U8_F32, bags=30_000, mean_len=30, idx64=True, weighted=True),
        # The single FullyConnected configuration.
        dict(name="fc_single", op="fc", M=128, K=1024, N=1024, symmetric=True, bias_i8=False),
        # A small ragged layer with asymmetric weights and an int8 bias.
        dict(name="fc_ragged", op="fc", M=61, K=415, N=509, symmetric=False, bias_i8=True),
        # A layer large enough to be bound by the matrix cores.
        dict(name="fc_large", op="fc", M=8192, K=4096, N=4096, symmetric=True, bias_i8=False),
        # The 3x3 convolution over 64 channels of an image network's first stage.
        dict(name="conv_3x3_64", op="conv", N=32, H=56, W=56, IC=64, OC=64, k=3, stride=1, group=1,
             symmetric=True, residual=False),
        # Odd image sizes, channel counts no tile divides, stride 2, residual add.
        dict(name="conv_ragged_add", op="conv", N=5, H=61, W=45, IC=96, OC=200, k=3, stride=2,
             group=1, symmetric=True, residual=True),
        # The elementwise instructions around a block, on bench.py's tensor.
        dict(name="elementwise", op="elementwise", n=4 * 64 * 56 * 56 * 64),
        # An image network answering one image (ordinary host arrays) ...
        dict(name="resnet50_one", op="resnet50", batch=1, size=224, pinned=False),
        # ... and a batch of 64 from the I/O buffers the device manager hands out.
        dict(name="resnet50_batch", op="resnet50", batch=64, size=224, pinned=True),
        # The ranking net at its benchmark batch: 26 tables of 1M x 64.
        dict(name="dlrm_batch", op="dlrm", batch=4096, rows=1_000_000, pinned=True),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["slws", "slws", "fc", "fc", "conv", "conv", "elementwise", "resnet50", "dlrm"])
    if op == "slws":
        bags, mean_len = _log(rng, 1, 65536), _log(rng, 2, 150)
        mean_len = max(1, min(mean_len, MAX_LOOKUPS // bags))
        return dict(op=op, rows=_log(rng, 1000, 4_000_000),
                    cols=rng.choice([16, 32, 48, 64, 64, 96, 100, 128, 128, 200, 256]),
                    kind=rng.choice([capi.FUSED_U8_F32, capi.FUSED_U8_F32, capi.FUSED_U8_F16,
                                     capi.FUSED_U4_F16, capi.FUSED_U4_F32]),
                    bags=bags, mean_len=mean_len, idx64=rng.random() < 0.5,
                    weighted=rng.random() < 0.5)
    if op == "fc":
        M, K, N = _log(rng, 1, 16384), _log(rng, 13, 4608), _log(rng, 1, 4096)
        if rng.random() < 0.5:     # layer widths are multiples of 64 as often as not
            K, N = max(64, K // 64 * 64), max(64, N // 64 * 64)
        return dict(op=op, M=max(1, min(M, MAX_FC_MACS // (K * N))), K=K, N=N,
                    symmetric=rng.random() < 0.7, bias_i8=rng.random() < 0.3)
    if op == "conv":
        h = _log(rng, 7, 112)
        w = max(7, min(112, h + rng.choice([0, 0, -3, 5])))
        ic = rng.choice([16, 24, 32, 64, 64, 96, 128, 128, 256, 512])
        oc = rng.choice([16, 40, 64, 64, 100, 128, 200, 256, 512])
        k, stride = rng.choice([1, 1, 3, 3, 5]), rng.choice([1, 1, 2])
        group = rng.choice([1, 1, 1, 2]) if oc % 2 == 0 else 1
        per = ((h + stride - 1) // stride) * ((w + stride - 1) // stride) * oc * k * k * (ic // group)
        return dict(op=op, N=max(1, min(_log(rng, 1, 64), MAX_CONV_MACS // per)), H=h, W=w, IC=ic,
                    OC=oc, k=k, stride=stride, group=group, symmetric=rng.random() < 0.8,
                    residual=rng.random() < 0.3)
    if op == "elementwise":
        return dict(op=op, n=_log(rng, 1000, 4 * 64 * 56 * 56 * 64))
    if op == "resnet50":
        return dict(op=op, batch=_log(rng, 1, 64), size=rng.choice([160, 192, 224]),
                    pinned=rng.random() < 0.5)
    return dict(op=op, batch=_log(rng, 16, 4096), rows=_log(rng, 10_000, 1_000_000),
                pinned=rng.random() < 0.5)


# ---- inputs --------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _ints(g, lo, hi, shape, dtype):
    return torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=dtype)


def _i32(v):
    return torch.as_tensor(np.ascontiguousarray(v, np.int32)).cuda()


def _uniform(g, lo, hi, shape):
    return torch.rand(shape, generator=g, device="cuda") * (hi - lo) + lo


def _prepare_slws(c, seed):
    """A table of random codes with plausible per-row scales and offsets,
    Poisson bag lengths, Zipf(1.05) indices scattered over the table."""
    g = _gen(seed)
    rows, cols, kind, bags = c["rows"], c["cols"], c["kind"], c["bags"]
    four = kind in (capi.FUSED_U4_F16, capi.FUSED_U4_F32)
    half = kind in (capi.FUSED_U8_F16, capi.FUSED_U4_F16)
    row_bytes = capi.fused_row_bytes(cols, kind)
    table = _ints(g, 0, 256, (rows, row_bytes), torch.uint8)
    so = torch.stack([_uniform(g, 4.0, 8.0, rows) / (15.0 if four else 255.0),
                      torch.randn(rows, generator=g, device="cuda") * 0.5 - 3.0], dim=1)
    table[:, cols // 2 if four else cols:] = so.to(torch.float16 if half else torch.float32).view(torch.uint8)
    lengths = torch.poisson(torch.full((bags,), float(c["mean_len"]), device="cuda"), generator=g)
    lengths = lengths.to(torch.int32)
    total = int(lengths.sum())
    u = torch.rand(max(total, 1), generator=g, device="cuda", dtype=torch.float64)
    a = 1.0 - 1.05
    rank = (u * ((rows + 1.0) ** a - 1.0) + 1.0) ** (1.0 / a)
    rank = (rank.floor().to(torch.int64) - 1).clamp(0, rows - 1)
    idx = (rank * 2654435761 + 12345) % rows
    return dict(c, table=table, lengths=lengths, total=total, row_bytes=row_bytes, half=half,
                idx=idx if c["idx64"] else idx.to(torch.int32),
                w=torch.rand(max(total, 1), generator=g, device="cuda") if c["weighted"] else None,
                out=torch.empty((bags, cols), device="cuda",
                                dtype=torch.float16 if half else torch.float32))


def _run_slws(s):
    # tables with fp16 scales pool into fp16 results, as Glow types them
    w = s["w"]
    capi.launch_frwq_slws(s["out"].data_ptr(), s["half"], s["table"].data_ptr(), s["rows"], s["kind"],
                          None if w is None else w.data_ptr(), False, s["idx"].data_ptr(),
                          s["idx64"], s["total"], s["lengths"].data_ptr(), s["bags"],
                          s["row_bytes"], s["cols"])
    return s["out"]


def _requant(g, n, fan_in, in_scale, w_range, spread, bias_i8):
    """Per-channel weight scales and the integer parameters the code generator
    derives from them; the output scale keeps most results inside int8."""
    ws = _uniform(g, *w_range, n).cpu().numpy().astype(np.float32)
    mm = np.float32(in_scale) * ws
    out_scale = math.sqrt(fan_in) * spread * in_scale * float(ws.mean()) / 40
    bpre, bpost, bscale = workloads.s32to8_vec(np.full(n, 37.0 if bias_i8 else 1.0, np.float32))
    opre, opost, oscale = workloads.s32to8_vec(mm / np.float32(out_scale))
    return [_i32(v) for v in (bpre, bpost, bscale, opre, opost, oscale)]


def _bias(g, n, bias_i8):
    return _ints(g, -128, 128, (n,), torch.int8) if bias_i8 else _ints(g, -20000, 20001, (n,), torch.int32)


def _prepare_fc(c, seed):
    g = _gen(seed)
    M, K, N = c["M"], c["K"], c["N"]
    x = (torch.randn((M, K), generator=g, device="cuda") * 40).round().clamp(-128, 127).to(torch.int8)
    w = _ints(g, -127, 128, (N, K), torch.int8)
    offs = torch.zeros(N, dtype=torch.int32, device="cuda") if c["symmetric"] else \
        _ints(g, -20, 21, (N,), torch.int32)
    sums = torch.empty(N, dtype=torch.int32, device="cuda")
    capi.launch_rowsum_i8(sums.data_ptr(), w.data_ptr(), N, K)     # constants: once per network
    return dict(c, x=x, w=w, bias=_bias(g, N, c["bias_i8"]), offs=offs, sums=sums,
                params=_requant(g, N, K, 0.05, (0.001, 0.02), 40 * 73, c["bias_i8"]),
                in_offset=seed % 21 - 10, out=torch.empty((M, N), dtype=torch.int8, device="cuda"))


def _run_fc(s):
    capi.launch_rwq_fc_i8(s["out"].data_ptr(), s["x"].data_ptr(), s["w"].data_ptr(),
                          s["bias"].data_ptr(), s["bias_i8"], s["offs"].data_ptr(),
                          *[p.data_ptr() for p in s["params"]], s["M"], s["K"], s["N"], 3,
                          s["in_offset"], 0, w_offsets_all_zero=s["symmetric"],
                          w_row_sums=s["sums"].data_ptr())
    return s["out"]


def _conv_geom(c):
    p = c["k"] // 2
    return workloads.default_host().conv_geom(c["N"], c["H"], c["W"], c["IC"], c["OC"],
                                              (c["k"], c["k"]), (c["stride"], c["stride"]),
                                              (p, p, p, p), c["group"])


def _prepare_conv(c, seed):
    g = _gen(seed)
    geom, oc = _conv_geom(c), c["OC"]
    per = c["k"] * c["k"] * (c["IC"] // c["group"])
    x = _ints(g, -128, 128, (c["N"], c["H"], c["W"], c["IC"]), torch.int8)
    filt = _ints(g, -127, 128, (oc, per), torch.int8)
    zeros = torch.zeros(oc, dtype=torch.int32, device="cuda")
    sums = torch.empty(oc, dtype=torch.int32, device="cuda")
    capi.launch_rowsum_i8(sums.data_ptr(), filt.data_ptr(), oc, per)
    out = torch.empty((c["N"], geom.OH, geom.OW, oc), dtype=torch.int8, device="cuda")
    s32 = capi.quantize_scale_offset_32to8
    return dict(c, geom=geom, x=x, filt=filt, bias=_bias(g, oc, False), b_offs=zeros, sums=sums,
                f_offs=zeros if c["symmetric"] else _ints(g, -10, 11, (oc,), torch.int32),
                params=_requant(g, oc, per, 0.05, (0.002, 0.02), 74 * 74, False), out=out,
                res=_ints(g, -128, 128, tuple(out.shape), torch.int8) if c["residual"] else None,
                add=capi.fused_add(-5, 4, s32(0.8)[:3], s32(0.6)[:3], True, -128, s32(1.1)[:3]))


def _run_conv(s):
    args = (s["out"].data_ptr(), s["x"].data_ptr(), s["filt"].data_ptr(), s["bias"].data_ptr(), False,
            s["geom"], -3, -128, s["f_offs"].data_ptr(), s["b_offs"].data_ptr(),
            *[p.data_ptr() for p in s["params"]])
    if s["residual"]:
        capi.launch_cwq_conv2d_add_i8(*args, capi.ACT_NONE, (), s["symmetric"], s["sums"].data_ptr(),
                                      s["res"].data_ptr(), s["add"])
    else:
        capi.launch_cwq_conv2d_i8(*args, capi.ACT_RELU, (), s["symmetric"], s["sums"].data_ptr())
    return s["out"]


def _prepare_elementwise(c, seed):
    g, n = _gen(seed), c["n"]
    def i8():
        return torch.empty(n, dtype=torch.int8, device="cuda")
    s32 = capi.quantize_scale_offset_32to8
    return dict(c, x=torch.randn(n, generator=g, device="cuda"), q=i8(), r=i8(), t=i8(),
                f=torch.empty(n, device="cuda"), to_r=s32(0.02 / 0.028)[:3],
                add=(s32(0.02 / 0.04)[:3], s32(0.028 / 0.04)[:3]))


def _run_elementwise(s):
    n = s["n"]
    x, q, r, t, f = (s[k].data_ptr() for k in "xqrtf")
    capi.launch_quantize_i8(q, x, n, 0.02, -3)
    capi.launch_rescale_i8(r, q, n, 3, -3, *s["to_r"])
    capi.launch_add_i8(t, q, r, n, 1, -3, 3, *s["add"])
    capi.launch_dequantize_i8(f, t, n, 0.04, 1)
    return s["q"], s["r"], s["t"], s["f"]


# A server loads a network once and keeps it; requests bring new inputs.

def _resident(net):
    module, fn = netlib.to_module(net)
    module.compile(fn)
    dm = H.DeviceManager().init()
    dm.add_network(module)
    return dm


@functools.lru_cache(maxsize=2)
def _resnet_profile(size):
    steps = resnet50.build_fp32(0)
    return steps, resnet50.profile(steps, resnet50.synthetic_images(1, 3, size))


@functools.lru_cache(maxsize=1)
def _resnet_server(batch, size):
    return _resident(resnet50.build_int8(*_resnet_profile(size), batch, size))


@functools.lru_cache(maxsize=1)
def _dlrm_server(batch, rows):
    net, max_idx = dlrm.make(tables=TABLES, rows=rows, batch=batch, bottom=BOTTOM, top=TOP,
                             dense_features=DENSE)
    return _resident(net), net, max_idx


def _request(inputs, outputs, pinned):
    if pinned:
        inputs = {k: capi.pinned_copy(v) for k, v in inputs.items()}
        outputs = {k: capi.pinned_copy(v) for k, v in outputs.items()}
    return dict(bindings=dict(inputs, **outputs), outputs=outputs)


def _prepare_resnet50(c, seed):
    dm = _resnet_server(c["batch"], c["size"])
    g = _gen(seed)
    shape = (c["batch"], c["size"], c["size"], 3)
    x = (torch.randn(shape, generator=g, device="cuda") * 0.25 + 0.45).cpu().numpy()
    out = dict(prob=np.zeros((c["batch"], 1000), np.float32),
               logits_q=np.zeros((c["batch"], 1000), np.int8))
    return dict(c, dm=dm, **_request({"input": x}, out, c["pinned"]))


def _prepare_dlrm(c, seed):
    dm, net, max_idx = _dlrm_server(c["batch"], c["rows"])
    inp = dlrm.Inputs(seed % 1_000_003, TABLES, c["rows"], c["batch"], 20, 1.1, DENSE)
    out = dict(prob=np.zeros((c["batch"], 1), np.float32),
               logit_q=np.zeros((c["batch"], 1), np.int8))
    return dict(c, dm=dm, **_request(dlrm.bindings(net, inp, max_idx), out, c["pinned"]))


def _run_request(s):
    s["dm"].run("main", s["bindings"])
    return s["outputs"]


_PREPARE = dict(slws=_prepare_slws, fc=_prepare_fc, conv=_prepare_conv,
                elementwise=_prepare_elementwise, resnet50=_prepare_resnet50, dlrm=_prepare_dlrm)
_RUN = dict(slws=_run_slws, fc=_run_fc, conv=_run_conv, elementwise=_run_elementwise,
            resnet50=_run_request, dlrm=_run_request)


@functools.lru_cache(maxsize=None)
def _init():
    capi.init(0)


def prepare(case, seed):
    _init()
    return _PREPARE[case["op"]](case, seed)


def run(state):
    return _RUN[state["op"]](state)


# ---- what a pass cannot do without ------------------------------------------------

def _resnet_work(c):
    """(multiply-accumulates, weights) of the network at this batch."""
    size = (c["size"] + 1) // 2
    macs, weights = size * size * 64 * 147, 64 * 147
    size, ch = (size + 1) // 2, 64
    for planes, blocks, stride in resnet50.LAYERS:
        for b in range(blocks):
            s = stride if b == 0 else 1
            after = (size + s - 1) // s
            if b == 0:
                weights += ch * planes * 4
                macs += after * after * ch * planes * 4
            weights += ch * planes + 9 * planes * planes + 4 * planes * planes
            macs += size * size * ch * planes + after * after * 13 * planes * planes
            size, ch = after, planes * 4
    return c["batch"] * (macs + ch * 1000), weights + ch * 1000


def _dlrm_work(c):
    b, macs, weights = c["batch"], 0, 0
    vectors = TABLES + 1
    for sizes, k in ((BOTTOM, DENSE), (TOP, BOTTOM[-1] + vectors * (vectors - 1) // 2)):
        for n in sizes:
            weights, k = weights + n * k, n
    macs = b * (weights + vectors * (vectors - 1) // 2 * BOTTOM[-1])
    lookups = b * 20 * TABLES
    # per lookup its 36-byte row and its index (on the host and as the kernel reads it)
    return macs, weights + lookups * (36 + 2 * 8) + b * (TABLES * 4 * 2 + DENSE * 4 * 2 + 5)


def work(case):
    c, op = case, case["op"]
    if op == "slws":
        looked = c["bags"] * c["mean_len"]
        row = capi.fused_row_bytes(c["cols"], c["kind"])
        out = 2 if c["kind"] in (capi.FUSED_U8_F16, capi.FUSED_U4_F16) else 4
        n = looked * ((8 if c["idx64"] else 4) + (4 if c["weighted"] else 0)) + c["bags"] * (4 + c["cols"] * out)
        # a row that several lookups share has to be read once
        return dict(bytes=n + min(looked, c["rows"]) * row, flops=looked * c["cols"] * 4)
    if op == "fc":
        M, K, N = c["M"], c["K"], c["N"]
        return dict(bytes=M * K + N * K + M * N + 9 * 4 * N, flops=2 * M * K * N)
    if op == "conv":
        g = _conv_geom(c)
        outs = c["N"] * g.OH * g.OW * c["OC"]
        per = c["k"] * c["k"] * (c["IC"] // c["group"])
        return dict(bytes=c["N"] * c["H"] * c["W"] * c["IC"] + c["OC"] * (per + 40) +
                    outs * (2 if c["residual"] else 1), flops=2 * outs * per)
    if op == "elementwise":
        return dict(bytes=c["n"] * (4 + 1 + 1 + 1 + 4), flops=c["n"] * 8)
    if op == "resnet50":
        macs, weights = _resnet_work(c)
        pixels = c["batch"] * c["size"] * c["size"] * 3
        # the image once on the host and once on the device, the weights, the answer
        return dict(bytes=pixels * 4 * 2 + weights + c["batch"] * 1000 * 5, flops=2 * macs)
    macs, nbytes = _dlrm_work(c)
    return dict(bytes=nbytes, flops=2 * macs)


def tolerance(case):
    op = case["op"]
    if op == "slws":
        # fp32 sums in any order; fp16 results are those rounded to 11 bits
        return {"rel": 1e-3 if case["kind"] in (capi.FUSED_U8_F16, capi.FUSED_U4_F16) else 1e-5}
    if op == "elementwise":
        return {"rel": 1e-6}       # the bytes are the same; the floats are products of them
    if op == "resnet50":
        return {"rel": 1e-5}       # int8 logits are the same; fp32 softmax
    if op == "dlrm":
        # the fp32 sum of a bag may land on the other side of a rounding tie, which
        # moves an int8 logit by one step in at most 2 of 1000 samples
        return {"rel": 2e-3, "max": 0.05, "differ": 0.002}
    return "exact"
