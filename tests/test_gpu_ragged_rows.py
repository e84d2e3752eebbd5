"""Row staging of convs whose rows are no multiple of 8 pixels.

Every candidate variant runs each geometry twice: with the row staging that
mlvc_hip_conv_plan asks for, and with vector_io = 0, the per-pixel staging.
Both give the same bits (one K order, the same padding), and both are within
the rounding bound of a 64-bit convolution. The input lies inside a buffer of
NaNs, so a staged element from outside the image would show.
"""

import ctypes as C
import sys

import numpy as np
import pytest
import torch
import torch.nn.functional as F

import mlvc_hip
from test_conv_candidates import ConvDesc

pytestmark = pytest.mark.gpu

NONE, LRELU, RESIDUAL, CLAMP = 0, 1, 2, 4
ALPHA, LO, HI = 0.01, -0.5, 0.75

# (n, ic, h, w, oc, k, stride, pad, epilogue, d2s, concat split)
CASES = [
    (1, 64, 7, 1, 64, 3, 1, 1, LRELU, 0, 0),        # one column
    (1, 64, 5, 7, 128, 3, 1, 1, NONE, 0, 0),        # one short segment, odd
    (1, 64, 6, 9, 64, 3, 1, 1, RESIDUAL, 0, 0),     # one pixel past a segment
    (1, 64, 7, 10, 64, 3, 1, 1, CLAMP, 0, 0),
    (1, 128, 9, 33, 256, 3, 1, 1, LRELU, 2, 0),     # one pixel past a 32-wide tile, shuffled out
    (1, 96, 10, 54, 192, 3, 1, 1, LRELU, 0, 0),     # even; partial channel pass (96 = 64 + 32)
    (1, 72, 13, 31, 40, 3, 1, 1, RESIDUAL, 0, 0),   # 8 channels past a 16-channel step, odd plane
    (1, 13, 7, 11, 12, 3, 1, 1, NONE, 2, 0),        # channels no multiple of 8, recon-like
    (2, 64, 5, 13, 64, 3, 1, 1, LRELU, 0, 0),       # two images, even plane offset
    (2, 13, 5, 13, 32, 3, 1, 1, LRELU, 0, 0),       # two images, second one off 4 bytes: per-pixel staging
    (1, 64, 9, 14, 64, 3, 1, 0, NONE, 0, 0),        # no padding: 12 output columns
    (1, 64, 9, 18, 64, 3, 1, 0, NONE, 0, 0),        # ragged in, 16 columns out
    (1, 64, 17, 33, 128, 3, 2, 1, LRELU, 0, 0),
    (1, 128, 9, 26, 256, 3, 2, 1, RESIDUAL, 0, 0),
    (1, 192, 8, 40, 128, 3, 2, 1, LRELU, 0, 0),     # aligned rows in, 20 columns out
    (1, 40, 11, 103, 72, 3, 2, 1, NONE, 0, 0),
    (1, 64, 5, 13, 96, 1, 1, 0, LRELU, 0, 0),       # 65 flattened pixels
    (1, 48, 9, 58, 64, 1, 1, 0, RESIDUAL, 0, 0),    # 522
    (2, 64, 3, 5, 32, 1, 1, 0, CLAMP, 0, 0),
    (1, 128, 7, 18, 64, 1, 1, 0, LRELU, 0, 64),     # channel concat
    (1, 64, 7, 11, 96, 1, 1, 0, LRELU, 0, 32),      # concats of odd planes: the second input's rows shift by a half too
    (1, 64, 7, 11, 64, 3, 1, 1, NONE, 0, 32),
    (1, 64, 9, 14, 64, 3, 1, 1, RESIDUAL, 0, 32),
    (1, 77, 6, 13, 32, 3, 1, 1, LRELU, 0, 64),      # the second input's 13 channels end inside a chunk
    (2, 77, 5, 13, 32, 3, 1, 1, LRELU, 0, 64),      # ...and its second image lies off 4 bytes: per-pixel staging
    (2, 45, 5, 13, 64, 1, 1, 0, CLAMP, 0, 32),
    (2, 96, 6, 13, 64, 3, 1, 1, NONE, 0, 48),       # two images, both inputs on 4 bytes
    (1, 768, 7, 11, 96, 1, 1, 0, LRELU, 0, 0),      # split K
]


def guarded(values, offset=8):
    """`values` as FP16 on the GPU between NaNs, `offset` halves past a 16-byte boundary (a multiple of 8 keeps it aligned)."""
    flat = values.half().reshape(-1)
    buf = torch.full((flat.numel() + offset + 64,), float("nan"), dtype=torch.float16, device="cuda")
    buf[offset:offset + flat.numel()] = flat.cuda()
    return buf, buf.data_ptr() + 2 * offset


def reference(x, w, b, r, case):
    """The conv in 64 bits, and a bound of any FP32-accumulated FP16 result's distance from it."""
    n, ic, h, wd, oc, k, s, p, epi, d2s, _ = case
    y = F.conv2d(x.double(), w.double(), b.double(), stride=s, padding=p)
    # FP32 accumulation of K products: K rounding steps of 2^-24 over the
    # absolute sum; then one FP16 rounding (2^-11) per operation, FP16
    # subnormals (2^-24) below that.
    tol = 2.0 ** -24 * ic * k * k * F.conv2d(x.double().abs(), w.double().abs(), b.double().abs(), stride=s, padding=p)
    tol = tol + 2.0 ** -11 * y.abs()
    if epi == LRELU:
        y = torch.where(y < 0, y * np.float32(ALPHA).item(), y)
        tol = tol + 2.0 ** -11 * y.abs()
    elif epi == RESIDUAL:
        y = y + r.double()
        tol = tol + 2.0 ** -11 * y.abs()
    elif epi == CLAMP:
        y = y.clamp(LO, HI)
    tol = tol * 1.01 + 2.0 ** -23
    return (F.pixel_shuffle(y, 2), F.pixel_shuffle(tol, 2)) if d2s else (y, tol)


def setup(case, offset=8):
    n, ic, h, w, oc, k, s, p, epi, d2s, split = case
    lib = mlvc_hip.device_lib()
    lib.mlvc_hip_conv_variant_name.restype = C.c_char_p
    lib.mlvc_hip_conv_plan.argtypes = lib.mlvc_hip_conv_pack.argtypes = None
    for f in (lib.mlvc_hip_conv_packed_bytes, lib.mlvc_hip_conv_bias_len, lib.mlvc_hip_conv_workspace_bytes):
        f.argtypes, f.restype = [C.POINTER(ConvDesc)], C.c_size_t
    g = torch.Generator().manual_seed(ic * 1000 + w)
    oh, ow = (h + 2 * p - k) // s + 1, (w + 2 * p - k) // s + 1
    x = torch.empty(n, ic, h, w).uniform_(-1, 1, generator=g).half()
    wt = (torch.randn(oc, ic, k, k, generator=g) * (2.0 / (ic * k * k)) ** 0.5).half()
    b = (0.1 * torch.randn(oc, generator=g)).half()
    r = torch.randn(n, oc, oh, ow, generator=g).half()
    d = ConvDesc(n=n, ic=ic, ih=h, iw=w, oc=oc, oh=oh, ow=ow, kh=k, kw=k, stride_h=s, stride_w=s, pad_h=p, pad_w=p,
                 epilogue=epi, alpha=ALPHA, clip_lo=LO, clip_hi=HI, out_d2s_block=d2s)
    keep = []
    if split:
        (ka, d.x), (kb, d.x2) = guarded(x[:, :split], offset), guarded(x[:, split:], offset)
        d.ic_split = split
        keep += [ka, kb]
    else:
        ka, d.x = guarded(x, offset)
        keep.append(ka)
    kr, d.residual = guarded(r)
    keep.append(kr)
    assert lib.mlvc_hip_conv_plan(C.byref(d)) == 0, lib.mlvc_hip_last_error()
    ws = lib.mlvc_hip_conv_workspace_bytes(C.byref(d))
    if ws:
        keep.append(torch.empty(ws, dtype=torch.uint8, device="cuda"))
        d.workspace, d.workspace_bytes = keep[-1].data_ptr(), ws
    shape = (n, oc // 4, 2 * oh, 2 * ow) if d2s else (n, oc, oh, ow)
    return lib, d, wt, b, keep, shape, reference(x, wt, b, r, case)


def run(lib, d, wt, b, shape, variant, vector_io):
    e = ConvDesc.from_buffer_copy(d)
    e.variant, e.vector_io = variant, vector_io
    packed = np.zeros(lib.mlvc_hip_conv_packed_bytes(C.byref(e)), np.uint8)
    rows = wt.contiguous()
    assert lib.mlvc_hip_conv_pack(C.byref(e), C.c_void_p(rows.data_ptr()), C.c_void_p(packed.ctypes.data)) == 0
    pw = torch.from_numpy(packed).cuda()
    bias = torch.zeros(lib.mlvc_hip_conv_bias_len(C.byref(e)), device="cuda")
    bias[:b.numel()] = b.float().cuda()
    count = int(np.prod(shape))
    y = torch.full((count + 80,), 123.0, dtype=torch.float16, device="cuda")
    e.packed_w, e.bias, e.y = pw.data_ptr(), bias.data_ptr(), y.data_ptr() + 16
    name = lib.mlvc_hip_conv_variant_name(variant).decode()
    print(f"{name} vector_io={vector_io}", flush=True)
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.mlvc_hip_conv_launch(C.byref(e), stream) == 0, (name, lib.mlvc_hip_last_error())
    out = y.cpu()
    assert (out[:8] == 123).all() and (out[8 + count:] == 123).all(), f"{name} wrote outside its output"
    return out[8:8 + count].reshape(shape)


@pytest.mark.parametrize("case", CASES, ids=lambda c: "n{}_ic{}_{}x{}_oc{}_k{}s{}p{}_e{}_d{}_c{}".format(*c))
def test_row_staging_equals_pixel_staging(case):
    print(case, flush=True)
    lib, d, wt, b, keep, shape, (want, tol) = setup(case)
    buf, count = (C.c_int * 512)(), C.c_int()
    assert lib.mlvc_hip_conv_candidates(C.byref(d), buf, 512, C.byref(count)) == 0
    assert d.vector_io == 1
    first = None
    for v in buf[:count.value]:
        for rows in (1, 0):
            name = lib.mlvc_hip_conv_variant_name(v).decode()
            if name.startswith("ws_") and not rows and case[3] % 8 == 0 and shape[3] % 8 == 0:
                continue
            got = run(lib, d, wt, b, shape, v, rows)
            if first is None:
                first = got
                worst = ((got.double() - want).abs() / tol).max().item()
                assert worst <= 1.0, f"{name}: {worst} of the bound"
            assert torch.equal(got.view(torch.int16), first.view(torch.int16)), f"{name}, rows={rows}"


# Operands off 16 bytes keep running, whatever the plan chooses: by per-pixel
# staging. Every variant of the cost table either runs them, with the same
# bits, or is one that no plan chooses and refuses them.
UNALIGNED = [CASES[3], CASES[12], CASES[16], (1, 96, 12, 32, 192, 3, 1, 1, LRELU, 0, 0), (1, 128, 16, 32, 256, 3, 1, 1, LRELU, 2, 0),
             (1, 64, 16, 48, 128, 3, 2, 1, RESIDUAL, 0, 0), (1, 128, 8, 16, 96, 1, 1, 0, LRELU, 0, 0)]
COSTED = ("ws_bm128_8x32_k3x3_s1_sc64_occ2", "ws_bm256_4x32_k3x3_s1_sc32_occ2_r3_pipe", "ws_bm256_8x16_k3x3_s1_sc32_occ2_r3_pipe",
          "ws_bm128_4x16_k3x3_s1_sc64_occ2_r18", "ws_bm64_2x32_k3x3_s1_sc64_occ4_w2_r9", "ws_bm128_4x40_k3x3_s1_sc64_occ2_r9",
          "ws_bm256_4x8_k3x3_s2_sc64_occ2_w8_r9")


@pytest.mark.parametrize("case", UNALIGNED, ids=lambda c: "n{}_ic{}_{}x{}_oc{}_k{}s{}p{}_e{}_d{}_c{}".format(*c))
def test_unaligned_input_pointer(case):
    print(case, flush=True)
    lib, d, wt, b, keep, shape, (want, tol) = setup(case)
    aligned = run(lib, d, wt, b, shape, d.variant, 1)
    buf, count = (C.c_int * 512)(), C.c_int()
    assert lib.mlvc_hip_conv_candidates(C.byref(d), buf, 512, C.byref(count)) == 0
    names = {lib.mlvc_hip_conv_variant_name(v).decode(): v for v in buf[:count.value]}
    lib, d, wt, b, keep, shape, _ = setup(case, offset=9)
    for v in {d.variant, *(names[n] for n in COSTED if n in names)}:
        assert torch.equal(run(lib, d, wt, b, shape, v, 1).view(torch.int16), aligned.view(torch.int16))


@pytest.mark.parametrize("case", [CASES[1], (1, 64, 5, 16, 128, 3, 1, 1, LRELU, 0, 0), (1, 64, 6, 9, 64, 3, 1, 1, LRELU, 2, 0), CASES[12],
                                  CASES[16], (1, 64, 5, 14, 96, 1, 1, 0, LRELU, 0, 0)],
                         ids=lambda c: "n{}_ic{}_{}x{}_oc{}_k{}s{}p{}_e{}_d{}_c{}".format(*c))
def test_slope_zero_of_an_infinity(monkeypatch, case):
    """LeakyReLU with slope 0 is a product: a sum past FP16's range, -inf, gives NaN on every width and variant."""
    monkeypatch.setattr(sys.modules[__name__], "ALPHA", 0.0)
    case = case[:8] + (LRELU,) + case[9:]
    print(case, flush=True)
    lib, d, wt, b, keep, shape, _ = setup(case)
    n, ic, h, w, oc, k, s, p = case[:8]
    wt = (wt.float() * (60000.0 / wt.abs().max().item())).half()  # sums of around 100000
    x = keep[0][8:8 + n * ic * h * w].cpu().reshape(n, ic, h, w)
    y = F.conv2d(x.double(), wt.double(), b.double(), stride=s, padding=p)
    y = F.pixel_shuffle(y, 2) if case[9] else y
    low, high, mid = y < -66000, y > 66000, (y < -1) & (y > -65000)  # away from FP16's largest value, 65504
    assert low.any() and high.any() and mid.any()
    buf, count = (C.c_int * 512)(), C.c_int()
    assert lib.mlvc_hip_conv_candidates(C.byref(d), buf, 512, C.byref(count)) == 0
    for v in buf[:count.value]:
        for rows in (1, 0):
            if rows == 0 and lib.mlvc_hip_conv_variant_name(v).decode().startswith("ws_"):
                continue
            got = run(lib, d, wt, b, shape, v, rows)
            assert got[low].isnan().all() and (got[high] == float("inf")).all() and (got[mid] == 0).all()
