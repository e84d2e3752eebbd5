"""Groups of eight elements on any alignment: planes of a length that is no
multiple of 8 give, element for element, what the same planes give padded to
one (the operators are elementwise over the planes), and nothing past a
plane's end is written. Large launches, with non-temporal accesses, too: the
feature update on three channels of 9000003 pixels, both tails on one.
"""

import ctypes as C

import pytest
import torch

import mlvc_hip

pytestmark = pytest.mark.gpu

Y0 = ("latent", "prior", "quant_scale", "update_scale0", "update_scale1", "normalized", "clipped", "y_raw", "concat2", "concat3")
Y1 = ("normalized", "prior", "quant_scale", "update_scale0", "update_scale1", "concat2", "clipped", "y_raw", "out")
Y0_PLANES = (2, 4, 2, 1, 1, 2, 2, 1, 2, 6)
Y1_PLANES = (2, 2, 2, 1, 1, 2, 2, 1, 2)


class Y0Desc(C.Structure):
    _fields_ = [(f, C.c_void_p) for f in Y0] + [("n", C.c_int), ("q", C.c_int), ("hw", C.c_size_t), ("clip_min", C.c_float)]


class Y1Desc(C.Structure):
    _fields_ = [(f, C.c_void_p) for f in Y1] + [("n", C.c_int), ("q", C.c_int), ("hw", C.c_size_t)]


def ok(rc):
    assert rc == 0, mlvc_hip.device_lib().mlvc_hip_last_error()


def planes(g, count, hw):
    """`count` planes of hw elements, and the same padded to a multiple of 8, on the GPU; guards behind both."""
    x = torch.randn(count, hw, generator=g).half()
    padded = torch.zeros(count, -(-hw // 8) * 8, dtype=torch.float16)
    padded[:, :hw] = x
    return tuple(torch.cat([t.reshape(-1), torch.full((64,), 9.0, dtype=torch.float16)]).cuda() for t in (x, padded))


def same(ragged, padded, count, hw):
    p8 = -(-hw // 8) * 8
    a, b = ragged[:count * hw].reshape(count, hw), padded[:count * p8].reshape(count, p8)[:, :hw]
    assert torch.equal(a.view(torch.int16), b.contiguous().view(torch.int16))
    assert (ragged[count * hw:] == 9).all() and (padded[count * p8:] == 9).all()


# 9 million pixels of one channel: over 256 MB, so non-temporal, in the tails;
# of three channels (309 MB) in the feature update, where one moves 103 MB.
SIZES = [(1, 3, 1), (1, 3, 7), (2, 5, 9), (1, 16, 30), (1, 7, 135 * 241), (1, 1, 9000003)]
FEATURE_SIZES = SIZES + [(1, 3, 9000003)]


@pytest.mark.parametrize("n,c,hw", FEATURE_SIZES)
def test_feature_update(n, c, hw):
    print(n, c, hw, flush=True)
    g = torch.Generator().manual_seed(hw)
    x, hist = planes(g, 3 * n * c, hw), planes(g, n * c, hw)
    scale = torch.rand(c, generator=g).half().cuda()
    out = planes(g, 2 * n * c, hw)
    lib, stream = mlvc_hip.device_lib(), C.c_void_p(torch.cuda.current_stream().cuda_stream)
    for i, m in enumerate((hw, -(-hw // 8) * 8)):
        ok(lib.mlvc_hip_feature_update(*(C.c_void_p(t.data_ptr()) for t in (x[i], hist[i], scale, out[i])), None, None, n, c,
                                       C.c_size_t(m), stream))
    torch.cuda.synchronize()
    same(*out, 2 * n * c, hw)


@pytest.mark.parametrize("n,q,hw", SIZES)
def test_quantisation_tails(n, q, hw):
    print(n, q, hw, flush=True)
    g = torch.Generator().manual_seed(hw + 1)
    lib, stream = mlvc_hip.device_lib(), C.c_void_p(torch.cuda.current_stream().cuda_stream)
    for desc, counts, outs, launch in ((Y0Desc, Y0_PLANES, 5, lib.mlvc_hip_y0_tail), (Y1Desc, Y1_PLANES, 2, lib.mlvc_hip_y1_tail)):
        t = [planes(g, n * q * k, hw) for k in counts]
        for i, m in enumerate((hw, -(-hw // 8) * 8)):
            d = desc(*(x[i].data_ptr() for x in t), n, q, m, *([0.11] if desc is Y0Desc else []))
            ok(launch(C.byref(d), stream))
        torch.cuda.synchronize()
        for x, k in list(zip(t, counts))[-outs:]:
            same(*x, n * q * k, hw)
