"""Descriptors changed after their plan: a variant chosen for one conv runs
another one (another epilogue, block, size, split or fusion) with the bits of
that conv's own plan, or refuses it. The weights are packed after the change,
as the packed layout is the variant's.
"""

import ctypes as C

import pytest
import torch

import test_gpu_ragged_rows as rows
from test_conv_candidates import ConvDesc
from test_gpu_ragged_rows import LRELU, NONE

pytestmark = pytest.mark.gpu

REGLU = 3


def planned(lib, case, **fields):
    """The variant and staging that `case` is planned onto, without tensors."""
    n, ic, h, w, oc, k, s, p, epi, d2s, split = case
    d = ConvDesc(n=n, ic=ic, ih=h, iw=w, oc=oc, oh=(h + 2 * p - k) // s + 1, ow=(w + 2 * p - k) // s + 1, kh=k, kw=k, stride_h=s,
                 stride_w=s, pad_h=p, pad_w=p, epilogue=epi, alpha=rows.ALPHA, out_d2s_block=d2s, ic_split=split, **fields)
    assert lib.mlvc_hip_conv_plan(C.byref(d)) == 0, lib.mlvc_hip_last_error()
    return d


def check(before, after, kind, refused=False, ksplit=None, **fields):
    """`after` (its descriptor with `fields` set, its split K as given) run with
    the variant of `before`, whose name starts with `kind`."""
    print(before, after, ksplit, fields, flush=True)
    lib, d, wt, b, keep, shape, _ = rows.setup(after)
    for f, v in fields.items():
        setattr(d, f, v)
    if after[8] == REGLU:
        shape = (d.n, d.oc // 2, d.oh, d.ow)
    elif d.out_d2s_block > 1:
        bs = d.out_d2s_block
        shape = (d.n, d.oc // bs ** 2, d.oh * bs, d.ow * bs)
    a = planned(lib, before)
    assert lib.mlvc_hip_conv_variant_name(a.variant).decode().startswith(kind)
    if refused:
        with pytest.raises(AssertionError):
            rows.run(lib, d, wt, b, shape, a.variant, a.vector_io)
        return
    assert lib.mlvc_hip_conv_plan(C.byref(d)) == 0, lib.mlvc_hip_last_error()
    if ksplit:
        d.ksplit, d.split_c = ksplit
    ws = torch.empty(max(16, lib.mlvc_hip_conv_workspace_bytes(C.byref(d))), dtype=torch.uint8, device="cuda")
    d.workspace, d.workspace_bytes = ws.data_ptr(), ws.numel()
    buf, count = (C.c_int * 512)(), C.c_int()
    assert lib.mlvc_hip_conv_candidates(C.byref(d), buf, 512, C.byref(count)) == 0
    general = [v for v in buf[:count.value] if lib.mlvc_hip_conv_variant_name(v).decode().startswith("mfma_bm")][0]
    want = rows.run(lib, d, wt, b, shape, general, 0)
    for staging in {a.vector_io, 0}:
        got = rows.run(lib, d, wt, b, shape, a.variant, staging)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), staging


def conv3(oc=128, epi=NONE, d2s=0, h=30, w=40, ic=64, split=0, stride=1, n=1):
    return (n, ic, h, w, oc, 3, stride, 1, epi, d2s, split)


@pytest.mark.parametrize("w", [40, 41, 54])
def test_epilogues_the_weight_streaming_kernel_lacks(w):
    check(conv3(w=w), conv3(w=w, epi=REGLU), "ws_")
    check(conv3(w=w, oc=144), conv3(w=w, oc=144, d2s=3), "ws_")
    check(conv3(w=w, epi=LRELU, d2s=2), conv3(w=w, epi=LRELU, d2s=4), "ws_")
    check(conv3(w=w, stride=2), conv3(w=w, stride=2, epi=REGLU), "ws_")


def test_reglu_needs_whole_64_channel_blocks():
    check(conv3(oc=64, h=100, w=200, ic=16), conv3(oc=64, h=100, w=200, ic=16, epi=REGLU), "mfma_bm32_", refused=True)


def conv1(ic=64, oc=96, h=10, w=14, epi=LRELU, d2s=0, split=0, n=1):
    return (n, ic, h, w, oc, 1, 1, 0, epi, d2s, split)


DEEP = conv1(ic=1024, oc=256, h=23, w=40)


@pytest.mark.parametrize("ksplit", [(1, 1024), (2, 512), (7, 160), (11, 96), (16, 64)])
def test_splits_of_a_conv_planned_split(ksplit):
    check(DEEP, DEEP, "mfma_ptk", ksplit=ksplit)


def test_splits_of_a_conv_planned_whole():
    plain = conv1(ic=512, oc=128, h=16, w=20)
    check(plain, plain, "mfma_pt_", ksplit=(2, 256))
    check(plain, plain, "mfma_pt_", ksplit=(16, 32))
    check(conv3(oc=64), conv3(oc=64), "ws_", ksplit=(2, 32))


def test_fusions_of_a_conv_planned_plain():
    check(conv1(), conv1(split=40), "mfma_pt_")           # a concat off a 16-channel step
    check(DEEP, conv1(ic=1024, oc=256, h=23, w=40, split=256), "mfma_ptk")
    check(conv1(oc=128), conv1(oc=128, epi=REGLU), "mfma_pt_w2")
    check(conv1(), conv1(d2s=2), "mfma_pt_")
    check(conv1(), conv1(), "mfma_pt_", in_s2d_block=2)
    check(DEEP, DEEP, "mfma_ptk", in_s2d_block=2)
    check(conv3(), conv3(split=24), "ws_")
    check(conv3(), conv3(), "ws_", in_s2d_block=2)


def test_sizes_of_another_plan():
    check(conv1(h=10, w=14), conv1(h=9, w=15), "mfma_pt_")  # an odd plane
    check(conv1(ic=64), conv1(ic=72), "mfma_pt_")           # no whole passes of channels
    check(DEEP, conv1(ic=608, oc=40, h=9, w=16), "mfma_ptk")
    check(conv3(ic=64), conv3(ic=80), "ws_")                # no whole rings
