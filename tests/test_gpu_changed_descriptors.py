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


def check(before, after, kind, refused=False):
    """`after` run with the variant of `before` (whose name starts with `kind`)."""
    print(before, after, flush=True)
    lib, d, wt, b, keep, shape, _ = rows.setup(after)
    n, oc, oh, ow = d.n, d.oc, d.oh, d.ow
    if after[8] == REGLU:
        shape = (n, oc // 2, oh, ow)
    elif d.out_d2s_block > 1:
        bs = d.out_d2s_block
        shape = (n, oc // bs ** 2, oh * bs, ow * bs)
    a = planned(lib, before)
    assert lib.mlvc_hip_conv_variant_name(a.variant).decode().startswith(kind)
    if refused:
        with pytest.raises(AssertionError):
            rows.run(lib, d, wt, b, shape, a.variant, a.vector_io)
        return
    want = rows.run(lib, d, wt, b, shape, d.variant, d.vector_io)
    got = rows.run(lib, d, wt, b, shape, a.variant, a.vector_io)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


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
