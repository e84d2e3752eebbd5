"""The 1x1 kernels over flattened pixels (LDS DMA and transposing LDS reads),
with all splits of a split conv in one workgroup where there are any.

Every candidate variant runs each geometry with its row staging and with
vector_io = 0 (the per-pixel staging of the general kernel; split convs then
sum through memory): the same bits, within the rounding bound of a 64-bit
convolution. Inputs lie between NaNs, outputs between guards.
"""

import ctypes as C

import pytest
import torch

import test_gpu_ragged_rows as rows
from test_gpu_ragged_rows import CLAMP, LRELU, NONE, RESIDUAL

pytestmark = pytest.mark.gpu

# (n, ic, h, w, oc, k, stride, pad, epilogue, d2s, concat split)
CASES = [
    (1, 32, 1, 2, 32, 1, 1, 0, NONE, 0, 0),       # two pixels
    (1, 64, 5, 6, 33, 1, 1, 0, LRELU, 0, 0),      # 30: short of a 32-pixel tile; one channel past a block
    (1, 64, 2, 17, 96, 1, 1, 0, RESIDUAL, 0, 0),  # 34: one pair past it
    (1, 128, 3, 42, 64, 1, 1, 0, LRELU, 0, 0),    # 126, short of a 128-pixel tile
    (1, 128, 16, 8, 192, 1, 1, 0, NONE, 0, 0),    # 128
    (1, 256, 10, 13, 200, 1, 1, 0, CLAMP, 0, 0),  # 130
    (1, 512, 4, 33, 31, 1, 1, 0, LRELU, 0, 0),    # 132, several passes of channels
    (1, 96, 9, 32, 128, 1, 1, 0, NONE, 0, 0),     # channels a multiple of 32 only
    (1, 160, 8, 40, 256, 1, 1, 0, RESIDUAL, 0, 0),
    (3, 64, 5, 26, 40, 1, 1, 0, LRELU, 0, 0),     # three images
    (1, 128, 7, 20, 64, 1, 1, 0, LRELU, 0, 64),   # concats: on a pass, inside one, off a step (general kernel only)
    (2, 192, 6, 22, 96, 1, 1, 0, NONE, 0, 48),
    (1, 64, 6, 22, 96, 1, 1, 0, NONE, 0, 40),
    (1, 768, 5, 8, 96, 1, 1, 0, LRELU, 0, 0),     # six splits of 128
    (1, 576, 3, 22, 33, 1, 1, 0, RESIDUAL, 0, 0), # the last split half a pass
    (2, 640, 2, 31, 64, 1, 1, 0, CLAMP, 0, 0),
    (1, 1024, 17, 2, 256, 1, 1, 0, NONE, 0, 0),   # eight splits
    (1, 1024, 49, 118, 32, 1, 1, 0, LRELU, 0, 0), # 5782 pixels
    (1, 768, 168, 168, 96, 1, 1, 0, NONE, 0, 0),  # two splits of 384
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "n{}_ic{}_{}x{}_oc{}_k{}s{}p{}_e{}_d{}_c{}".format(*c))
def test_point_kernels(case):
    rows.test_row_staging_equals_pixel_staging(case)


@pytest.mark.parametrize("alpha", [1.5, -0.25])
def test_leaky_select_form(monkeypatch, alpha):
    """LeakyReLU slopes outside [0, 1] take the select form."""
    monkeypatch.setattr(rows, "ALPHA", alpha)
    rows.test_row_staging_equals_pixel_staging(CASES[1])
    rows.test_row_staging_equals_pixel_staging(CASES[13])


def test_planned_choice():
    """Large and small plain convs are planned onto the 1x1 kernels, odd planes onto the general one."""
    names = {}
    for case in (CASES[4], CASES[13], (1, 64, 5, 13, 96, 1, 1, 0, NONE, 0, 0)):
        lib, d = rows.setup(case)[:2]
        names[case] = lib.mlvc_hip_conv_variant_name(d.variant).decode()
    kinds = [n.split("_")[1] for n in names.values()]
    assert kinds[:2] == ["pt", "ptk"] and kinds[2].startswith("bm"), names


def test_extreme_values():
    """Infinities, NaN, subnormals and signed zeros come out as the general kernel's bits."""
    case = CASES[5]
    lib, d, wt, b, keep, shape, _ = rows.setup(case)
    x = keep[0][8:8 + case[1] * case[2] * case[3]]
    special = torch.tensor([float("inf"), float("-inf"), float("nan"), 0.0, -0.0, 6e-8, -6e-8, 65504.0], dtype=torch.float16)
    x[::37] = special.repeat(x[::37].numel() // 8 + 1)[:x[::37].numel()].cuda()
    buf, count = (C.c_int * 512)(), C.c_int()
    assert lib.mlvc_hip_conv_candidates(C.byref(d), buf, 512, C.byref(count)) == 0
    want = rows.run(lib, d, wt, b, shape, buf[0], 0)
    for v in buf[:count.value]:
        got = rows.run(lib, d, wt, b, shape, v, 1)
        nan = torch.isnan(want)
        assert torch.equal(torch.isnan(got), nan)
        assert torch.equal(got[~nan].view(torch.int16), want[~nan].view(torch.int16))


# (case, ksplit, split_c): splits set by hand, as a tuner of its own sets them.
# The kernel that keeps all splits in one workgroup multiplies 64 channels at a
# time; other splits (a last half of 32 channels) sum through memory.
HAND_SPLITS = [((1, 1024, 23, 40, 256, 1, 1, 0, LRELU, 0, 0), 7, 160), ((1, 1024, 5, 34, 96, 1, 1, 0, RESIDUAL, 0, 0), 8, 128),
               ((2, 768, 3, 22, 64, 1, 1, 0, NONE, 0, 0), 8, 96), ((1, 640, 5, 8, 33, 1, 1, 0, CLAMP, 0, 0), 2, 320)]


@pytest.mark.parametrize("case,ksplit,split_c", HAND_SPLITS, ids=lambda v: str(v))
def test_splits_set_by_hand(case, ksplit, split_c):
    """A planned descriptor runs them with its variant; the sums are those of a general tile's two kernels."""
    print(case, ksplit, split_c, flush=True)
    lib, d, wt, b, keep, shape, (want, tol) = rows.setup(case)
    d.ksplit, d.split_c = ksplit, split_c
    ws = torch.empty(lib.mlvc_hip_conv_workspace_bytes(C.byref(d)), dtype=torch.uint8, device="cuda")
    d.workspace, d.workspace_bytes = ws.data_ptr(), ws.numel()
    assert lib.mlvc_hip_conv_variant_name(d.variant).decode().startswith("mfma_ptk")
    buf, count = (C.c_int * 512)(), C.c_int()
    assert lib.mlvc_hip_conv_candidates(C.byref(d), buf, 512, C.byref(count)) == 0
    first = rows.run(lib, d, wt, b, shape, buf[0], 0)
    assert lib.mlvc_hip_conv_variant_name(buf[0]).decode().startswith("mfma_bm")
    assert ((first.double() - want).abs() / tol).max().item() <= 1.0
    for v in {d.variant, *buf[:count.value]}:
        for staging in (1, 0):
            assert torch.equal(rows.run(lib, d, wt, b, shape, v, staging).view(torch.int16), first.view(torch.int16))
