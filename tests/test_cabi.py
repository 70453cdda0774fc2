"""The C-ABI library loads on a machine without a GPU and exports every symbol the header declares."""
import ctypes
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared(header):
    with open(os.path.join(ROOT, "include", header)) as f:
        text = re.sub(r"/\*.*?\*/", "", f.read(), flags=re.S)
    return sorted(set(re.findall(r"\b(espdl_\w+)\s*\(", text)))


def test_libespdl_hip_exports_header_symbols():
    path = os.path.join(ROOT, "esp-dl_amd", "lib", "libespdl_hip.so")
    assert os.path.exists(path), "run `python esp-dl_amd/build.py` (or __graft_entry__.build()) first"
    lib = ctypes.CDLL(path)
    names = _declared("espdl_hip.h")
    assert len(names) >= 12
    for name in names:
        assert hasattr(lib, name), f"{name} is declared in include/espdl_hip.h but not exported"


def test_validation_needs_no_gpu():
    import importlib
    m = importlib.import_module("esp-dl_amd")
    d = m.capi.make_desc((1, 56, 56, 64), 64, (3, 3), pads=(1, 1, 1, 1))
    assert m.conv_out_shape(d) == (56, 56)
    d = m.capi.make_desc((1, 100, 50, 3), 16, (3, 3), stride=(2, 2))
    assert m.conv_out_shape(d) == (49, 24)
    d.group = 5
    try:
        m.conv_out_shape(d)
        assert False
    except m.EspdlHipError as e:
        assert "group" in str(e)


def test_requantized_residual_is_refused_for_misaligned_operands():
    """A block whose shape alone passes for the workgroup-per-tile kernel but whose input is only 4-byte aligned
    falls to kernels that add the residual operand as it is: with residual_shift != 0 the call must fail with
    ESPDL_HIP_ENOTSUP before anything is launched (no GPU needed: the pointers are never followed)."""
    import ctypes as C
    import importlib
    m = importlib.import_module("esp-dl_amd")
    d = m.capi.MbconvDesc(1, 14, 14, 96, 576, 96, 1, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 0, 0, 1, 1, 1)
    d.residual_shift = 2
    assert m.lib().espdl_hip_mbconv_s8_supported(C.byref(d)) == 5
    base = 1 << 20  # a fake device address, 256-byte aligned
    w = m.capi.MbconvWeights(base * 3, None, base * 4, base * 5, None, base * 6, base * 7, None, base * 8)
    rc = m.lib().espdl_hip_mbconv_s8(C.byref(d), C.c_void_p(base + 4), C.byref(w), C.c_void_p(base * 9), C.c_void_p(base * 10), None)
    assert rc == -95, m.lib().espdl_hip_last_error()
    assert b"residual_shift" in m.lib().espdl_hip_last_error()


def test_conv2d_refuses_other_types_than_int8_and_int16():
    """The library would read the bytes of any other tensor as one of the two (no GPU needed: nothing is launched)."""
    import importlib
    import pytest
    import torch
    m = importlib.import_module("esp-dl_amd")
    f, shift = torch.zeros(16 * 16, dtype=torch.int8), torch.zeros(1, dtype=torch.int32)
    for dtype in (torch.uint8, torch.bool, torch.float16, torch.bfloat16, torch.int32, torch.float32):
        with pytest.raises(m.EspdlHipError, match="int8 or int16"):
            m.conv2d(torch.zeros((1, 4, 4, 16), dtype=dtype), f, None, shift, (1, 1), stream=0)


def test_two_launches_are_weighed_against_the_launch_that_a_block_with_an_add_takes():
    """The descriptor of a block has no residual operand, the launch has: where input and output have one shape the choice
    between one and two launches has to count the kernel that takes the operand.  Each of these takes 14 to 65 % longer as one
    launch (no GPU needed: the answer follows from estimates)."""
    import ctypes as C
    import importlib
    m = importlib.import_module("esp-dl_amd")
    for batch, hw, cin, ce, half_even in ((7, 56, 24, 144, 0), (8, 56, 24, 144, 1), (28, 28, 32, 96, 1), (14, 40, 32, 144, 1), (10, 28, 48, 144, 0)):
        d = m.capi.MbconvDesc(batch, hw, hw, cin, ce, cin, 1, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 0, half_even, ce, ce, cin)
        assert m.lib().espdl_hip_mbconv_s8_workspace(C.byref(d)) == batch * hw * hw * ce, (batch, hw, cin, ce, half_even)
    # a depthwise stride takes the operand away, and with it the reason
    d = m.capi.MbconvDesc(24, 56, 56, 24, 144, 24, 1, 3, 3, 2, 2, 1, 1, 1, 1, 1, 1, 1, 1, 0, 0, 144, 144, 24)
    assert m.lib().espdl_hip_mbconv_s8_workspace(C.byref(d)) == 0


def test_one_or_two_launches_of_a_block_by_what_each_takes():
    """Blocks that one form takes a tenth less time for and more (us as two launches, and as one or as separate
    convolutions): large ones that no single launch has a fast build for, and ones on either side of the line."""
    import ctypes as C
    import importlib
    m = importlib.import_module("esp-dl_amd")
    for batch, hw, cin, ce, cout, half_even, two in (
            (226, 56, 64, 384, 64, 0, True),     # 228, 327 as convolutions
            (362, 56, 40, 240, 40, 0, True),     # 274, 316
            (452, 56, 48, 192, 48, 0, True),     # 255, 323
            (177, 80, 40, 240, 40, 0, True),     # 285, 317
            (905, 28, 64, 384, 64, 0, True),     # 227, 329
            (215, 112, 48, 288, 48, 1, True),    # 787, 921
            (63, 32, 24, 144, 24, 1, False),     # 32.1, 19.5 as one launch
            (17, 64, 24, 144, 24, 1, False),     # 31.6, 19.9
            (122, 28, 32, 192, 32, 1, False),    # 36.2, 23.1
            (128, 14, 96, 576, 96, 0, False),    # 31.9, 16.5
            (40, 10, 96, 576, 96, 0, True),      # 11.5, 15.1
            (139, 12, 32, 192, 32, 1, True),     # 11.5, 17.5
            (65, 32, 20, 112, 20, 1, False),     # 22.7, 16.7
            (164, 20, 32, 192, 32, 1, False),    # 28.8, 22.4
            (6, 7, 160, 960, 160, 1, True)):     # 7.2, 24.6
        d = m.capi.MbconvDesc(batch, hw, hw, cin, ce, cout, 1, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 0, half_even, ce, ce, cout)
        assert m.lib().espdl_hip_mbconv_s8_workspace(C.byref(d)) == (batch * hw * hw * ce if two else 0), (batch, hw, cin, ce, cout, half_even)
    # with Clips between the stages: 21 images 22.1 us as two launches, 17.5 as one
    d = m.capi.MbconvDesc(21, 56, 56, 24, 144, 24, 1, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 0, 0, 144, 144, 24)
    d.clip_expand = d.clip_dw = 1
    d.clip_expand_max = d.clip_dw_max = 96
    assert m.lib().espdl_hip_mbconv_s8_workspace(C.byref(d)) == 0


def _dense_kernel(m, shape, out_c, k, stride=1, pad=None, dilation=1, lut=None, residual=None, half_even=0, out_pitch=0, group=1, dtype=None):
    import ctypes as C
    pad = k // 2 * dilation if pad is None else pad
    d = m.capi.make_desc(shape, out_c, (k, k), (stride, stride), (dilation, dilation), (pad,) * 4, group=group, round_mode=half_even,
                         n_shift=out_c, dtype=m.capi.S8 if dtype is None else dtype)
    d.out_pitch = out_pitch
    return m.lib().espdl_hip_conv2d_s8_kernel(C.byref(d), 1 << 20, 2 << 20, lut, residual, 3 << 20)


def test_dense_kernels_are_named_without_a_launch():
    """One layer of each kernel of the dense dispatch, and the calls it refuses (no GPU needed)."""
    import importlib
    m = importlib.import_module("esp-dl_amd")
    assert _dense_kernel(m, (256, 56, 56, 64), 64, 3) == b"conv2d_s8_walk"
    assert _dense_kernel(m, (64, 640, 640, 3), 16, 3, 2) == b"conv2d_s8_walk_stem"
    assert _dense_kernel(m, (64, 641, 641, 3), 16, 3, 2) == b"conv2d_s8_stem"
    assert _dense_kernel(m, (1, 20, 20, 16), 16, 3) == b"conv2d_s8_narrow"
    assert _dense_kernel(m, (80, 30, 31, 31), 64, 5, 2) == b"conv2d_s8_unitgemm"
    assert _dense_kernel(m, (256, 14, 14, 576), 96, 1) == b"conv2d_s8_pwgemm"
    assert _dense_kernel(m, (256, 56, 56, 64), 64, 3, half_even=1) == b"conv2d_s8_tiled"
    assert _dense_kernel(m, (256, 80, 80, 32), 48, 1, half_even=1) == b"conv2d_s8"
    assert _dense_kernel(m, (1, 1, 20480, 120), 6625, 1) == b"conv2d_s8_wide"
    assert _dense_kernel(m, (1, 20, 20, 16), 16, 3, out_pitch=8) is None
    assert _dense_kernel(m, (1, 20, 20, 16), 16, 3, group=16) is None
    assert _dense_kernel(m, (1, 20, 20, 16), 16, 3, dtype=m.capi.S16) is None


def test_block_kernels_are_named_without_a_launch():
    import ctypes as C
    import importlib
    m = importlib.import_module("esp-dl_amd")
    base = 1 << 20

    def kernel(batch, hw, cin, ce, cout, stride=1, residual=False, shift=0, aligned=True, stem=False):
        d = m.capi.MbconvDesc(batch, hw, hw, cin, ce, cout, 1, 3, 3, stride, stride, 1, 1, 1, 1, 1, 1, 1, 1, 0, 0, ce, ce, cout)
        d.residual_shift = shift
        if stem:
            d.exp_k_h = d.exp_k_w = 3
            d.exp_stride_h = d.exp_stride_w = 2
            d.exp_pad_top = d.exp_pad_bottom = d.exp_pad_left = d.exp_pad_right = 1
        w = m.capi.MbconvWeights(base * 3, None, base * 4, base * 5, None, base * 6, base * 7, None, base * 8)
        return m.lib().espdl_hip_mbconv_s8_kernel(C.byref(d), base + (0 if aligned else 4), C.byref(w), base * 9 if residual else None, base * 10)

    assert kernel(256, 56, 24, 144, 24, residual=True) == b"mbconv_s8_walk"
    assert kernel(256, 28, 32, 192, 32, residual=True) == b"mbconv_s8_wave"
    assert kernel(256, 14, 96, 576, 96, residual=True) == b"mbconv_s8_group"
    assert kernel(256, 224, 3, 32, 16, stem=True) == b"mbconv_s8_walk_stem"
    assert kernel(4, 224, 3, 32, 16, stem=True) == b"mbconv_s8_wave"
    assert kernel(256, 14, 96, 576, 96, residual=True, shift=2, aligned=False) is None


def test_dense_layers_go_to_the_faster_kernel():
    """Layers that one kernel takes less time for, most of them a tenth and more (measured with operands that change from
    launch to launch; us there and on the other kernel)."""
    import importlib
    m = importlib.import_module("esp-dl_amd")
    for shape, out_c, k, stride, kernel in (
            ((194, 79, 72, 17), 202, 1, 1, b"conv2d_s8"),          # 120, 181
            ((14, 35, 43, 16), 96, 5, 1, b"conv2d_s8_unitgemm"),   # 7.5, 10.6
            ((43, 75, 11, 16), 240, 5, 2, b"conv2d_s8_unitgemm"),  # 7.8, 8.9
            ((9, 13, 43, 16), 64, 3, 1, b"conv2d_s8_narrow"),      # 3.3, 3.9
            ((1, 20, 20, 240), 16, 3, 1, b"conv2d_s8_narrow"),     # 3.9, 9.0
            ((15, 42, 21, 84), 24, 3, 2, b"conv2d_s8_narrow"),     # 4.3, 6.3
            ((1, 1, 40, 120), 6625, 1, 1, b"conv2d_s8_pwgemm"),    # 4.7, 8.4
            ((2, 4, 32, 96), 6576, 3, 2, b"conv2d_s8_narrow"),     # 8.1, 62
            ((286, 4, 1, 96), 4969, 3, 1, b"conv2d_s8_walk"),      # 30, 402
            ((364, 5, 1, 16), 6078, 5, 1, b"conv2d_s8_walk"),      # 45, 340
            ((1, 56, 56, 64), 64, 3, 1, b"conv2d_s8_walk"),        # 4.1, 4.2
            ((82, 15, 19, 16), 171, 1, 1, b"conv2d_s8_walk"),      # 4.9, 7.7
            ((39, 8, 8, 116), 107, 1, 1, b"conv2d_s8_walk"),       # 3.2, 4.4
            ((10, 18, 26, 43), 25, 3, 1, b"conv2d_s8_walk"),       # 4.4, 6.5
            ((4, 44, 8, 125), 14, 1, 1, b"conv2d_s8_walk"),        # 3.0, 4.2
            ((153, 12, 69, 240), 16, 3, 1, b"conv2d_s8_walk")):    # 17.6, 43
        assert _dense_kernel(m, shape, out_c, k, stride) == kernel, (shape, out_c, k, stride)
