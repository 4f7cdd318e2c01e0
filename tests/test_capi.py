"""The C-ABI library: loads, exports the header, host utilities (CPU only).

No call here launches a kernel: only host-side functions and argument
validation paths that return before touching the device.
"""

import ctypes
import re
from pathlib import Path

import numpy as np
import pytest
import torch

from sparseflow_amd import _lib

HEADER = Path(__file__).resolve().parents[1] / "include" / "sparseflow.h"


def header_functions():
    text = HEADER.read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(sf_[a-z0-9_]+)\s*\(", text)))


def test_library_loads_and_exports_every_declared_symbol():
    lib = _lib.lib()
    names = header_functions()
    assert len(names) >= 15
    for name in names:
        assert hasattr(lib, name), f"{name} declared in sparseflow.h but not exported"
        assert name in _lib.EXPORTS, f"{name} has no ctypes signature in _lib.EXPORTS"
    assert set(_lib.EXPORTS) == set(names)


def test_version_and_empty_error():
    assert _lib.version() == 101
    assert isinstance(_lib.lib().sf_last_error(), bytes)


@pytest.mark.parametrize("thr", [1e-6, 0.0, 5e-7, 1e-3, 0.3, 1.0, 65504.0, 1e-9, -1.0, 2.0 ** -25])
def test_activity_cutoff_matches_fp16_semantics(thr):
    c = _lib.activity_cutoff(thr)
    # Oracle: |v| is active iff fp16(|v|) > fp16(thr).  Check around c.
    probes = np.array([c, np.nextafter(np.float32(c), np.float32(0)), np.nextafter(np.float32(c), np.float32(np.inf)),
                       0.0, 1e-9, 1e-6, 1.0, 7e4], dtype=np.float32)
    with np.errstate(over="ignore"):
        want = np.abs(probes.astype(np.float16)) > np.float16(thr)
    got = np.abs(probes) >= np.float32(c)
    np.testing.assert_array_equal(got, want)


def test_activity_cutoff_special_values():
    assert np.isnan(_lib.activity_cutoff(float("nan")))
    assert np.isnan(_lib.activity_cutoff(float("inf")))
    assert _lib.activity_cutoff(-0.5) == 0.0
    # f16(1e-6) = 17 * 2^-24; the boundary to 18 * 2^-24 ties to even (18).
    assert _lib.activity_cutoff(1e-6) == np.float32(17.5 * 2.0 ** -24)


def test_words_per_pixel_and_sizes():
    assert [_lib.words_per_pixel(c) for c in (1, 3, 32, 33, 64, 65, 96, 128, 256, 512, 2048)] == \
        [1, 1, 1, 2, 2, 4, 4, 4, 8, 16, 64]
    L = _lib.lib()
    assert L.sf_prescan_bitmap_bytes(32, 64, 32, 32) == 32 * 1024 * 2 * 4
    chunk = _lib.chunk_pixels(32, 64, 32, 32)
    assert chunk in (64, 128, 256)
    assert L.sf_prescan_flags_bytes(32, 64, 32, 32) == 32 * (-(-1024 // chunk)) * 4
    d = _lib.conv_desc(32, 64, 32, 32, 64, 32, 32, 3, 1, 1, 0, 0)
    ws = _lib.conv2d_workspace_size(d)
    assert ws >= L.sf_prescan_bitmap_bytes(32, 64, 32, 32) + L.sf_prescan_flags_bytes(32, 64, 32, 32)
    assert ws % 256 == 0
    assert _lib.conv_lif_workspace_size(d, 4) == _lib.conv2d_workspace_size(
        _lib.conv_desc(128, 64, 32, 32, 64, 32, 32, 3, 1, 1, 0, 0))


def _status(fn, *args):
    return int(fn(*args))


def test_validation_rejects_bad_descriptors_without_touching_the_device():
    L = _lib.lib()
    dummy = ctypes.c_void_p(16)
    bad_pattern = _lib.conv_desc(1, 8, 8, 8, 8, 8, 8, 5, 1, 2, 0, 0)
    assert _status(L.sf_conv2d_sparse, ctypes.byref(bad_pattern), dummy, dummy, dummy, dummy, None, dummy, None) \
        == _lib.SF_ERR_UNSUPPORTED
    assert b"supported patterns" in L.sf_last_error()
    wrong_out = _lib.conv_desc(1, 8, 8, 8, 8, 7, 8, 3, 1, 1, 0, 0)
    assert _status(L.sf_conv2d_sparse, ctypes.byref(wrong_out), dummy, dummy, dummy, dummy, None, dummy, None) \
        == _lib.SF_ERR_INVALID
    bad_dtype = _lib.conv_desc(1, 8, 8, 8, 8, 8, 8, 3, 1, 1, 7, 0)
    assert _status(L.sf_conv2d_sparse, ctypes.byref(bad_dtype), dummy, dummy, dummy, dummy, None, dummy, None) \
        == _lib.SF_ERR_INVALID
    mixed = _lib.conv_desc(1, 8, 8, 8, 8, 8, 8, 3, 1, 1, 0, 1)  # f32 in -> f16 out
    assert _status(L.sf_conv2d_sparse, ctypes.byref(mixed), dummy, dummy, dummy, dummy, None, dummy, None) \
        == _lib.SF_ERR_UNSUPPORTED
    too_wide = _lib.conv_desc(1, 4096, 8, 8, 8, 8, 8, 3, 1, 1, 0, 0)
    assert _status(L.sf_conv2d_sparse, ctypes.byref(too_wide), dummy, dummy, dummy, dummy, None, dummy, None) \
        == _lib.SF_ERR_UNSUPPORTED
    ok = _lib.conv_desc(1, 8, 8, 8, 8, 8, 8, 3, 1, 1, 0, 0)
    assert _status(L.sf_conv2d_sparse, ctypes.byref(ok), None, dummy, dummy, dummy, None, dummy, None) \
        == _lib.SF_ERR_INVALID
    assert _status(L.sf_conv2d_forward, ctypes.byref(ok), dummy, dummy, None, 1e-6, dummy, 16, dummy, None) \
        == _lib.SF_ERR_WORKSPACE
    # Fused conv-LIF: stride 2 unsupported, T < 1 invalid.
    s2 = _lib.conv_desc(1, 8, 8, 8, 8, 4, 4, 3, 2, 1, 0, 0)
    lif = _lib.LifParams(2.0, 1.0, 0.0, 1, 1)
    assert _status(L.sf_conv_lif_forward, ctypes.byref(s2), 2, dummy, dummy, None, ctypes.byref(lif), 1e-6, None,
                   dummy, dummy, dummy, 1 << 20, None) == _lib.SF_ERR_UNSUPPORTED
    assert _status(L.sf_conv_lif_forward, ctypes.byref(ok), 0, dummy, dummy, None, ctypes.byref(lif), 1e-6, None,
                   dummy, dummy, dummy, 1 << 20, None) == _lib.SF_ERR_INVALID
    # Tiles: group size must be a power of two >= 16; kernel < stride rejected.
    assert _status(L.sf_prescan_tiles, dummy, 1, 8, 8, 8, 8, 8, 3, 1, 1, 8, 8, 12, None, None, None, dummy, None,
                   None) == _lib.SF_ERR_UNSUPPORTED
    assert _status(L.sf_prescan_tiles, dummy, 1, 8, 8, 8, 4, 4, 1, 2, 0, 8, 8, 16, None, None, None, dummy, None,
                   None) == _lib.SF_ERR_UNSUPPORTED


def test_zero_frames_is_a_noop():
    L = _lib.lib()
    empty = _lib.conv_desc(0, 8, 8, 8, 8, 8, 8, 3, 1, 1, 0, 0)
    assert _status(L.sf_conv2d_sparse, ctypes.byref(empty), None, None, None, None, None, None, None) == _lib.SF_OK
    assert _status(L.sf_prescan_pack, None, 0, 0, 8, 8, 8, 1e-6, None, None, None) == _lib.SF_OK


def test_linear_bmm_attention_sizes_and_validation():
    L = _lib.lib()
    # Row bitmap: ceil(k/32) words, rounded up to a multiple of 4 beyond two.
    assert L.sf_linear_bitmap_bytes(10, 20) == 10 * 1 * 4
    assert L.sf_linear_bitmap_bytes(10, 64) == 10 * 2 * 4
    assert L.sf_linear_bitmap_bytes(10, 65) == 10 * 4 * 4
    assert L.sf_linear_bitmap_bytes(10, 384) == 10 * 12 * 4
    assert L.sf_linear_flags_bytes(33) == 3 * 4
    assert L.sf_linear_workspace_size(0, 10) == 0
    assert L.sf_linear_workspace_size(10, 384) == 512 + 256
    p = ctypes.c_void_p(1)  # never dereferenced: every call below fails validation or has no work
    # c_out not a multiple of 4 -> unsupported; m = 0 -> nothing to do.
    assert L.sf_linear_sparse(p, p, p, 0, 8, 32, p, None, 6, p, 0, None) == _lib.SF_ERR_UNSUPPORTED
    assert L.sf_linear_sparse(p, p, p, 0, 0, 32, p, None, 8, p, 0, None) == _lib.SF_OK
    assert L.sf_linear_forward(p, 0, 8, 32, p, None, 8, 1e-6, p, 1, p, 0, None) == _lib.SF_ERR_WORKSPACE
    # MFMA linear: kp must be k rounded up to 32; k <= 8192.
    assert L.sf_linear_mfma(p, 0, 8, 40, p, p, 40, None, 8, 1e-6, p, 0, None) == _lib.SF_ERR_INVALID
    assert L.sf_linear_mfma(p, 0, 8, 9000, p, p, 9024, None, 8, 1e-6, p, 0, None) == _lib.SF_ERR_UNSUPPORTED
    assert L.sf_linear_mfma(p, 0, 0, 40, p, p, 64, None, 8, 1e-6, p, 0, None) == _lib.SF_OK
    assert L.sf_linear_mfma_bits(p, p, p, 0, 8, 40, p, p, 40, None, 8, 1e-6, p, 0, None) == _lib.SF_ERR_INVALID
    assert L.sf_linear_mfma_bits(p, p, p, 0, 8, 9000, p, p, 9024, None, 8, 1e-6, p, 0, None) == _lib.SF_ERR_UNSUPPORTED
    assert L.sf_linear_mfma_bits(None, p, p, 0, 8, 40, p, p, 64, None, 8, 1e-6, p, 0, None) == _lib.SF_ERR_INVALID
    assert L.sf_linear_mfma_bits(p, p, p, 0, 0, 40, p, p, 64, None, 8, 1e-6, p, 0, None) == _lib.SF_OK
    # The output leaves as 16-byte row pieces: c_out must be a multiple of 4
    # (rejected before any launch).
    for c_out in (1, 130):
        assert L.sf_linear_mfma(p, 0, 8, 40, p, p, 64, None, c_out, 1e-6, p, 0, None) == _lib.SF_ERR_UNSUPPORTED
        assert L.sf_linear_mfma_bits(p, p, p, 0, 8, 40, p, p, 64, None, c_out, 1e-6, p, 0, None) == _lib.SF_ERR_UNSUPPORTED
    # Batched matmul: B's 64-column block of k rows must fit 64 KB of LDS.
    assert L.sf_bmm_supported(252, 10) and not L.sf_bmm_supported(253, 10)
    assert L.sf_bmm_sparse(p, p, 0, 2, 4, 300, 8, 0, 1, 300, 1e-6, 1.0, p, 0, None) == _lib.SF_ERR_UNSUPPORTED
    assert L.sf_bmm_sparse(p, p, 0, 0, 4, 30, 8, 0, 8, 1, 1e-6, 1.0, p, 0, None) == _lib.SF_OK
    assert L.sf_bmm_sparse(p, p, 0, 2, 4, 30, 8, 0, -1, 1, 1e-6, 1.0, p, 0, None) == _lib.SF_ERR_INVALID
    # Fused attention: head_dim 16/32/64 and the declared lengths.
    assert L.sf_spike_attention_supported(196, 32) and not L.sf_spike_attention_supported(196, 48)
    assert not L.sf_spike_attention_supported(700, 64)
    for d, s in ((16, 1271), (32, 623), (64, 287)):
        assert L.sf_spike_attention_supported(s, d) and L.sf_spike_attention_supported(1, d)
        assert not L.sf_spike_attention_supported(s + 1, d) and not L.sf_spike_attention_supported(0, d)
    st = (ctypes.c_int64 * 3)(0, 0, 0)
    assert L.sf_spike_attention(p, p, p, 0, 2, 196, 12, 48, st, 0.2, 1e-6, p, st, 0, None) == _lib.SF_ERR_UNSUPPORTED
    assert L.sf_spike_attention(p, p, p, 0, 0, 196, 12, 32, st, 0.2, 1e-6, p, st, 0, None) == _lib.SF_OK
    assert L.sf_spike_attention(p, p, p, 0, 2, 196, 12, 32, None, 0.2, 1e-6, p, st, 0, None) == _lib.SF_ERR_INVALID


def test_fused_conv1x1_lif_validation_without_touching_the_device():
    L = _lib.lib()
    d = ctypes.c_void_p(16)
    lif = _lib.LifParams(2.0, 1.0, 0.0, 1, 1)
    ok = _lib.conv_desc(2, 64, 8, 8, 64, 8, 8, 1, 1, 0, 0, 0)
    k3 = _lib.conv_desc(2, 64, 8, 8, 64, 8, 8, 3, 1, 1, 0, 0)
    args = (d, d, d, d, None)  # bits, flags, x, wt, bias
    for fn, extra in ((L.sf_conv1x1_lif_sparse, None), (L.sf_conv1x1_lif_sparse_binres, d)):
        # 3x3 is not this entry's pattern; T < 1 and a NULL spikes pointer are invalid.
        assert _status(fn, ctypes.byref(k3), 2, *args, extra, ctypes.byref(lif), None, d, d, None, None, None) \
            == _lib.SF_ERR_UNSUPPORTED
        assert _status(fn, ctypes.byref(ok), 0, *args, extra, ctypes.byref(lif), None, d, d, None, None, None) \
            == _lib.SF_ERR_INVALID
        assert _status(fn, ctypes.byref(ok), 2, *args, extra, ctypes.byref(lif), None, None, d, None, None, None) \
            == _lib.SF_ERR_INVALID
        # out_bits and out_flags go together.
        assert _status(fn, ctypes.byref(ok), 2, *args, extra, ctypes.byref(lif), None, d, d, d, None, None) \
            == _lib.SF_ERR_INVALID
    # The binary-residual entry needs its residual map.
    assert _status(L.sf_conv1x1_lif_sparse_binres, ctypes.byref(ok), 2, *args, None, ctypes.byref(lif), None, d, d,
                   None, None, None) == _lib.SF_ERR_INVALID
    assert b"res_bits" in L.sf_last_error()


def test_noalloc_entry_point_refuses_oversized_bitmaps_on_the_host():
    # Returns SF_ERR_WORKSPACE from the size check, before any device call.
    L = _lib.lib()
    d = _lib.conv_desc(4096, 256, 56, 56, 64, 56, 56, 3, 1, 1, 0, 0)
    assert _lib.conv2d_workspace_size(d) > _lib.NOALLOC_SCRATCH_BYTES
    dummy = ctypes.c_void_p(16)
    rc = L.sf_conv2d_forward_noalloc(ctypes.byref(d), dummy, dummy, None, ctypes.c_float(1e-6), dummy, None)
    assert rc == _lib.SF_ERR_WORKSPACE
    assert b"scratch" in L.sf_last_error()
    # Bad descriptors are refused before the size check, as sf_conv2d_forward does.
    bad = _lib.conv_desc(1, 8, 8, 8, 8, 8, 8, 5, 1, 2, 0, 0)
    assert L.sf_conv2d_forward_noalloc(ctypes.byref(bad), dummy, dummy, None, ctypes.c_float(1e-6), dummy,
                                       None) == _lib.SF_ERR_UNSUPPORTED


def test_bitmap_layout_query_follows_the_stage2_choice():
    P, M = _lib.SF_BITMAP_PLANES, _lib.SF_BITMAP_PIXEL_MAJOR

    def q(n, ci, h, w, co, ho, wo, k, s, p):
        return _lib.conv2d_bitmap_layout(_lib.conv_desc(n, ci, h, w, co, ho, wo, k, s, p, 0, 0))

    # Pixel-tile 3x3 (layer1, layer2, the stride-2 layers) and the K-chunked
    # row kernel (layer3 at 14x14) read word planes.
    assert q(512, 64, 56, 56, 64, 56, 56, 3, 1, 1) == P
    assert q(512, 128, 28, 28, 128, 28, 28, 3, 1, 1) == P
    assert q(512, 256, 14, 14, 256, 14, 14, 3, 1, 1) == P
    assert q(512, 512, 14, 14, 512, 7, 7, 3, 2, 1) == P
    # The row-band kernel (32-wide frames, C_in <= 64), the matrix-core stem
    # and the 1x1 kernels read pixel-major words.
    assert q(32, 64, 32, 32, 64, 32, 32, 3, 1, 1) == M
    assert q(64, 3, 32, 32, 384, 32, 32, 3, 1, 1) == M
    assert q(512, 256, 56, 56, 64, 56, 56, 1, 1, 0) == M
    assert q(0, 64, 56, 56, 64, 56, 56, 3, 1, 1) == P  # no frames: still the shape's choice
    with pytest.raises(_lib.SparseFlowLibError):       # inconsistent output size
        q(4, 64, 56, 56, 64, 9, 9, 3, 1, 1)
    d = _lib.conv_desc(4, 64, 56, 56, 64, 9, 9, 3, 1, 1, 0, 0)
    assert _lib.lib().sf_conv2d_bitmap_layout(ctypes.byref(d)) == -_lib.SF_ERR_INVALID


def test_layout_entry_points_reject_unknown_layouts_before_launching():
    L = _lib.lib()
    d = _lib.conv_desc(2, 64, 8, 8, 64, 8, 8, 3, 1, 1, 0, 0)
    dummy = ctypes.c_void_p(16)
    assert L.sf_conv2d_sparse_layout(ctypes.byref(d), dummy, 7, dummy, dummy, dummy, None, dummy, None) == \
        _lib.SF_ERR_INVALID
    lif = _lib.LifParams(2.0, 1.0, 0.0, 1, 1)
    assert L.sf_lif_multistep_layout(dummy, None, 0, 2, 1, 64, 64, ctypes.byref(lif), None, dummy, 0, dummy, dummy,
                                     dummy, 5, None) == _lib.SF_ERR_INVALID
    d1 = _lib.conv_desc(2, 64, 8, 8, 64, 8, 8, 1, 1, 0, 0, 0)
    assert L.sf_conv1x1_lif_sparse_layout(ctypes.byref(d1), 2, dummy, dummy, dummy, dummy, None, None,
                                          ctypes.byref(lif), None, dummy, dummy, dummy, dummy, -1, None) == \
        _lib.SF_ERR_INVALID


def test_layout_requests_pick_planes_only_when_every_consumer_asks():
    from sparseflow_amd.Kernels.spike_map import PIXEL_MAJOR, PLANES, LayoutRequests

    r = LayoutRequests()
    assert r.layout == PIXEL_MAJOR                    # nobody asked yet
    r.note("conv2", PLANES)
    assert r.layout == PLANES
    r.note("pool", PIXEL_MAJOR)
    assert r.layout == PIXEL_MAJOR                    # one consumer reads pixel-major words
    r.note("pool", PLANES)
    assert r.layout == PLANES
    for i in range(40):                               # bounded: old consumers drop out
        r.note(("c", i), PLANES)
    assert r.layout == PLANES and len(r._wants) == LayoutRequests._MAX
    r.clear()
    assert r.layout == PIXEL_MAJOR


# ---- launch plans of the tile kernels ----------------------------------------

CUS = 256  # of the MI355X; assumed where there is no GPU


def _plan(n, c_in, h, w, c_out, s=1, lif=False):
    ho, wo = -(-h // s), -(-w // s)
    d = _lib.conv_desc(n, c_in, h, w, c_out, ho, wo, 3, s, 1, _lib.SF_F32, _lib.SF_F32)
    return _lib.conv2d_launch_plan(d, lif)


# One workgroup fills a CU's LDS, so workgroups past the CUs wait for a second
# round.  Wherever workgroups of 16 tiles fit the chip at once, the spread ones
# do too, and one tile less would not have fitted.
@pytest.mark.parametrize("c_in,size,lif", [(256, 14, False), (192, 28, False), (256, 8, False), (130, 17, False),
                                           (100, 16, False), (64, 20, False), (256, 14, True), (150, 28, True),
                                           (128, 14, True), (40, 28, True)])
def test_tiles_spread_within_one_round_of_cus(c_in, size, lif):
    rows = not lif and c_in > 128 and size in (14, 28)          # four- and two-row tiles
    streamed = not lif and c_in > 128 and not rows               # 64-pixel tiles over all frames
    co_group = 32 if lif or 64 < c_in <= 128 else 64
    for groups in list(range(1, 25)) + [40, 64]:
        for n in (1, 2, 3, 5, 8, 10, 16, 19, 32, 37, 48, 64, 96, 100, 128, 200, 256, 320):
            wg, nt, _ = _plan(n, c_in, size, size, groups * co_group, lif=lif)
            px = size * size
            tiles = n * (size // 2 if size == 28 else -(-size // 4)) if rows else \
                -(-n * px // 64) if streamed else n * -(-px // 64)
            assert 1 <= nt <= 16 and wg % groups == 0
            if groups * -(-tiles // 16) <= CUS:
                assert wg <= CUS, (n, groups)
                assert nt * (wg // groups) >= tiles, (n, groups)
                assert nt == 1 or groups * -(-tiles // (nt - 1)) > CUS, (n, groups)


# The kernels that stream their weights give every pass a workgroup of its own
# (spikes that come in bursts keep a workgroup for long: the CUs take the others
# as they come free); those with resident weights make passes.
def test_streamed_tiles_take_a_workgroup_per_pass():
    for n, groups in ((512, 4), (300, 4), (512, 8), (1024, 4), (2000, 1)):
        wg, nt, _ = _plan(n, 256, 14, 14, 64 * groups)                  # row tiles
        assert nt * (wg // groups) >= 4 * n > nt * (wg // groups - 1)
        wg, nt, _ = _plan(n, 256, 14, 14, 32 * groups, lif=True)        # fused LIF
        assert nt * (wg // groups) >= 4 * n > nt * (wg // groups - 1)
        wg, nt, _ = _plan(n, 256, 16, 16, 64 * groups)                  # flattened tiles
        assert nt * (wg // groups) >= 4 * n > nt * (wg // groups - 1)
        wg, nt, _ = _plan(n, 128, 16, 16, 32 * groups)                  # resident
        assert wg <= CUS
    assert _plan(300, 256, 14, 14, 256) == (4 * 120, 10, 1)             # two rounds, evenly
    assert _plan(90, 256, 28, 28, 512) == (8 * 79, 16, 1)               # three: full workgroups


# Past the threads that a launch holds they make passes too (bitmaps of more
# frames than their x would fit the card).
def test_launch_plan_very_many_tiles():
    for n, c_in, c_out, lif in ((1 << 26, 129, 4, False), (1 << 26, 129, 200, False), (1 << 26, 129, 4, True),
                                (1 << 26, 100, 4, False)):
        wg, nt, _ = _plan(n, c_in, 14, 14, c_out, lif=lif)
        assert 0 < wg <= 1 << 21 and nt == 16


def test_launch_plan_known_shapes():
    # six groups of 128 four-row tiles: three tiles each would be 6 x 43 = 258 workgroups
    assert _plan(32, 256, 14, 14, 384) == (6 * 32, 4, 1)
    assert _plan(128, 256, 14, 14, 192) == (3 * 74, 7, 1)
    assert _plan(16, 256, 14, 14, 384, lif=True) == (12 * 16, 4, 1)
    # four wavefronts to a tile: up to four tiles a workgroup, two where the
    # slices are of 32 channels
    for c_in, lif, upto in ((40, False, 4), (200, False, 4), (100, False, 2), (100, True, 4), (200, True, 0)):
        seen = {_plan(n, c_in, 16, 16, 64, lif=lif)[1:] for n in range(1, 400)}
        assert {w for t, w in seen if t <= upto} <= {4} and {w for t, w in seen if t > upto} == {1}
        assert {t for t, _ in seen} >= {1, 2, 3, 4, 5}
    # other kernels have no such plan
    d = _lib.conv_desc(4, 64, 8, 8, 64, 8, 8, 1, 1, 0, 0, 0)
    with pytest.raises(_lib.UnsupportedError):
        _lib.conv2d_launch_plan(d)


# ---- which Linear kernel a shape takes -----------------------------------------

F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16

# (m, k, c_out, dtype, offset of x past 16 bytes, the fastest of "tiles" (128 x
# 128), "wide" (384 columns) and "bitmap", by a quarter or more unless noted,
# binary x).
LINEAR_ROUTES = [
    # wide: the aligned shapes that fill its tiles, 16-bit and ragged x
    (50176, 1536, 384, F32, 0, "wide"), (50176, 384, 384, F32, 0, "wide"), (3136, 768, 1152, F32, 0, "wide"),
    (50176, 384, 384, F16, 0, "wide"), (8192, 512, 768, BF16, 0, "wide"), (50176, 1535, 384, F32, 0, "wide"),
    (1000, 383, 384, F32, 0, "wide"), (8192, 512, 768, F32, 4, "wide"), (701, 1790, 100, F16, 0, "wide"),
    (200, 1001, 12, F32, 0, "wide"), (34277, 742, 1456, F16, 0, "wide"),
    # tiles: columns past the next 384 that are not there, short k
    (65536, 132, 128, F32, 0, "tiles"), (56000, 132, 128, F16, 0, "tiles"), (65536, 164, 128, F16, 0, "tiles"),
    (65536, 512, 512, F32, 0, "tiles"), (100000, 128, 128, F32, 0, "tiles"), (65536, 129, 128, F32, 0, "tiles"),
    (40000, 384, 256, F32, 0, "tiles"), (112945, 64, 96, F16, 0, "tiles"),
    # bitmap: outputs from twice the input on, large or with columns to spare
    (50176, 384, 1536, F32, 0, "bitmap"), (32768, 512, 2048, F32, 0, "bitmap"), (65536, 160, 1280, F32, 0, "bitmap"),
    (65536, 128, 1536, F32, 0, "bitmap"), (58638, 192, 744, F32, 4, "bitmap"), (30000, 132, 772, F32, 0, "bitmap"),
    (66745, 68, 324, F32, 0, "bitmap"), (60774, 111, 320, F32, 0, "bitmap"), (31712, 157, 604, F32, 0, "bitmap"),
    (25088, 395, 1732, F32, 0, "bitmap"), (56000, 200, 772, F32, 0, "bitmap"),
    # direct although the output is wide: small calls
    (1000, 384, 1536, F32, 0, "wide"), (8192, 768, 2048, F16, 0, "wide"), (10000, 64, 256, F32, 0, "tiles"),
]


@pytest.mark.parametrize("case", LINEAR_ROUTES)
def test_linear_route(case):
    m, k, c_out, dtype, offset, want = case
    bits = _lib.linear_mfma_bits_pays(m, k, c_out, dtype, offset)
    tiles = _lib.linear_mfma_row_tiles(m, k, c_out, dtype, offset)
    assert tiles in (0, 4, 8, 13)
    assert ("bitmap" if bits else "wide" if tiles else "tiles") == want


# Every shape gets a kernel that takes it: W's rows within the 31-bit buffer
# offsets of the wide kernel, x's bitmap below 2^31 bytes.
def test_linear_route_limits():
    assert _lib.linear_mfma_row_tiles(300, 8192, 131072, F16) == 0
    assert _lib.linear_mfma_row_tiles(300, 8192, 131068, F16) > 0
    assert not _lib.linear_mfma_bits_pays(1 << 28, 40, 128, F16)
    assert _lib.linear_mfma_bits_pays((1 << 28) - 1, 40, 128, F16)
    for m, k, c in ((0, 64, 64), (64, 0, 64), (64, 64, 0)):
        assert _lib.linear_mfma_row_tiles(m, k, c, F32) == 0 and not _lib.linear_mfma_bits_pays(m, k, c, F32)
