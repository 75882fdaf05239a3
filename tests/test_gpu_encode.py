"""The GPU encoder writes byte-identical streams to the reference encoder
(golden vectors) and to the oracle on larger seeded inputs."""

from __future__ import annotations

import numpy as np
import pytest

from conftest import GOLDEN_NAMES, load_golden
from gpu_helpers import bf16_tensor, heavy_tailed_bf16, uniform_bits
from oracle import se12_codec as o

pytestmark = pytest.mark.gpu


def _encode(bits: np.ndarray, device):
    from se12_amd.hip import encode_on_device

    dt = encode_on_device(bf16_tensor(bits, device))
    h = dt.to_host()
    s = h.streams
    t = dt.tile_grid[0] * dt.tile_grid[1]
    return {
        "sm": s.primary.sm.value, "ec": s.primary.ec.value, "esc": s.escape_handling.esc.value.reshape(t, 16),
        "fallback_bitmap": s.escape_handling.fallback.bitmap.value, "fallback_raw": s.escape_handling.fallback.raw.value,
        "codebook": np.array(h.metadata.codebook.exponents, dtype=np.uint8),
    }


def _assert_same(got, expect):
    for k in ("sm", "ec", "esc", "fallback_bitmap", "fallback_raw", "codebook"):
        assert np.array_equal(np.asarray(got[k]).reshape(-1), np.asarray(expect[k]).reshape(-1)), k


@pytest.mark.parametrize("name", GOLDEN_NAMES)
def test_encoder_matches_reference_bytes(gpu, name):
    g = load_golden(name)
    _assert_same(_encode(g["bits"].reshape(g["rows"], g["cols"]), gpu), g)


@pytest.mark.parametrize("rows,cols,kind", [(2304, 9216, "normal"), (300, 1000, "uniform"), (129, 4700, "heavy")])
def test_encoder_matches_oracle(gpu, rows, cols, kind):
    if kind == "normal":
        bits = o.normal_bf16(rows, cols, seed=0, std=0.02)
    elif kind == "uniform":
        bits = uniform_bits(rows, cols, seed=1)
    else:
        bits = heavy_tailed_bf16(rows, cols, seed=2)
    _assert_same(_encode(bits, gpu), o.encode(bits.reshape(-1), rows, cols))


def _streams(dt):
    return {"sm": dt.sm, "ec": dt.ec, "esc": dt.esc, "fallback_bitmap": dt.fallback_bitmap,
            "fallback_raw": dt.fallback_raw, "codebook": dt.codebook}


@pytest.mark.parametrize("rows,cols,kind", [
    (1, 1, "normal"), (1, 7, "uniform"), (16, 256, "heavy"), (15, 255, "uniform"), (17, 257, "heavy"),
    (1000, 8, "normal"), (1000, 9, "heavy"), (128, 256, "uniform"), (129, 256, "uniform"),     # 8 and 9 tiles: bitmap bytes
    (9000, 700, "mixed"),       # 1,689 tiles, more bitmap bytes than one step of a wave's rank count
])
def test_encoder_at_tile_and_bitmap_edges(gpu, rows, cols, kind):
    """Byte equality with the oracle for an aligned tensor and for one at an odd offset of its buffer, and of the two-call
    C interface on rows further apart than their length."""
    import ctypes

    import torch

    from se12_amd import _native as nat
    from se12_amd.hip import encode_on_device

    if kind == "normal":
        bits = o.normal_bf16(rows, cols, seed=rows, std=0.02)
    elif kind == "uniform":
        bits = uniform_bits(rows, cols, seed=rows)
    else:
        bits = heavy_tailed_bf16(rows, cols, seed=rows)
    if kind == "mixed":          # every third tile row full of escapes
        u = uniform_bits(rows, cols, seed=1)
        pick = (np.arange(rows) // 16) % 3 == 1
        bits = np.where(pick[:, None], u, bits)
    want = o.encode(bits.reshape(-1), rows, cols)
    _assert_same(_encode(bits, gpu), want)
    buf = torch.full((rows * cols + 9,), float("inf"), dtype=torch.bfloat16, device=gpu)
    w = buf[3:3 + rows * cols].view(rows, cols)
    w.copy_(bf16_tensor(bits, gpu))
    odd = _streams(encode_on_device(w))
    aligned = _streams(encode_on_device(bf16_tensor(bits, gpu)))
    for k, v in aligned.items():
        assert torch.equal(odd[k], v), k
    ld = cols + 5
    wide = torch.full((rows, ld), float("nan"), dtype=torch.bfloat16, device=gpu)
    wide[:, :cols] = w
    cb, n = (ctypes.c_uint8 * 15)(), ctypes.c_int64()
    nat.check(nat.lib().se12_encode_prepare(nat.ptr(wide), rows, cols, ld, cb, ctypes.byref(n), nat.stream_ptr()))
    assert tuple(cb) == tuple(aligned["codebook"].tolist()) and n.value * 4096 == aligned["fallback_raw"].numel()
    got = {k: torch.empty_like(v) for k, v in aligned.items()}
    out = nat.StreamsOut(sm_dev=got["sm"].data_ptr(), ec_dev=got["ec"].data_ptr(), esc_dev=got["esc"].data_ptr(),
                         fallback_bitmap_dev=got["fallback_bitmap"].data_ptr(),
                         fallback_raw_dev=got["fallback_raw"].data_ptr() if n.value else None, fallback_raw_tiles=n.value)
    total = ctypes.c_int64()
    nat.check(nat.lib().se12_encode(nat.ptr(wide), rows, cols, ld, cb, ctypes.byref(out), ctypes.byref(total),
                                    nat.stream_ptr()))
    assert total.value == n.value
    for k in got:
        if k != "codebook":
            assert torch.equal(got[k], aligned[k]), k


def test_nothing_is_pending_after_an_encode(gpu):
    """A matrix of fallback tiles packed on a side stream is complete when the
    call returns: another stream decodes it, and the weights' memory is given
    back, without a wait of the caller's."""
    import torch

    from se12_amd.hip import HipSe12WeightDecoder, encode_on_device

    g = torch.Generator(device=gpu)
    g.manual_seed(5)
    bits = torch.randint(-32768, 32768, (32768, 2304), generator=g, device=gpu, dtype=torch.int16)
    w = bits.clone().view(torch.bfloat16)
    torch.cuda.synchronize()
    side, other = torch.cuda.Stream(gpu), torch.cuda.Stream(gpu)
    with torch.cuda.stream(side):
        t = encode_on_device(w)
    assert side.query()
    assert t.fallback_raw.numel() == bits.numel()      # every tile is raw
    w.zero_()
    with torch.cuda.stream(other):
        got = HipSe12WeightDecoder().decode_to_device(t)
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), bits)


def test_streams_can_be_written_again_from_one_codebook(gpu):
    import ctypes

    import torch

    from se12_amd import _native as nat
    from se12_amd.hip import encode_on_device

    rows, cols = 100, 1000
    w = bf16_tensor(uniform_bits(rows, cols, seed=3), gpu)
    want = encode_on_device(w)
    lib, st = nat.lib(), nat.stream_ptr()
    cb_dev = torch.empty(15, dtype=torch.uint8, device=gpu)
    ws = torch.empty(lib.se12_encode_workspace(), dtype=torch.uint8, device=gpu)
    nat.check(lib.se12_encode_codebook(nat.ptr(w), rows, cols, cols, nat.ptr(cb_dev), nat.ptr(ws), ws.numel(), st))
    for _ in range(3):
        sm, ec, esc, bitmap = (torch.empty_like(t) for t in (want.sm, want.ec, want.esc, want.fallback_bitmap))
        out = nat.StreamsOut(sm_dev=sm.data_ptr(), ec_dev=ec.data_ptr(), esc_dev=esc.data_ptr(),
                             fallback_bitmap_dev=bitmap.data_ptr(), fallback_raw_dev=None, fallback_raw_tiles=0)
        result = torch.empty(lib.se12_encode_result_bytes(), dtype=torch.uint8, pin_memory=True)
        cb, n = (ctypes.c_uint8 * 15)(), ctypes.c_int64()
        nat.check(lib.se12_encode_streams(nat.ptr(w), rows, cols, cols, ctypes.byref(out), cb, ctypes.byref(n), nat.ptr(result),
                                          nat.ptr(ws), ws.numel(), st))
        assert n.value * 4096 == want.fallback_raw.numel() > 0 and tuple(cb) == want.codebook_host
        assert torch.equal(sm, want.sm) and torch.equal(bitmap, want.fallback_bitmap)


# rows of fewer columns than a load, than a group of 8 lanes' loads, than a wave's, and of several of a wave's; fewer rows
# than groups of lanes (segments) and more than there are of 8 or 64 lanes
@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 7), (40000, 5), (40000, 8), (9, 63), (300, 64), (300, 65), (5000, 511),
                                       (5000, 513), (3, 40000), (1, 70001), (17, 8192)])
def test_histogram_of_rows_with_gaps(gpu, rows, cols):
    """The codebook and the fallback count of rows further apart than their length, NaNs between them, are those of the rows
    alone."""
    import ctypes

    import torch

    from se12_amd import _native as nat
    from se12_amd.hip import encode_on_device

    g = torch.Generator(device=gpu)
    g.manual_seed(rows + cols)
    w = (torch.randn((rows, cols), generator=g, device=gpu) * 10.0 ** torch.randint(-4, 4, (rows, 1), generator=g,
                                                                                     device=gpu)).to(torch.bfloat16)
    want = encode_on_device(w)
    counts = torch.bincount((w.view(torch.int16).to(torch.int32).reshape(-1) >> 7) & 0xFF, minlength=256)
    order = sorted(range(256), key=lambda e: (-int(counts[e]), -e))
    assert want.codebook_host == tuple(order[:15])
    wide = torch.full((rows, cols + 3), float("nan"), dtype=torch.bfloat16, device=gpu)
    wide[:, :cols] = w
    cb, n = (ctypes.c_uint8 * 15)(), ctypes.c_int64()
    nat.check(nat.lib().se12_encode_prepare(nat.ptr(wide), rows, cols, cols + 3, cb, ctypes.byref(n), nat.stream_ptr()))
    assert tuple(cb) == want.codebook_host and n.value * 4096 == want.fallback_raw.numel()
