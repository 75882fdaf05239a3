"""HIP decode-only kernel vs the oracle: bit-exact (int16 compare), as the
reference's GPU decode test asks (tests/test_spec_gpu_decode.py:75-113 in the
reference), on the golden vectors, edge cases, ragged shapes, forced fallback
tiles, escape-heavy data and the 2304x9216 benchmark shape."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import GOLDEN_NAMES, golden_as_encoding, load_golden
from gpu_helpers import bf16_tensor, escape_count_bf16, heavy_tailed_bf16, normal_case, to_device, uniform_bits
from oracle import se12_codec as o

pytestmark = pytest.mark.gpu


def _decode(enc, device) -> np.ndarray:
    from se12_amd.hip import HipSe12WeightDecoder

    dt = to_device(enc, device)
    out = HipSe12WeightDecoder().decode_to_device(dt)
    torch.cuda.synchronize()
    return out.view(torch.int16).cpu().numpy()


@pytest.mark.parametrize("name", GOLDEN_NAMES)
def test_decode_golden_vectors_bit_exact(gpu, name):
    g = load_golden(name)
    got = _decode(golden_as_encoding(g), gpu)
    assert got.shape == (g["rows"], g["cols"])
    assert np.array_equal(got.reshape(-1), g["decoded"])


def test_decode_uniform_random_bits(gpu):
    bits = uniform_bits(64, 512, seed=7)
    enc = o.encode(bits.reshape(-1), 64, 512)
    assert o.fallback_tile_count(enc) > 0
    assert np.array_equal(_decode(enc, gpu), bits)


@pytest.mark.parametrize("rows,cols", [(1, 1), (36, 1), (33, 300), (17, 257), (16, 4096), (160, 2560), (5, 1030)])
def test_decode_ragged_shapes(gpu, rows, cols):
    bits = heavy_tailed_bf16(rows, cols, seed=rows + cols)
    enc = o.encode(bits.reshape(-1), rows, cols)
    assert np.array_equal(_decode(enc, gpu), bits)


def test_decode_benchmark_shape_bit_exact(gpu):
    bits, enc = normal_case(2304, 9216, seed=0)
    got = _decode(enc, gpu)
    assert np.array_equal(got, bits)


def test_decode_escape_heavy(gpu):
    bits = heavy_tailed_bf16(512, 4608, seed=3)
    enc = o.encode(bits.reshape(-1), 512, 4608)
    codes = o.unpack_codes(enc["ec"])
    assert (codes == 15).sum() > 100
    assert np.array_equal(_decode(enc, gpu), bits)


def test_decode_rows_in_request_order(gpu):
    from se12_amd.hip import HipSe12WeightDecoder, RowIndices

    bits = uniform_bits(48, 512, seed=4)
    enc = o.encode(bits.reshape(-1), 48, 512)
    dt = to_device(enc, gpu)
    dec = HipSe12WeightDecoder()
    got = dec.decode_rows(dt, RowIndices(values=(5, 0, 47, 12, 5)))
    assert np.array_equal(got.bit_pattern, bits[[5, 0, 47, 12, 5], :].reshape(-1))
    with pytest.raises(IndexError):
        dec.decode_rows(dt, RowIndices(values=(48,)))
    # device indices out of range give rows of zeros
    out = dec.decode_rows_to_device(dt, torch.tensor([3, -1, 99], device=gpu))
    torch.cuda.synchronize()
    o_np = out.view(torch.int16).cpu().numpy()
    assert np.array_equal(o_np[0], bits[3])
    assert not o_np[1:].any()


def test_decode_rows_ragged_and_fallback(gpu):
    from se12_amd.hip import HipSe12WeightDecoder, RowIndices

    g = load_golden("mixed_48x768")
    enc = golden_as_encoding(g)
    bits = g["bits"].reshape(48, 768)
    rows = tuple(range(47, -1, -5))
    got = HipSe12WeightDecoder().decode_rows(to_device(enc, gpu), RowIndices(values=rows))
    assert np.array_equal(got.bit_pattern, bits[list(rows)].reshape(-1))


def test_decode_every_escape_count(gpu):
    """Tiles with 0..16 escapes (listed in the bind-time sidecar up to 8, more
    decoded to raw tiles at bind) and a fallback tile: bit-exact, whole matrix
    and row subsets."""
    from se12_amd.hip import HipSe12WeightDecoder, RowIndices

    bits, counts = escape_count_bf16(seed=11)
    enc = o.encode(bits.reshape(-1), 64, 1024)
    codes = o.unpack_codes(enc["ec"]).reshape(16, 4096)
    assert (codes == 15).sum(axis=1).tolist() == counts
    assert o.fallback_tile_count(enc) == sum(1 for n in counts if n > 16)
    assert np.array_equal(_decode(enc, gpu), bits)
    dt = to_device(enc, gpu)
    rows = [63, 0, 17, 31, 40, 15, 48]
    got = HipSe12WeightDecoder().decode_rows(dt, RowIndices(tuple(rows)))
    assert np.array_equal(got.bit_pattern, bits[rows].reshape(-1))



def test_bind_stats_count_the_raw_decoded_tiles(gpu):
    """se12_handle_bind_stats: the tiles holding 9..16 escapes (more than a
    side record lists, fewer than a fallback tile) are the ones bind decodes
    to raw BF16; the sidecar bytes are 64 per tile, the 1 KiB pair table and
    8 KiB per such tile. A raw-twin handle derives nothing."""
    from se12_amd.hip import RawBf16MatVecKernel, Se12MatVecKernel

    bits, counts = escape_count_bf16(seed=11)
    enc = o.encode(bits.reshape(-1), 64, 1024)
    st = Se12MatVecKernel(to_device(enc, gpu), max_batch=1).bind_stats()
    raw = sum(1 for n in counts if 8 < n <= 16)
    assert raw == 5
    assert st == {"raw_tiles": raw, "sidecar_bytes": 16 * 64 + 1024 + raw * 8192}
    import ctypes

    from se12_amd import _native as nat

    w = torch.from_numpy(bits.astype(np.int16)).to(gpu).view(torch.bfloat16)
    rk = RawBf16MatVecKernel(w, max_batch=1)
    a, b = ctypes.c_int64(-1), ctypes.c_int64(-1)
    nat.check(nat.lib().se12_handle_bind_stats(rk.handle.raw, ctypes.byref(a), ctypes.byref(b)))
    assert (a.value, b.value) == (0, 0)


@pytest.mark.parametrize("shapes", [
    [(33, 300)],
    [(2048, 2304), (1024, 2304), (1024, 2304)],   # q, k, v
    [(1, 1), (2304, 4096), (17, 257), (160, 2560)],  # one tile beside several per wave
])
def test_decode_group_equals_the_oracle(gpu, shapes):
    """Each matrix of a launch decodes with its own codebook, to its own output."""
    from se12_amd.hip import Se12MatVecKernel, decode_group

    want = [uniform_bits(r, c, seed=i) if i == 0 and r * c < 65536 else o.normal_bf16(r, c, seed=i, std=0.02 * 4.0 ** i)
            for i, (r, c) in enumerate(shapes)]
    ks = [Se12MatVecKernel(to_device(o.encode(b.reshape(-1), r, c), gpu)) for b, (r, c) in zip(want, shapes)]
    outs = [torch.full((r, c), float("nan"), dtype=torch.bfloat16, device=gpu) for r, c in shapes]
    decode_group(ks, outs)
    for b, out in zip(want, outs):
        assert np.array_equal(out.view(torch.int16).cpu().numpy().reshape(-1), b.reshape(-1))
    with pytest.raises(ValueError):
        decode_group(ks, outs[:-1])
    with pytest.raises(ValueError):
        decode_group(ks * 5, outs * 5)


@pytest.mark.parametrize("rows,cols,kind", [
    (1, 1, "normal"), (16, 15, "uniform"), (17, 256, "heavy"), (33, 257, "heavy"), (48, 1024, "heavy"),     # 1, 1, 1, 2, 4 K tiles
    (40, 1025, "uniform"), (64, 2304, "normal"), (64, 2304, "heavy"), (32, 1288, "uniform"),                # 5, 9, 9, 6
])
def test_decode_rows_equals_the_oracle_at_tile_edges(gpu, rows, cols, kind):
    """Every row (each position of a tile, escapes, tiles kept raw), repeated and out-of-range ones, plain and scaled."""
    from se12_amd.hip import Se12MatVecKernel

    bits = {"normal": lambda: o.normal_bf16(rows, cols, seed=3, std=0.02), "uniform": lambda: uniform_bits(rows, cols, seed=3),
            "heavy": lambda: heavy_tailed_bf16(rows, cols, seed=3)}[kind]()
    enc = o.encode(bits.reshape(-1), rows, cols)
    k = Se12MatVecKernel(to_device(enc, gpu))
    idx = torch.cat([torch.arange(rows), torch.tensor([rows - 1, 0, -1, rows, 2 ** 40])]).to(gpu)
    out = torch.empty((idx.numel(), cols), dtype=torch.bfloat16, device=gpu)
    got = k.decode_rows_into(idx, out).view(torch.int16).cpu().numpy()
    want = np.concatenate([bits, bits[[rows - 1, 0]], np.zeros((3, cols), dtype=bits.dtype)])
    assert np.array_equal(got, want.astype(np.int16))
    w = bf16_tensor(want, gpu)
    for scale in (48.0, 70.7107, -0.3):
        scaled = k.decode_rows_scaled_into(idx, torch.empty_like(out), scale)
        ref = w * torch.tensor(scale, dtype=torch.bfloat16, device=gpu)
        assert torch.equal(scaled.isnan(), ref.isnan())
        assert torch.equal(scaled.nan_to_num(), ref.nan_to_num())      # (0 == -0 in a row outside the matrix)
    with pytest.raises(Exception):
        k.decode_rows_scaled_into(idx, out, float("inf"))


@pytest.mark.parametrize("rows,cols,kind", [(1, 1, "tail"), (36, 300, "tail"), (48, 768, "uniform"), (17, 257, "uniform"),
                                            (2049, 1024, "tail"), (1, 214, "uniform"), (4096, 4104, "tail")])
def test_decode_from_the_streams_equals_decode_of_the_bound_matrix(gpu, rows, cols, kind):
    """Fallback tiles, tiles past the listed escapes, part tiles, more tiles than waves, bitmaps that end inside a byte; the
    unchecked repeat gives the same bits."""
    from se12_amd.hip import HipSe12WeightDecoder, Se12MatVecKernel, encode_on_device

    bits = uniform_bits(rows, cols, seed=rows) if kind == "uniform" else heavy_tailed_bf16(rows, cols, seed=cols)
    dt = encode_on_device(bf16_tensor(bits, gpu))
    dec = HipSe12WeightDecoder()
    first, again = dec.decode_to_device(dt), dec.decode_to_device(dt)
    bound = Se12MatVecKernel(dt, max_batch=1).decode_into(torch.empty((rows, cols), dtype=torch.bfloat16, device=gpu))
    for got in (first, again, bound):
        assert np.array_equal(got.view(torch.int16).cpu().numpy(), bits)


def test_decode_from_the_streams_refuses_what_bind_refuses(gpu):
    import dataclasses

    from se12_amd.hip import HipSe12WeightDecoder, encode_on_device

    dt = encode_on_device(bf16_tensor(uniform_bits(64, 512, seed=7), gpu))
    assert dt.fallback_raw.numel() > 4096
    dec = HipSe12WeightDecoder()
    with pytest.raises(Exception, match="fallback tiles"):
        dec.decode_to_device(dataclasses.replace(dt, fallback_raw=dt.fallback_raw[4096:].contiguous()))
    with pytest.raises(ValueError, match="codebook"):
        dec.decode_to_device(dataclasses.replace(dt, codebook_host=tuple(reversed(dt.codebook_host))))
    assert dec.decode_to_device(dt).shape == (64, 512)


def test_decoder_on_two_streams_and_two_threads(gpu):
    import threading

    from se12_amd.hip import HipSe12WeightDecoder, RowIndices, encode_on_device

    cases = [heavy_tailed_bf16(512, 1024 + 256 * i, seed=i) for i in range(4)]
    dec, bad = HipSe12WeightDecoder(), []

    def work(k):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for bits in cases[k::2] * 3:
                out = dec.decode_to_device(encode_on_device(bf16_tensor(bits, gpu)))
                s.synchronize()
                if not np.array_equal(out.view(torch.int16).cpu().numpy(), bits):
                    bad.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not bad
    dt = encode_on_device(bf16_tensor(cases[0], gpu))
    assert np.array_equal(dec.decode_to_device(dt).view(torch.int16).cpu().numpy(), cases[0])
    assert np.array_equal(dec.decode_rows(dt, RowIndices((3, 500))).bit_pattern.reshape(2, -1), cases[0][[3, 500]])


@pytest.mark.parametrize("scale", [48.0, -3.5, 1e-30, 2.0 ** -133, 1e38])
def test_scaled_lookup_gives_the_framework_product_of_every_weight(gpu, scale):
    """All 65,536 BF16 patterns, NaNs of every payload among them, and rows outside the matrix: the bits of the separate
    multiply."""
    from se12_amd.hip import Se12MatVecKernel, encode_on_device
    from se12_amd.runtime import CompressedEmbedding

    w = torch.arange(65536, device=gpu, dtype=torch.int32).to(torch.int16).view(256, 256).view(torch.bfloat16)
    k = Se12MatVecKernel(encode_on_device(w))
    ids = torch.arange(-1, 257, device=gpu)
    plain = k.decode_rows_into(ids, torch.empty((258, 256), dtype=torch.bfloat16, device=gpu))
    got = CompressedEmbedding(k, scale=scale)(ids)
    assert torch.equal(got.view(torch.int16), (plain * torch.tensor(scale, dtype=torch.bfloat16, device=gpu)).view(torch.int16))


@pytest.mark.parametrize("use", ["decode_to_device", "decode_rows"])
def test_copies_and_pickles_of_a_decoder_start_afresh(gpu, use):
    import copy
    import pickle

    from se12_amd.hip import HipSe12WeightDecoder, RowIndices, encode_on_device

    bits = heavy_tailed_bf16(64, 512, seed=1)
    dt = encode_on_device(bf16_tensor(bits, gpu))
    dec = HipSe12WeightDecoder()
    dec.decode_to_device(dt) if use == "decode_to_device" else dec.decode_rows(dt, RowIndices((1, 2)))
    small = len(pickle.dumps(HipSe12WeightDecoder()))
    assert len(pickle.dumps(dec)) == small                  # no streams travel with it
    for other in (copy.copy(dec), copy.deepcopy(dec), pickle.loads(pickle.dumps(dec))):
        assert other._known(dt) is None and other._lock is not dec._lock
        assert np.array_equal(other.decode_to_device(dt).view(torch.int16).cpu().numpy(), bits)
    assert dec._known(dt) is not None


@pytest.mark.parametrize("kind", ["normal", "heavy", "uniform"])
def test_a_matrix_decoded_again_is_bound(gpu, kind):
    """Decoded from its streams the first time and while a graph captures, from the binding's records after that."""
    from se12_amd.hip import HipSe12WeightDecoder, encode_on_device

    bits = {"normal": lambda: o.normal_bf16(300, 1100, seed=1, std=0.02), "heavy": lambda: heavy_tailed_bf16(300, 1100, seed=2),
            "uniform": lambda: uniform_bits(300, 1100, seed=3)}[kind]()
    dt = encode_on_device(bf16_tensor(bits, gpu))
    dec = HipSe12WeightDecoder()

    def check(out):
        torch.cuda.synchronize()
        assert np.array_equal(out.view(torch.int16).cpu().numpy(), bits)

    check(dec.decode_to_device(dt))
    assert dec._last.handle is None
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = dec.decode_to_device(dt)
    assert dec._last.handle is None
    for _ in range(2):
        out.zero_()
        g.replay()
        check(out)
    check(dec.decode_to_device(dt))
    handle = dec._last.handle
    assert handle is not None
    check(dec.decode_to_device(dt))
    side = torch.cuda.Stream(gpu)
    with torch.cuda.stream(side):
        again = dec.decode_to_device(dt)
    check(again)
    assert dec._last.handle is handle
    other = encode_on_device(bf16_tensor(np.ascontiguousarray(bits[:64]), gpu))
    assert dec.decode_to_device(other).shape == (64, 1100) and dec._last.handle is None


@pytest.mark.parametrize("rows,share", [(64032, 0.02), (64032, 0.5), (64032, 1.0), (480000, 0.3)])
def test_raw_tiles_of_a_matrix_of_many(gpu, rows, share):
    """36,018 tiles (36 per wave of the decode) and 270,000 (two turns per block of bind and of the raw copy), `share` of them
    raw at random: packed, decoded from the streams and from a binding, and looked up by row."""
    from se12_amd.hip import HipSe12WeightDecoder, Se12MatVecKernel, encode_on_device

    cols = 2304
    g = torch.Generator(device=gpu)
    g.manual_seed(int(100 * share))
    w = (torch.randn((rows, cols), generator=g, device=gpu) * 0.02).to(torch.bfloat16).view(torch.int16)
    raw = torch.rand((rows // 16, cols // 256), generator=g, device=gpu) < share
    mask = raw.repeat_interleave(16, 0).repeat_interleave(256, 1)
    w = torch.where(mask, torch.randint(-32768, 32768, (rows, cols), generator=g, device=gpu, dtype=torch.int16), w)
    dt = encode_on_device(w.view(torch.bfloat16))
    assert dt.fallback_raw.numel() >= 4096 * int(raw.sum())
    assert torch.equal(HipSe12WeightDecoder().decode_to_device(dt).view(torch.int16), w)
    k = Se12MatVecKernel(dt, max_batch=1)
    out = torch.empty((rows, cols), dtype=torch.bfloat16, device=gpu)
    assert torch.equal(k.decode_into(out).view(torch.int16), w)
    idx = torch.randint(0, rows, (500,), generator=g, device=gpu)
    assert torch.equal(k.decode_rows_into(idx, torch.empty((500, cols), dtype=torch.bfloat16, device=gpu)).view(torch.int16), w[idx])
