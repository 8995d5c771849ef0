"""Triangle multiplication parity on the GPU.

Mirrors test/triangle-multiplication-outgoing.gpu.test.ts and
test/evoformer-triangle-incoming.gpu.test.ts: the f32 path against the
fixtures at mean < 1e-5 / max < 1e-4 and against the oracle at 1e-5 of the
largest value; output blocking reproduces the whole result exactly; the f16
path within 1e-2. Incoming has no committed fixture; it is held to the oracle
and to the transpose identity incoming(z) = T(outgoing(T(z))).
"""
import os

import numpy as np
import pytest

from oracle import ref
from afhip.reference import load_triangle_reference_bundle
from conftest import GOLDEN

pytestmark = pytest.mark.gpu

FIXTURES = ["openfold-triangle-small", "alphafold-short-9", "alphafold-single-sequence-59", "alphafold-a3m-59"]


@pytest.fixture(scope="module")
def dev():
    import torch

    from afhip import device

    device.open_device(0)
    return torch.device("cuda", 0)


def bundle(name):
    return load_triangle_reference_bundle(os.path.join(GOLDEN, name, "manifest.json"))


def rel_max(actual, expected):
    a = np.asarray(actual, np.float64).reshape(-1)
    e = np.asarray(expected, np.float64).reshape(-1)
    return float(np.abs(a - e).max() / max(np.abs(e).max(), 1e-30))


def gpu_class(direction):
    from afhip import triangle

    return triangle.TriangleMultiplicationOutgoingGpu if direction == "outgoing" \
        else triangle.TriangleMultiplicationIncomingGpu


@pytest.mark.parametrize("name", FIXTURES)
def test_outgoing_f32_matches_fixture(dev, name):
    b = bundle(name)
    res = gpu_class("outgoing")().run(b["input"], {"precision": "f32"})
    m = ref.error_metrics(res["output"], b["expected"])
    assert m["meanAbsoluteError"] < 1e-5 and m["maxAbsoluteError"] < 1e-4
    assert res["elapsedMilliseconds"] > 0 and res["memory"]["peakBytes"] > 0


@pytest.mark.parametrize("name", FIXTURES)
def test_outgoing_f16_matches_fixture(dev, name):
    # f16 operands with f32 accumulation against the official f32 capture:
    # within the north star's 1e-2 of the largest value.
    b = bundle(name)
    out = gpu_class("outgoing")().run(b["input"], {"precision": "f16"})["output"]
    assert rel_max(out, b["expected"]) <= 1e-2


@pytest.mark.parametrize("name", FIXTURES)
@pytest.mark.parametrize("direction", ["outgoing", "incoming"])
def test_f32_matches_oracle(dev, name, direction):
    inp = bundle(name)["input"]
    expect = ref.triangle(direction, inp["z"], inp["mask"], inp["weights"], inp["epsilon"])
    out = gpu_class(direction)().run(inp, {"precision": "f32"})["output"]
    assert rel_max(out, expect) <= 1e-5


@pytest.mark.parametrize("direction", ["outgoing", "incoming"])
@pytest.mark.parametrize("block_rows", [4, 2])
def test_blocking_is_bit_identical(dev, direction, block_rows):
    inp = bundle("alphafold-short-9")["input"]
    whole = gpu_class(direction)().run(inp, {"precision": "f32"})["output"]
    blocked = gpu_class(direction)().run(inp, {"precision": "f32", "blockRows": block_rows})["output"]
    assert np.array_equal(whole.view(np.uint32), blocked.view(np.uint32))


def test_incoming_is_transposed_outgoing(dev):
    inp = bundle("alphafold-short-9")["input"]
    t = dict(inp)
    t["z"] = np.ascontiguousarray(inp["z"].transpose(1, 0, 2))
    t["mask"] = np.ascontiguousarray(inp["mask"].T)
    incoming = gpu_class("incoming")().run(inp, {"precision": "f32"})["output"].reshape(inp["z"].shape)
    via = gpu_class("outgoing")().run(t, {"precision": "f32"})["output"].reshape(inp["z"].shape).transpose(1, 0, 2)
    assert rel_max(incoming, via) <= 1e-6


@pytest.mark.parametrize("name", FIXTURES)
@pytest.mark.parametrize("direction", ["outgoing", "incoming"])
def test_f16_within_1e2(dev, name, direction):
    b = bundle(name)
    inp = b["input"]
    expect = ref.triangle(direction, inp["z"], inp["mask"], inp["weights"], inp["epsilon"])
    out = gpu_class(direction)().run(inp, {"precision": "f16"})["output"]
    m = ref.error_metrics(out, expect)
    assert m["meanAbsoluteError"] < 1e-3 and m["maxAbsoluteError"] < 1e-2
    if direction == "outgoing":
        m = ref.error_metrics(out, b["expected"])
        assert m["meanAbsoluteError"] < 1e-3 and m["maxAbsoluteError"] < 1e-2


@pytest.mark.parametrize("direction", ["outgoing", "incoming"])
@pytest.mark.parametrize("length,cz,ch", [(64, 128, 128), (37, 16, 24), (96, 128, 128), (100, 128, 128)])
def test_synthetic_against_oracle(dev, direction, length, cz, ch):
    inp = ref.deterministic_triangle_input(length, cz, ch, seed=length + cz)
    expect = ref.triangle(direction, inp["z"], inp["mask"], inp["weights"], inp["epsilon"])
    out = gpu_class(direction)().run(inp, {"precision": "f32"})["output"]
    assert rel_max(out, expect) <= 1e-5
    out16 = gpu_class(direction)().run(inp, {"precision": "f16"})["output"]
    err = np.abs(out16.reshape(expect.shape) - expect)
    assert np.all(err <= 1e-2 * np.maximum(1.0, np.abs(expect)))


def test_f16_pair_input_and_residual(dev):
    import torch

    from afhip import triangle

    L, cz, ch = 48, 128, 128
    inp = ref.deterministic_triangle_input(L, cz, ch, seed=3)
    z16 = ref.round_f16(inp["z"])
    expect = ref.triangle("outgoing", z16, inp["mask"], inp["weights"])
    op = triangle.TriangleMultiplication(L, cz, ch, precision="f16", pair_dtype="f16", out_dtype="f32",
                                         residual=True)
    op.prepare(inp["weights"])
    base = torch.full((L, L, cz), 0.5, dtype=torch.float32, device=dev)
    out = op(torch.from_numpy(z16).half().to(dev), torch.from_numpy(inp["mask"]).to(dev), out=base)
    got = out.cpu().numpy() - 0.5
    assert np.all(np.abs(got - expect) <= 1e-2 * np.maximum(1.0, np.abs(expect)))


@pytest.mark.parametrize("direction", ["outgoing", "incoming"])
@pytest.mark.parametrize("length,shift", [(37, 0.0), (100, 6.0), (300, -3.0)])
def test_f16_pair_input_against_oracle(dev, direction, length, shift):
    """f16 z (the kernels that take z's rows into the MFMA as loaded, with
    the LayerNorm mean subtracted in the accumulator): ragged last tiles
    (37 * 37 pairs), several tiles a CU (300 * 300), and rows whose mean is
    far from zero, where a lost mean correction would show at once. At
    300 * 300 the expectation is the f32 path (itself held to the oracle at
    1e-5 above), which the oracle would take ~20 s to produce."""
    import torch

    from afhip import triangle

    cz = ch = 128
    inp = ref.deterministic_triangle_input(length, cz, ch, seed=length + 7)
    z16 = ref.round_f16(inp["z"] + np.float32(shift))
    if length <= 128:
        expect = ref.triangle(direction, z16, inp["mask"], inp["weights"])
    else:
        f32 = triangle.TriangleMultiplication(length, cz, ch, direction=direction, precision="f32")
        f32.prepare(inp["weights"])
        expect = f32(torch.from_numpy(z16).to(dev), torch.from_numpy(inp["mask"]).to(dev)).cpu().numpy()
    op = triangle.TriangleMultiplication(length, cz, ch, direction=direction, precision="f16", pair_dtype="f16",
                                         out_dtype="f32")
    op.prepare(inp["weights"])
    out = op(torch.from_numpy(z16).half().to(dev), torch.from_numpy(inp["mask"]).to(dev)).cpu().numpy()
    err = np.abs(out.reshape(expect.shape) - expect)
    assert np.all(err <= 1e-2 * np.maximum(1.0, np.abs(expect)))


def test_invalid_input_raises_range_error(dev):
    from afhip import _lib

    inp = dict(bundle("openfold-triangle-small")["input"])
    inp["z"] = inp["z"].reshape(-1)[1:]
    with pytest.raises(_lib.RangeError, match="z has"):
        gpu_class("outgoing")().run(inp)


@pytest.mark.parametrize("direction", ["outgoing", "incoming"])
@pytest.mark.parametrize("length,cz,ch,pair_dtype,out_dtype,residual,shift", [
    (1, 4, 8, "f32", "f32", False, 0), (8, 31, 33, "f32", "f32", True, 1), (9, 128, 256, "f16", "f32", False, 0),
    (33, 100, 72, "f32", "f16", True, 1), (23, 64, 224, "f16", "f32", True, 3), (90, 128, 128, "f32", "f32", False, 0),
    (1, 64, 65, "f32", "f32", False, 0), (8, 67, 97, "f32", "f32", True, 1)])
def test_f32_pair_kernels(dev, direction, length, cz, ch, pair_dtype, out_dtype, residual, shift):
    # f32 precision's projection and output kernels, over pairs of f16 from 64
    # channels on both sides and on the f32 MFMA below: ragged
    # tiles of 64 pairs, channels short of their 32-wide padding, one to four
    # column splits, z and the output off 16-byte alignment (shift elements),
    # f16 storage, the residual. The input LayerNorm's scales and the columns of
    # the weights it feeds carry factors of 1e-6 to 1e6 that cancel, as any
    # weight may. f32 out: the f32 bound; f16 out: half an ulp besides.
    import torch

    from afhip import triangle

    inp = ref.deterministic_triangle_input(length, cz, ch, seed=length + ch)
    w = {k: np.array(v, np.float64) for k, v in inp["weights"].items()}
    fc, fh = 10.0 ** ref.uniform(61, (cz,), -6, 6), 10.0 ** ref.uniform(62, (ch,), -6, 6)
    for name, factor in (("layerNormIn", fc), ("layerNormOut", fh)):
        w[name + "Weight"] *= factor
        w[name + "Bias"] *= factor
    for name in ("AP", "AG", "BP", "BG", "G"):
        w[f"linear{name}Weight"] /= fc
    w["linearZWeight"] /= fh
    w = {k: v.astype(np.float32) for k, v in w.items()}
    z = ref.round_f16(inp["z"])
    old = ref.round_f16(ref.normal(63, z.shape))
    expect = ref.triangle(direction, z, inp["mask"], w) + (old if residual else 0)
    op = triangle.TriangleMultiplication(length, cz, ch, direction=direction, pair_dtype=pair_dtype,
                                         out_dtype=out_dtype, residual=residual)
    op.prepare(w)
    tdt = {"f32": torch.float32, "f16": torch.float16}

    def place(a, dtype):
        flat = torch.zeros(a.size + shift, dtype=tdt[dtype], device=dev)
        flat[shift:] = torch.from_numpy(np.ascontiguousarray(a)).to(dev).reshape(-1)
        return flat[shift:].reshape(a.shape)

    mask = torch.from_numpy(np.ascontiguousarray(inp["mask"], np.float32)).to(dev)
    out = op(place(z, pair_dtype), mask, out=place(old, out_dtype)).float().cpu().numpy()
    assert np.abs(out - expect).max() <= (1e-5 if out_dtype == "f32" else 1e-5 + 2.0 ** -11) * np.abs(expect).max()


@pytest.mark.parametrize("direction", ["outgoing", "incoming"])
@pytest.mark.parametrize("length,ch,storage,block_rows", [
    (59, 128, "f32", 0), (128, 128, "f32", 0), (100, 256, "f32", 0), (128, 256, "f16", 0), (90, 256, "f32", 0),
    (59, 256, "f16", 7), (150, 128, "f32", 32)])
def test_f32_in_place_is_bit_identical(dev, direction, length, ch, storage, block_rows):
    # The pair stack runs the triangle with z as its output. Out of place, up to
    # four workgroups share a tile of 64 pairs and each reads all 128 channels of
    # its rows of z; in place one has to read them all before any of them is
    # stored, and at 256 hidden channels more workgroups than the chip holds at
    # once would be launched otherwise. The same arithmetic either way.
    import torch

    from afhip import triangle

    cz = 128
    inp = ref.deterministic_triangle_input(length, cz, ch, seed=length + ch)
    z = torch.from_numpy(ref.round_f16(inp["z"])).to(dev)
    z = z.half() if storage == "f16" else z
    mask = torch.from_numpy(np.ascontiguousarray(inp["mask"], np.float32)).to(dev)
    op = triangle.TriangleMultiplication(length, cz, ch, direction=direction, precision="f32", pair_dtype=storage,
                                         out_dtype=storage, residual=True, block_rows=block_rows)
    op.prepare(inp["weights"])
    expect = op(z, mask, out=z.clone())
    got = op(z, mask, out=z)
    assert torch.equal(got, expect)


@pytest.mark.parametrize("cz,ch", [(16, 16), (48, 48), (32, 128), (128, 32)])
def test_f32_keeps_every_bit_of_short_sums(dev, cz, ch):
    # Below 64 channels the products stay on the f32 MFMA. A contraction of
    # +-2^20 leaves its LayerNorm as +-1, so with one weight a row of linearZ and
    # open gates the outputs are those weights, all 24 bits of them; pairs of f16
    # hold one in four to 23 bits.
    import torch

    from afhip import triangle

    inp = ref.deterministic_triangle_input(1, cz, ch, seed=cz + ch)
    w = {k: np.zeros_like(np.asarray(v, np.float32)) for k, v in inp["weights"].items()}
    sign = np.where(np.arange(ch) % 2 == 0, 1, -1).astype(np.float32)
    v = np.float32(1) + (2 * np.floor(ref.uniform(cz, (cz,), 0, 2 ** 22)) + 1).astype(np.float32) * np.float32(2 ** -23)
    w["layerNormInWeight"] += 1
    w["layerNormOutWeight"] += 1
    w["linearAPBias"] += 2 ** 10 * sign
    w["linearBPBias"] += 2 ** 10
    for name in ("linearAGBias", "linearBGBias", "linearGBias"):
        w[name] += 200
    w["linearZWeight"][np.arange(cz), np.arange(cz) % ch] = v
    op = triangle.TriangleMultiplication(1, cz, ch)
    op.prepare(w)
    got = op(torch.from_numpy(inp["z"]).to(dev), torch.ones(1, 1, device=dev)).cpu().numpy().reshape(-1)
    assert np.array_equal(got, v * sign[np.arange(cz) % ch])


def test_f32_largest_weights(dev):
    # Weights of 1.6e38 in a gate, which they open or shut, and of 4.5e37 in
    # linearZ, whose channel is compared by itself. The f32 bound.
    import torch

    from afhip import triangle

    length, cz, ch = 9, 64, 64
    inp = ref.deterministic_triangle_input(length, cz, ch, seed=5)
    w = {k: np.array(v, np.float32) for k, v in inp["weights"].items()}
    w["linearAGWeight"][7, 0] = 1.6e38
    w["linearZWeight"][9] = 0
    w["linearZWeight"][9, 3] = 4.5e37
    mask = np.ascontiguousarray(inp["mask"], np.float32)
    expect = ref.triangle("outgoing", inp["z"], mask, w)
    op = triangle.TriangleMultiplication(length, cz, ch)
    op.prepare(w)
    got = op(torch.from_numpy(np.ascontiguousarray(inp["z"], np.float32)).to(dev), torch.from_numpy(mask).to(dev))
    got = got.cpu().numpy().reshape(expect.shape)
    assert np.isfinite(expect).all() and np.abs(expect[..., 9]).max() > 1e37
    assert rel_max(got[..., 9] / 1e30, expect[..., 9] / 1e30) <= 1e-5
    rest = np.arange(cz) != 9
    assert rel_max(got[..., rest], expect[..., rest]) <= 1e-5
