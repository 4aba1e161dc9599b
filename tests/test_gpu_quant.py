"""GPU parity of the block formats: dequantization (GGUF layout and the repacked backend layout)
bit-exact against the oracle, and the device encoders byte-exact against the oracle's."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import ALL_TYPES, TYPES, random_blocks

pytestmark = pytest.mark.gpu


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("name", list(ALL_TYPES))
def test_dequant_gguf_bit_exact(gpu, name):
    from smallmind_amd.quantization import dequantize
    qt = ALL_TYPES[name]
    be = O.BLOCK_ELEMS[qt]
    for seed, nblocks in [(1, 1), (2, 7), (3, 333)]:
        b = random_blocks(qt, nblocks, seed)
        n = nblocks * be
        ref = O.dequant(qt, b, n)
        got = dequantize(qt, _dev(b), n).cpu().numpy()
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), (name, seed)
    if be == 1:
        return
    # a ragged tail (last block partially used), as the reference loops handle it
    b = random_blocks(qt, 3, 9)
    n = 3 * be - 5
    assert np.array_equal(dequantize(qt, _dev(b), n).cpu().numpy().view(np.uint32),
                          O.dequant(qt, b, n).view(np.uint32))


def test_dequant_f16_all_patterns(gpu):
    from smallmind_amd.quantization import dequantize
    h = np.arange(65536, dtype=np.uint16)
    got = dequantize(O.F16, _dev(h.view(np.uint8)), 65536).cpu().numpy().view(np.uint32)
    assert np.array_equal(got, O.dequant(O.F16, h.view(np.uint8), 65536).view(np.uint32))


@pytest.mark.parametrize("name", list(ALL_TYPES))
@pytest.mark.parametrize("rows,cols", [(3, 256), (64, 2048), (17, 5632)])
def test_weight_to_float32_bit_exact_after_repack(gpu, name, rows, cols):
    """IWeightTensor.ToFloat32 of the repacked backend layout equals the reference decode of
    the original upload bytes, for random bytes in every field."""
    from smallmind_amd.quantization import GpuWeightTensor
    qt = ALL_TYPES[name]
    nb = rows * cols // O.BLOCK_ELEMS[qt]
    b = random_blocks(qt, nb, rows * 31 + cols)
    w = GpuWeightTensor(qt, rows, cols, b)
    got = w.to_float32().cpu().numpy().reshape(-1)
    ref = O.dequant(qt, b, rows * cols)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
    w.close()


@pytest.mark.parametrize("name", list(TYPES) + ["SMQ_Q8", "SMQ_Q4", "F16"])
def test_device_encoder_matches_oracle_bytes(gpu, name):
    from smallmind_amd.quantization import quantize
    qt = ALL_TYPES[name]
    rng = np.random.default_rng(qt)
    x = np.concatenate([rng.normal(0, 0.02, 256 * 40), rng.normal(0, 3, 256 * 8),
                        np.zeros(256), np.full(256, 1e-6), rng.uniform(-1, 1, 256)]).astype(np.float32)
    # exact ties for the rounding path
    x[:64] = (np.arange(64) - 32) * 0.5
    got = quantize(qt, _dev(x)).cpu().numpy()
    assert np.array_equal(got, O.quantize(qt, x))


@pytest.mark.parametrize("name", list(ALL_TYPES))
@pytest.mark.parametrize("nblocks", [1, 3, 65])
def test_codecs_at_any_alignment(gpu, name, nblocks):
    """Four elements per thread: results and bytes are those of the oracle for blocks at an odd address
    (encoded through the C entry point too), floats at one that is only a multiple of 4, and every
    length of the last group; encoders keep what lies beside their output."""
    import torch

    from smallmind_amd._lib import call
    from smallmind_amd.quantization import dequantize
    qt = ALL_TYPES[name]
    be, s = O.BLOCK_ELEMS[qt], torch.cuda.current_stream().cuda_stream
    b = random_blocks(qt, nblocks, nblocks)
    odd = _dev(b) if name == "F32" else _dev(np.concatenate([np.zeros(1, np.uint8), b]))[1:]
    out = torch.full((nblocks * be + 5,), 7.0, device="cuda")
    for n in {max(1, nblocks * be - k) for k in range(6)}:
        ref = O.dequant(qt, b, n)
        assert np.array_equal(dequantize(qt, odd, n).cpu().numpy().view(np.uint32), ref.view(np.uint32))
        out.fill_(7.0)
        call("smx_dequant", int(qt), odd.data_ptr(), n, out.data_ptr() + 4, s)
        assert np.array_equal(out.cpu().numpy()[1:1 + n].view(np.uint32), ref.view(np.uint32))
        assert bool((out[1 + n:] == 7.0).all()) and float(out[0]) == 7.0
    if name == "F32":
        return
    x = np.random.default_rng(nblocks).normal(0, 1, nblocks * be + 1).astype(np.float32)
    got, xd = torch.full((b.size + 2,), 0xA5, dtype=torch.uint8, device="cuda"), _dev(x)
    call("smx_quantize", int(qt), xd.data_ptr() + 4, nblocks * be, got.data_ptr() + 1, s)
    got = got.cpu().numpy()
    assert np.array_equal(got[1:-1], O.quantize(qt, x[1:])) and got[0] == got[-1] == 0xA5


@pytest.mark.parametrize("name", ["Q4_K", "Q8_0"])
def test_codecs_beyond_one_launch(gpu, name):
    """More elements than one launch takes (2^34 and a few blocks: four per thread, and a launch of more
    than 2^32 threads does not run them all, without an error): the blocks and floats at the start, at multiples of 2^32 elements and at the
    end are those of the same elements by themselves."""
    import torch

    from smallmind_amd.quantization import dequantize, quantize
    qt = ALL_TYPES[name]
    n, part = 2 ** 34 + 768, 1024
    if torch.cuda.mem_get_info()[0] < 160 * 2 ** 30:
        pytest.skip("needs 160 GiB of free device memory")
    at = [k * 2 ** 32 + d for k in range(4) for d in (0, 2 ** 32 - part)] + [n - part]
    x = torch.zeros(n, device="cuda")
    for i, e in enumerate(at):
        x[e:e + part] = torch.randn(part, device="cuda", generator=torch.Generator("cuda").manual_seed(i))
    blocks = quantize(qt, x)
    per = O.BLOCK_BYTES[qt], O.BLOCK_ELEMS[qt]
    few = [quantize(qt, x[e:e + part].clone()) for e in at]
    for e, b in zip(at, few):
        assert torch.equal(blocks[e // per[1] * per[0]:(e + part) // per[1] * per[0]], b), e
    del x
    y = dequantize(qt, blocks, n)
    for e, b in zip(at, few):
        assert torch.equal(y[e:e + part], dequantize(qt, b, part)), e
    del y, blocks
    torch.cuda.empty_cache()


def test_fill_normal_statistics(gpu):
    from smallmind_amd.quantization import fill_normal
    v = fill_normal(5, 1_000_001, 0.02).cpu().numpy().astype(np.float64)
    assert abs(v.mean()) < 1e-4 and abs(v.std() - 0.02) < 1e-4
    w = O.fill_normal(5, 1001, 0.02)
    assert np.allclose(fill_normal(5, 1001, 0.02).cpu().numpy(), w, rtol=1e-5, atol=1e-8)


def test_quantize_roundtrip_on_device(gpu):
    from smallmind_amd.quantization import dequantize, quantize
    rng = np.random.default_rng(0)
    v = rng.normal(0, 0.02, 4096).astype(np.float32)
    b = quantize(O.Q8_0, _dev(v))
    y = dequantize(O.Q8_0, b, 4096).cpu().numpy()
    assert np.abs(y - v).max() < np.abs(v).max() / 127
