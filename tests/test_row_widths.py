"""Compress / restore over row widths and alignments at which the kernels'
row-dealing changes: one to a few columns, the octs per row at which a
workgroup takes more threads, whole and broken last octs, one row, row counts
around a group of eight, tensors that start between 16-byte boundaries, and
(GPU only) tensors long enough for four pieces per thread.  Bit for bit
against the oracles, with supplied and with generated noise."""
import numpy as np
import pytest
import torch

import exact_oracle as o
import exact_oracle_half as oh
from exact_amd import ops
from exact_amd.conf import config
from gpu_util import FixedNoise, bytes_equal

F32 = np.float32


def _shifted(array, backend, shift):
    """The array on the device, `shift` elements behind the start of its buffer."""
    flat = torch.from_numpy(array).reshape(-1)
    buffer = torch.zeros(flat.numel() + shift, dtype=flat.dtype)
    buffer[shift:] = flat
    return buffer.to(backend)[shift:].view(array.shape)


def _check(backend, N, G, bits, half, shift, supplied):
    rng = np.random.default_rng(N * 1031 + G * 17 + bits + half)
    x = (rng.standard_normal((N, G)) * 3).astype(np.float16 if half else F32)
    x[0] = x[0, 0]                                              # a constant row
    noise = rng.random((N, G), dtype=F32)
    config.activation_compression_bits = [bits]
    xt = _shifted(x, backend, shift)
    if supplied:
        config.noise_source = FixedNoise([_shifted(noise, backend, shift)])
    else:
        config.noise_source = None
        seed, offset = 0x1234567855, 8
        import exact_amd.cpp_extension.quantization as extq
        real, extq.next_philox = extq.next_philox, lambda device: (seed, offset)
        noise = o.philox_noise_rows(seed, offset, N, G)
    try:
        packed, qbits, scale, mn = ops.quantize_activation(xt, None)
    finally:
        if not supplied:
            extq.next_philox = real
    if half:
        wp, ws, wm = oh.quantize_activation(x, bits, noise)
        want = oh.unpack(wp, bits, ws, wm, N, G)
    else:
        wp, _, ws, wm = o.quantize_activation(x, bits, noise)[:4]
        want = o.dequantize_activation(wp, bits, ws, wm, (N, G))
    assert bytes_equal(packed, wp)
    restored = ops.dequantize_activation((packed, qbits, scale, mn), xt.shape).cpu().numpy()
    kind = np.uint16 if half else np.uint32
    ok = ~np.isnan(want)
    assert np.array_equal(restored.view(kind)[ok], want.view(kind)[ok])


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("bits", [1, 2, 4, 8])
@pytest.mark.parametrize("N,G", [(1, 1), (2, 1), (9, 2), (300, 7), (1, 9), (7, 15), (8, 33), (9, 64), (65, 99), (16, 301),
                                 (5, 511), (9, 512), (3, 513), (17, 520), (2, 639), (3, 641), (1, 1023), (9, 1024)])
def test_compress_restore_at_the_edges_of_the_row_widths(backend, N, G, bits, half):
    _check(backend, N, G, bits, half, shift=0, supplied=True)
    _check(backend, N, G, bits, half, shift=0, supplied=False)


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("N,G,shift", [(33, 256, 1), (33, 256, 3), (40, 100, 2), (21, 77, 1), (9, 1024, 5)])
def test_compress_restore_of_a_tensor_between_16_byte_boundaries(backend, N, G, shift, half):
    for supplied in (True, False):
        _check(backend, N, G, 2, half, shift, supplied)


@pytest.mark.gpu
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("N,G", [(60001, 301), (150013, 50), (45007, 602), (9001, 1000)])
def test_compress_restore_of_long_tensors(cuda, N, G, half):
    for bits in (1, 4):
        _check(cuda, N, G, bits, half, shift=0, supplied=False)
