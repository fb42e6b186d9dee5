"""frexp, ldexp and the class tests have a device form of one instruction each (include/blackframe_math.h).
Against the bit forms that the host and the oracle use: every exponent with the mantissas at its ends and
random ones, subnormals of every width, zeros, infinities and NaN, scaled by exponents that leave the
result normal, subnormal (rounded once, to nearest even), zero or infinite. Kernel and bit forms are built
from one source (tests/device)."""
import ctypes as C
import subprocess
from pathlib import Path

import numpy as np
import pytest
import torch  # its HIP runtime is the one that the library has to find

LIBRARY = Path(__file__).resolve().parent / "device" / "libfloat_forms.so"


@pytest.fixture(scope="module")
def library():
    if not LIBRARY.exists():
        subprocess.run(["make", "-s", "-C", str(LIBRARY.parent)], check=True)
    return C.CDLL(str(LIBRARY))


def inputs():
    rng = np.random.default_rng(6)
    exponents = np.arange(256, dtype=np.uint32)
    mantissas = np.concatenate([[0, 1, 2, 3, 0x3FFFFF, 0x400000, 0x400001, 0x7FFFFE, 0x7FFFFF],
                                1 << np.arange(23), (1 << np.arange(23)) - 1, rng.integers(0, 1 << 23, size=200)])
    bits = (exponents[:, None] << 23 | mantissas.astype(np.uint32)[None, :]).reshape(-1)
    bits = np.concatenate([bits, bits | 0x80000000, rng.integers(0, 1 << 32, size=1 << 18, dtype=np.uint32)]).astype(np.uint32)
    bits = np.tile(bits, 4)
    n = rng.integers(-300, 301, size=bits.size).astype(np.int32)
    # a quarter lands among the subnormals, where the rounding is
    magnitude = (bits >> 23 & 0xFF).astype(np.int32)
    low = rng.uniform(size=bits.size) < 0.25
    n[low] = (-magnitude - rng.integers(-3, 26, size=bits.size))[low]
    n[:6] = [0, 1, -1, 1 << 20, -(1 << 20), 2 ** 31 - 1]
    return bits, n


def as_floats(bits):
    return np.ascontiguousarray(bits).view(np.float32)


def host_forms(library, bits, n):
    out = np.zeros((bits.size, 4), dtype=np.uint32)
    library.float_forms_host(bits.ctypes.data_as(C.c_void_p), n.ctypes.data_as(C.c_void_p), C.c_uint32(bits.size),
                             out.ctypes.data_as(C.c_void_p))
    return out


def test_bit_forms_are_those_of_numpy(library):
    bits, n = inputs()
    got = host_forms(library, bits, n)
    x = as_floats(bits)
    assert np.array_equal(got[:, 0], np.isnan(x) * 1 + np.isfinite(x) * 2)
    finite = np.isfinite(x)
    mantissa, exponent = np.frexp(x[finite])
    assert np.array_equal(as_floats(got[finite, 1]), mantissa) and np.array_equal(got[finite, 2].view(np.int32), exponent)
    with np.errstate(over="ignore", under="ignore"):
        scaled = np.ldexp(x[finite].astype(np.float64), np.clip(n[finite], -600, 600)).astype(np.float32)
    assert np.array_equal(got[finite, 3], scaled.view(np.uint32))


@pytest.mark.gpu
def test_device_forms_are_the_bit_forms(library):
    bits, n = inputs()
    want = host_forms(library, bits, n)
    d_bits, d_n = torch.from_numpy(bits.view(np.int32)).cuda(), torch.from_numpy(n).cuda()
    d_out = torch.zeros((bits.size, 4), dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    assert library.float_forms_device(C.c_void_p(d_bits.data_ptr()), C.c_void_p(d_n.data_ptr()), C.c_uint32(bits.size),
                                      C.c_void_p(d_out.data_ptr())) == 0
    torch.cuda.synchronize()
    got = d_out.cpu().numpy().view(np.uint32)
    nan = np.isnan(as_floats(bits))
    assert np.array_equal(got[:, 0], want[:, 0])
    assert np.array_equal(got[:, 2], want[:, 2])
    for column in (1, 3):  # a NaN's payload is nobody's
        assert np.array_equal(np.isnan(as_floats(got[:, column])), nan)
        differ = np.nonzero((got[:, column] != want[:, column]) & ~nan)[0]
        assert differ.size == 0, [(hex(bits[i]), int(n[i]), hex(got[i, column]), hex(want[i, column])) for i in differ[:4]]
