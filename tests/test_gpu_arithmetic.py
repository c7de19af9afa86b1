"""The kernels' shortened FP32 operations against their correctly rounded
values, mantissa by mantissa on the device: the reciprocal of a root, the
reciprocal and the root of a number of at least 1 (all of their exponents,
zeros, infinities and NaN), and the quotients by the cell sizes and volumes of
the setups. Bit parity with the oracle rests on them, and a particle test
meets the critical mantissas (all ones) hardly ever."""
import numpy as np
import pytest

from picongpu_amd import abi, setups

pytestmark = pytest.mark.gpu


def test_shortened_operations_are_correctly_rounded():
    sts = [setups.thermal(), setups.kelvin_helmholtz(), setups.khi_growth_rate(), setups.laser_plasma(),
           setups.differentiable(), setups.two_stream()]
    sizes = set()
    for st in sts:
        cell = np.asarray(abi.constants_from_config(st.config()).cell[:3], np.float32)
        sizes.update(cell.tolist())
        sizes.add(float(cell[0] * cell[1] * cell[2]))
    # and what other boxes may have: the all-ones and smallest mantissas, powers of 2, a long cell
    sizes.update([float(np.nextafter(np.float32(2), np.float32(0))), 1.0, float(np.nextafter(np.float32(1), np.float32(2))),
                  4.0, 37.25])
    print(f"case arithmetic sweep, {len(sizes)} divisors", flush=True)
    got = abi.arithmetic_mismatches(sorted(sizes))
    assert got == [0, 0, 0, 0], dict(zip(("1/root", "1/x", "sqrt", "x/cell"), got))


def test_arithmetic_check_rejects_unusable_divisors():
    for bad in (0.0, -1.0, np.inf, np.nan):
        with pytest.raises(abi.PicError):
            abi.arithmetic_mismatches([1.5, bad])
