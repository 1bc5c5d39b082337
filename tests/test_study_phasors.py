"""The studies' complex phasors hold what re +- 1j*im holds: signs of zeros
(the phase of a real value is 0 or pi by them), infinities and NaN."""
import warnings
from types import SimpleNamespace

import numpy as np
import pytest

from oidt_amd import variants

PARTS = np.array([0.0, -0.0, 1.5, -2.5, np.inf, -np.inf, np.nan], np.float32)


@pytest.mark.parametrize('scheme', ['tm', 'te', '3d'])
def test_phasors_equal_the_complex_expression(scheme):
    re, im = (a.reshape(7, 7, 1) for a in np.meshgrid(PARTS, PARTS, indexing='ij'))
    c = SimpleNamespace(scheme=scheme, study='scattering_loss', nx=7, ny=7)
    mon = SimpleNamespace(box=[(0, 7), (0, 7)])
    with warnings.catch_warnings():
        warnings.simplefilter('ignore', RuntimeWarning)
        got = variants._output(c, 'ez', mon, (re, im))
        z = 1j * im.astype(np.complex64)
        ref = (re + z if scheme == '3d' else re - z).astype(np.complex64)[:, :, 0]
    assert got.dtype == np.complex64 and got.shape == (7, 7)
    for x, y in ((got.real, ref.real), (got.imag, ref.imag)):
        assert np.array_equal(x, y, equal_nan=True)
        assert np.array_equal(np.signbit(x)[~np.isnan(x)], np.signbit(y)[~np.isnan(y)])
