"""Sensitivities that a module marks as newly allocated are taken over by the signal, all others are copied."""
import functools

import numpy as np

import pymoto_amd as pm
from pymoto_amd.core import returns_new_arrays


class Fresh(pm.Module):
    def __call__(self, x):
        return 2.0 * x

    @returns_new_arrays
    def _sensitivity(self, dy):
        self.last = 2.0 * dy
        return self.last


class Overridden(Fresh):
    def _sensitivity(self, dy):
        return super()._sensitivity(dy)


def run(cls, sig):
    m = cls()
    out = m(sig)
    out.sensitivity = np.ones_like(out.state)
    m.sensitivity()
    return m


def test_marked_result_is_taken_over_and_added_to():
    x = pm.Signal("x", np.arange(4.0))
    m = run(Fresh, x)
    assert x.sensitivity is m.last
    m2 = run(Fresh, x)  # a second term adds in place and is not kept
    np.testing.assert_array_equal(x.sensitivity, 4.0)
    np.testing.assert_array_equal(m2.last, 2.0)


def test_override_and_slice_get_private_copies():
    x = pm.Signal("x", np.arange(4.0))
    m = run(Overridden, x)
    assert x.sensitivity is not m.last
    np.testing.assert_array_equal(x.sensitivity, 2.0)
    y = pm.Signal("y", np.arange(6.0))
    m = run(Fresh, y[1:4])
    m.last[:] = 7.0
    np.testing.assert_array_equal(y.sensitivity, [0.0, 2.0, 2.0, 2.0, 0.0, 0.0])
    z = pm.Signal("z", np.arange(4.0), sensitivity=np.zeros(4))
    m = run(Fresh, z)
    assert z.sensitivity is not m.last
    np.testing.assert_array_equal(z.sensitivity, 2.0)


def test_wrapper_of_a_marked_function_gets_private_copies():
    """functools.wraps copies a function's attributes: a wrapper that keeps what it returns is not marked by them."""
    kept = []

    def recorded(f):
        @functools.wraps(f)
        def wrapper(*args):
            kept.append(f(*args))
            return kept[-1]
        return wrapper

    class Recorded(Fresh):
        _sensitivity = recorded(Fresh._sensitivity)

    x = pm.Signal("x", np.arange(4.0))
    run(Recorded, x)
    run(Recorded, x)
    np.testing.assert_array_equal(x.sensitivity, 4.0)
    np.testing.assert_array_equal(kept[0], 2.0)
