"""CPU check of the fan-beam backprojection table (cmi_fan2d_bp_table, the plans' own): angles that
are quarter turns apart to within what FP32 holds get entries that are exact quarter turns, the
condition of the backprojection by quarter turns, however many digits the angles were written with."""
import numpy as np
import pytest

from curadon_amd import _lib


def _turned(t):
    A = len(t)
    f = t[:A // 4]
    for k in range(1, 4):
        x = (-f[:, 1], -f[:, 0], f[:, 1])[k - 1]
        y = (f[:, 0], -f[:, 1], -f[:, 0])[k - 1]
        q = t[k * (A // 4):(k + 1) * (A // 4)]
        for got, want in ((q[:, 0], x), (q[:, 1], y)):
            zero = (np.abs(got) < 1e-13) & (np.abs(want) < 1e-13)
            if not bool(((got == want) | zero).all()):
                return False
    return True


@pytest.mark.parametrize("A", [4, 180, 720, 4096])
@pytest.mark.parametrize("digits", [16, 12, 11, 10, 9])
def test_quarter_turns_of_rounded_angles(A, digits):
    # quarters that start on the same digits: rounding moves them by less than 1e-9
    q = np.linspace(0.0, np.pi / 2, A // 4, endpoint=False)
    ang = np.concatenate([q + k * np.pi / 2 for k in range(4)])
    ang = np.round(ang, digits)
    apart = np.abs(ang.reshape(4, -1) - ang[:A // 4] - np.arange(4)[:, None] * np.pi / 2)
    t = _lib.fan2d_bp_table(ang, np.full(A, 300.0), np.full(A, 450.0))
    exact = np.stack([-np.sin(ang), np.cos(ang)], axis=1)
    assert np.abs(t[:, :2] - exact).max() <= 2.0 ** -25 + 1.1e-9
    if apart.max() <= 1e-9:
        assert _turned(t)


def test_other_angles_keep_their_own():
    ang = np.linspace(0, 2 * np.pi, 64, endpoint=False)
    ang[40] += 1e-6                                        # not a quarter turn: every entry its own
    t = _lib.fan2d_bp_table(ang, np.full(64, 300.0), np.full(64, 450.0))
    assert np.array_equal(t[:, 0], (-np.sin(ang)).astype(np.float32))
    assert np.array_equal(t[:, 1], np.cos(ang).astype(np.float32))
    ang[40] -= 1e-6
    dso = np.full(64, 300.0)
    dso[7] = 301.0                                         # nor are distances equal
    t = _lib.fan2d_bp_table(ang, dso, np.full(64, 450.0))
    assert np.array_equal(t[:, 0], (-np.sin(ang)).astype(np.float32))
