"""Coefficients of the short-argument form of tanh in sigmoid_or_tanh (wechat-tfcc_amd/csrc/lstm_sequence.hip):
tanh(v) = v + v^3 P(v^2) for |v| below T, P of degree 5 with the smallest relative error that such a polynomial has
(Lawson's reweighted least squares on nodes that crowd at the upper end).

Up to T the polynomial's roundings cost less (0.73 units in the last place at most) than those of the quotient that takes
over, which carries the error of an exponential (0.9 there, less beyond).  Prints the coefficients rounded to float, lowest power first, and the
largest relative error they leave.  Not used at build or run time: tests/test_tanh_fit.py runs fit() and compares what it
returns with the constants committed in the kernel source."""
import numpy as np

T, DEGREE = 0.65, 5


def fit():
    """The coefficients as float32, lowest power first, and the largest relative error they leave on (0, T]."""
    x = T * np.sin(np.linspace(1e-3, np.pi / 2, 4001))
    exact, s = np.tanh(x), x * x
    basis = np.stack([x * s ** (i + 1) / exact for i in range(DEGREE + 1)], 1)
    y = (exact - x) / exact
    lawson = np.ones_like(x) / len(x)
    for _ in range(4000):
        w = np.sqrt(lawson)
        c, *_ = np.linalg.lstsq(basis * w[:, None], y * w, rcond=None)
        lawson *= np.abs(basis @ c - y) + 1e-30
        lawson /= lawson.sum()
    c32 = c.astype(np.float32)
    x = np.linspace(1e-4, T, 200001)
    approx = x + x ** 3 * np.polyval(c32.astype(np.float64)[::-1], x * x)
    return c32, float(np.abs(approx / np.tanh(x) - 1).max())


def main():
    c32, worst = fit()
    print(", ".join("%.9ef" % x for x in c32))
    print("largest relative error with these coefficients: %.2e" % worst)


if __name__ == "__main__":
    main()
