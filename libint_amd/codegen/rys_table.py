"""Roots and weights of the Rys quadrature, tabulated for the device.

The core integrals of an ERI class with total angular momentum L are moments
F_m(T) = int_0^1 t^(2m) exp(-T t^2) dt, m <= L, and the n-point Gauss rule of
that weight in u = t^2 reproduces them exactly for n = L // 2 + 1 (H. F. King
and M. Dupuis, J. Comput. Phys. 21, 144 (1976)).  Nodes u_r(T) and weights
w_r(T) come from the discretised Stieltjes procedure (W. Gautschi, Orthogonal
Polynomials, 2004, section 2.2) on a Gauss-Legendre rule in t, in 80-bit
arithmetic, at the Chebyshev points of unit intervals of T; each is stored as
the polynomial in x = 2 (T - iv) - 1 that interpolates it there.  From T = NI
on the upper limit of the moments no longer matters at double precision and
u_r = h_r / T, w_r = g_r / sqrt(T), with the positive nodes and the weights of
the 2n-point Gauss-Hermite rule.
"""
from __future__ import annotations

import numpy as np

LD = np.longdouble
PI = LD('3.14159265358979323846264338327950288')
NI = 128      # unit intervals of T; interval NI holds (h_r, g_r)
ND = 12       # coefficients per polynomial
NRMAX = 7     # up to (ff|ff), L = 12


def _gauss_legendre01(n):
    x = np.polynomial.legendre.leggauss(n)[0].astype(LD)
    for _ in range(3):  # Newton in 80 bits on P_n
        p0, p1 = np.ones_like(x), x.copy()
        for k in range(2, n + 1):
            p0, p1 = p1, ((2 * k - 1) * x * p1 - (k - 1) * p0) / LD(k)
        d = n * (x * p1 - p0) / (x * x - 1)
        x = x - p1 / d
    p0, p1 = np.ones_like(x), x.copy()
    for k in range(2, n + 1):
        p0, p1 = p1, ((2 * k - 1) * x * p1 - (k - 1) * p0) / LD(k)
    d = n * (x * p1 - p0) / (x * x - 1)
    return (x + 1) / 2, 1 / ((1 - x * x) * d * d)


def _rule(u, w, n):
    """n-point Gauss rules (nodes, weights: shape (n, batch)) of the discrete measures w (batch, m) at the points u (m)."""
    batch = w.shape[0]
    norm = w.sum(1)
    a, b = np.zeros((n, batch), LD), np.zeros((n, batch), LD)
    p0, p1 = np.zeros_like(w), np.ones_like(w)
    prev = None
    for k in range(n):
        s = (w * p1 * p1).sum(1)
        a[k] = (w * p1 * p1 * u).sum(1) / s
        b[k] = norm if k == 0 else s / prev
        prev = s
        p0, p1 = p1, (u - a[k][:, None]) * p1 - (b[k][:, None] if k else 0) * p0
    J = np.zeros((batch, n, n))
    for k in range(n):
        J[:, k, k] = a[k].astype(float)
        if k:
            J[:, k, k - 1] = J[:, k - 1, k] = np.sqrt(b[k].astype(float))
    x = np.linalg.eigvalsh(J).T.astype(LD)
    for _ in range(4):
        q0, q1 = np.zeros_like(x), np.ones_like(x)
        d0, d1 = np.zeros_like(x), np.zeros_like(x)
        for k in range(n):
            bk = b[k] if k else 0
            q0, q1, d0, d1 = q1, (x - a[k]) * q1 - bk * q0, d1, q1 + (x - a[k]) * d1 - bk * d0
        x = x - q1 / d1
    # weights: beta_0 / sum of squared orthonormal polynomials
    s, q0, q1, h = np.zeros_like(x), np.zeros_like(x), np.ones_like(x), np.ones(batch, LD)
    for k in range(n):
        if k:
            h = h * b[k]
        s += q1 * q1 / h
        q0, q1 = q1, (x - a[k]) * q1 - (b[k] if k else 0) * q0
    return x, norm / s


_GL = None


def rys(T, n):
    """(u, w) of shape (n, len(T)) for the weights exp(-T t^2) dt on [0, 1]."""
    global _GL
    if _GL is None:
        _GL = _gauss_legendre01(128)
    t, g = _GL
    T = np.asarray(T, LD)
    return _rule(t * t, g * np.exp(-T[:, None] * t * t), n)


def hermite(n):
    """(h, g): squares of the positive nodes and the weights of the 2n-point Gauss-Hermite rule."""
    x, g = _gauss_legendre01(240)
    x = x * 14  # exp(-196) is far below 80-bit precision
    h, w = _rule(x * x, (g * 14 * np.exp(-x * x))[None], n)
    return h[:, 0], w[:, 0]


def table(n):
    """Coefficients [interval][root][u, w][degree] of the n-point rule, the last interval the asymptotic constants."""
    k = np.arange(ND)
    node = np.cos(PI * (2 * k + 1) / (2 * ND))
    T = (np.arange(NI)[:, None] + (node + 1) / 2).reshape(-1)
    u, w = rys(T, n)
    f = np.stack([u, w]).reshape(2, n, NI, ND)
    cheb = np.cos(PI * np.outer(k, 2 * k + 1) / (2 * ND)) * (np.where(k == 0, 1, 2).astype(LD) / ND)[:, None]
    c = np.einsum('jk,frik->frij', cheb, f)
    P = np.zeros((ND, ND), LD)  # T_j as polynomials in x
    P[0, 0] = P[1, 1] = 1
    for j in range(2, ND):
        P[j, 1:] = 2 * P[j - 1, :-1]
        P[j] -= P[j - 2]
    out = np.zeros((NI + 1, n, 2, ND), LD)
    out[:NI] = np.einsum('frij,jd->irfd', c, P)
    h, g = hermite(n)
    out[NI, :, 0, 0], out[NI, :, 1, 0] = h, g
    return out.astype(float)


def offset(n):
    """First double of the n-point rule's section in the concatenated table."""
    return sum((NI + 1) * m * 2 * ND for m in range(1, n))


def emit():
    """C++ source of the table: sections n = 1 .. NRMAX back to back."""
    out = ['// generated by libint_amd/codegen/rys_table.py - do not edit', 'extern const double l2g_rys_table[] = {']
    for n in range(1, NRMAX + 1):
        t = table(n).reshape(-1)
        out += [','.join(float(v).hex() for v in t[k:k + 2 * ND]) + ',' for k in range(0, t.size, 2 * ND)]
    out += ['};', f'extern const int l2g_rys_table_size = {offset(NRMAX + 1)};']
    return '\n'.join(out) + '\n'
