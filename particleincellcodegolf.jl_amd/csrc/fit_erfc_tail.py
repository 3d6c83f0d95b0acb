"""Generates erfc_tail.h: polynomials of erfc(x) on [3, 4], [4, 5] and [5, 6].

erf(x) = 1 - erfc(x) there, and erfc is below 2.3e-5, so erf(x) as the msun
algorithm rounds it is fixed by erfc to a small absolute error delta except
where 1 - erfc lies within delta of the middle of two doubles (those take the
whole algorithm; see gauss_edges.h).  The polynomials are Chebyshev
interpolants in u = x - (m + 1/2), computed in 60-digit decimals from erfc's
continued fraction erfc(x) = exp(-x^2)/sqrt(pi) * 1/(x + (1/2)/(x + 1/(x +
(3/2)/(x + ...)))), converted to powers of u and rounded to double.

    python fit_erfc_tail.py > erfc_tail.h
"""
from decimal import Decimal, getcontext

getcontext().prec = 60
PI = Decimal("3.14159265358979323846264338327950288419716939937510582097494459")
# degrees: interpolation errors below 1.1e-21 in erfc
DEGREE = {3: 19, 4: 17, 5: 15}


def erfc(x):
    f = Decimal(x)
    for k in range(400, 0, -1):
        f = x + Decimal(k) / 2 / f
    return (-x * x).exp() / PI.sqrt() / f


def cos(x):
    # Taylor series after halving; x in [0, pi]
    y, s, t, k = x / 64, Decimal(1), Decimal(1), 0
    while abs(t) > Decimal(10) ** -58:
        k += 2
        t = -t * y * y / (k * (k - 1))
        s += t
    for _ in range(6):
        s = 2 * s * s - 1
    return s


def fit(m, deg):
    n = deg + 1
    nodes = [cos(PI * (2 * i + 1) / (2 * n)) / 2 for i in range(n)]
    div = [erfc(Decimal(m) + Decimal("0.5") + u) for u in nodes]   # Newton's divided differences
    for k in range(1, n):
        for i in range(n - 1, k - 1, -1):
            div[i] = (div[i] - div[i - 1]) / (nodes[i] - nodes[i - k])
    c = [Decimal(0)] * n
    for i in range(n - 1, -1, -1):
        c = [(c[j - 1] if j else Decimal(0)) - nodes[i] * c[j] for j in range(n)]
        c[0] += div[i]
    err = Decimal(0)
    for i in range(401):
        u = Decimal(i) / 400 - Decimal("0.5")
        p = Decimal(0)
        for a in reversed(c):
            p = p * u + a
        err = max(err, abs(p - erfc(Decimal(m) + Decimal("0.5") + u)))
    return [float(a) for a in c], float(err)


def main():
    print("// erfc_tail.h -- GENERATED by fit_erfc_tail.py; do not edit.")
    print("// erfc(m + 1/2 + u), u in [-1/2, 1/2], in powers of u.")
    print("#pragma once")
    print("#include <hip/hip_runtime.h>\n")
    print("namespace pic {")
    for m, deg in DEGREE.items():
        c, err = fit(m, deg)
        print(f"// interpolation error {err:.1e}")
        print("template <typename T>")
        print(f"__host__ __device__ __forceinline__ T erfc_tail{m}(T u) {{")
        print(f"    T p = T({c[-1].hex()});")
        for a in reversed(c[:-1]):
            print(f"    p = __builtin_elementwise_fma(p, u, T({a.hex()}));")
        print("    return p;\n}")
    print("}  // namespace pic")


if __name__ == "__main__":
    main()
