// Division of right-hand sides and steppers in the IEEE precisions (single and
// double): the quotient x / y by a constant whole number y.
//
// An IEEE division is 11 instructions, one of them a reciprocal that holds the
// SIMD for 16 cycles, and two waits between them: 84 cycles of a lone wave for
// a double, 62 with four waves per SIMD.  Models divide by constants all the
// time (membrane capacitance, slopes, time constants; 6 in rk4's update).  For
// a whole y below the limit of divide_exact_below the quotient needs four
// instructions, 22 and 17 cycles:
//   q = x z,  r = x - y q,  q' = q + r z   with z = RN(1/y), then fixup(q').
// q is within 2 ulp of x / y, so r is a multiple of ulp(q) (y is whole) of
// magnitude under 3 y ulp(q): exact, down to the smallest subnormal.  The
// last step rounds q + (r/y)(1 + e), |e| <= u, once: wrong by 2 u ulp before
// the rounding, while x / y with y = D 2^f, D odd, is 1/(2 D) ulp or more away
// from the middle between two neighbours, so for D < 1/(8 u) it rounds as the
// exact quotient does.  The fixup instruction gives signed zeros, infinities
// and NaN as a division does.  Only in a subnormal quotient by an even y can
// x / y be the middle itself; it is then rounded to the neighbour nearer to
// zero, not to the even one (both half a unit, 2^-1075, away).
//
// Kernel times before and after: lactotroph (4 such divisions in a right-hand
// side), 65,536 members, dopri5, double, transient + warm-up + features
// 180.1 -> 164.0 ms; 1,000 members, rk4, single, 5.98 -> 4.85 ms; van der Pol,
// 4,096 members, rk4, double (2 in the update), 8.31 -> 7.43 ms.  The same
// bits but for those subnormal middles.
//
// Right-hand sides are written with "/": the program builder replaces the
// token by "*CLODE_DIV*" inside function bodies (same precedence, same
// associativity), and the operators below give every pair of types the value
// of "/": a pair of arithmetic types through divide(), any other through its own
// operator.  Which path a division takes is decided by the optimiser:
// a divisor that is not a constant there takes the ordinary division.
#ifndef CLODE_DIVIDE_H
#define CLODE_DIVIDE_H

namespace clode_div {

template <class T>
struct Real {
    static constexpr bool fast = false;
};
template <>
struct Real<double> {
    static constexpr bool fast = true;
    static constexpr double below = 0x1p48;
    static CM_FN bool power_of_two(double y) { return !(__builtin_bit_cast(unsigned long long, y) << 12); }
    static CM_FN double fma(double a, double b, double c) { return __builtin_fma(a, b, c); }
    static CM_FN double fixup(double q, double y, double x) { return __builtin_amdgcn_div_fixup(q, y, x); }
};
template <>
struct Real<float> {
    static constexpr bool fast = true;
    static constexpr float below = 0x1p19f;
    static CM_FN bool power_of_two(float y) { return !(__builtin_bit_cast(unsigned int, y) << 9); }
    static CM_FN float fma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
    static CM_FN float fixup(float q, float y, float x) { return __builtin_amdgcn_div_fixupf(q, y, x); }
};

// x / y for double and float; both forms are written out and one is dropped
// when the optimiser knows whether y is constant (no branch in between)
template <class T>
CM_FN T divide(T x, T y)
{
    typedef Real<T> R;
    const T z = (T)1 / y;
    const T q = x * z;
    const T f = R::fixup(R::fma(R::fma(-y, q, x), z, q), y, x);
    const T a = y < (T)0 ? -y : y;
    const bool whole = a < R::below && (T)(long long)(a < R::below ? a : (T)0) == a;
    const T plain = x / y;  // by a power of two: the compiler multiplies
    return __builtin_constant_p(y) && !__builtin_constant_p(x) && whole && !R::power_of_two(y) ? f : plain;
}

struct Tag {
};
template <class A>
struct Lhs {
    A a;
};

template <bool Fast>
struct Quotient {
    template <class A, class B>
    static constexpr CM_FN auto of(A a, B b) -> decltype(a / b) { return a / b; }
};
template <>
struct Quotient<true> {
    template <class A, class B>
    static constexpr CM_FN auto of(A a, B b) -> decltype(a / b)
    {
        typedef decltype(a / b) T;
        return __builtin_is_constant_evaluated() ? a / b : divide<T>((T)a, (T)b);
    }
};

template <class A>
constexpr CM_FN Lhs<A> operator*(A a, Tag)
{
    return Lhs<A>{a};
}
template <class A, class B>
constexpr CM_FN auto operator*(Lhs<A> l, B b) -> decltype(l.a / b)
{
    // a type of the user's own keeps its operator, also where that gives a real
    return Quotient<Real<decltype(l.a / b)>::fast && __is_arithmetic(A) && __is_arithmetic(B)>::of(l.a, b);
}

}  // namespace clode_div

#define CLODE_DIV (clode_div::Tag{})

#endif  // CLODE_DIVIDE_H
