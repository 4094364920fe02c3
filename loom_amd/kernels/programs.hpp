// -*- C++ -*-
/// @file programs.hpp
/// @brief Integer and small floating-point kernels in Loom IR.
///
/// `fib` is the README kernel of the reference (README.md:133-151, the same
/// program as tests/programs.hpp:201-218): it must compile unchanged, so its
/// statements are the DSL text of that listing.  The other kernels exercise
/// each part of the op contract and of the block structure; their expected
/// results are closed forms checked by the tests (reference validators:
/// tests/programs.hpp:288-389).
#pragma once

#include <vm/core.hpp>
#include <vm/macros.hpp>
#include <vm/operators.hpp>

#include <cstdint>

namespace loom_amd::programs
{
// clang-format off

// Fibonacci number F(n) (README.md:133-151).
template <std::unsigned_integral T>
TKERNEL1(fib, n)
    TLE(cmp, n, 1),
    TCMOV(c, cmp, n, 1),
    IPJMP2(cmp, work, HALT),
    LABEL(work),
    TMOV(p, 0),
    TMOV(c, 1),
    TMOV(i, 2),
    LABEL(loop),
    TADD(t, p, c),
    TMOV(p, c),
    TMOV(c, t),
    TADD(i, i, 1),
    TLE(cmp, i, n),
    IPJMP2(cmp, HALT, loop)
TKERNEL_END1(c);

// Collatz total stopping time: number of x -> x/2 (even) or 3x+1 (odd) steps
// until x == 1; 0 for x <= 1.  A loop whose body branches on parity, so lanes
// of a wave diverge on every iteration and finish after very different trip
// counts.  The count leaves the kernel as a u32 register (a second register
// width next to the u64 state).
template <std::unsigned_integral T>
TKERNEL1(collatz, x)
    IMOV(cnt, 0),
    ILE(fin, x, 1),
    IPJMP2(fin, step, done),
    LABEL(step),
    IBAND(odd, x, 1),
    IPJMP2(odd, even, odd3),
    LABEL(even),
    IRSHFT(x, x, 1),
    JMP(next),
    LABEL(odd3),
    IMUL(x, x, 3),
    IADD(x, x, 1),
    LABEL(next),
    IADD(cnt, cnt, 1),
    IEQ(fin, x, 1),
    IPJMP2(fin, step, done),
    LABEL(done),
    MOV(VAR(std::uint32_t, steps), IVAR(cnt))
KERNEL_END(VAR(std::uint32_t, steps));

// a! for a <= 20 (u64), 1 for a <= 1: a loop counting down.
template <std::unsigned_integral T>
TKERNEL1(factorial, a)
    TLE(small, a, 1),
    TCMOV(r, small, 1, a),
    IPJMP2(small, init, HALT),
    LABEL(init),
    TSUB(k, a, 1),
    LABEL(body),
    TMUL(r, r, k),
    TSUB(k, k, 1),
    TEQ(z, k, 0),
    IPJMP2(z, body, HALT)
TKERNEL_END1(r);

// Four-way jump table: i in {0,1,2,3} -> {1,3,7,11}; other values halt at
// once (out-of-range ParmJump index -> HALT) and return i unchanged.
template <typename T>
KERNEL(jump4, IVAR(i))
    IPJMP4(i, c0, c1, c2, c3),
    LABEL(c0),
    IMOV(i, 1),
    JMP(HALT),
    LABEL(c1),
    IMOV(i, 3),
    JMP(HALT),
    LABEL(c2),
    IMOV(i, 7),
    JMP(HALT),
    LABEL(c3),
    IMOV(i, 11)
KERNEL_END(IVAR(i));

// A loop inside a loop, its body four ways (one of them straight back to the
// inner loop's head, one out of both loops) with a join: every shape of
// control flow that the other kernels leave out.
template <std::unsigned_integral T>
TKERNEL2(nested, a, b)
    IBAND(n, a, 15),
    IMOV(s, b),
    IMOV(c, 0),
    IEQ(f, n, 0),
    IPJMP2(f, outer, HALT),
    LABEL(outer),
    IBAND(m, s, 7),
    LABEL(inner),
    IEQ(f, m, 0),
    IPJMP2(f, work, tail),
    LABEL(work),
    IADD(c, c, 1),
    IBAND(k, s, 3),
    IPJMP4(k, add, mix, again, out),
    LABEL(add),
    IADD(s, s, n),
    IADD(s, s, 1),
    JMP(join),
    LABEL(mix),
    IMUL(s, s, 5),
    IADD(s, s, m),
    JMP(join),
    LABEL(again),
    IRSHFT(s, s, 1),
    ISUB(m, m, 1),
    JMP(inner),
    LABEL(out),
    IRSHFT(s, s, 2),
    IBAND(f, s, 16),
    IPJMP2(f, join, HALT),
    LABEL(join),
    ISUB(m, m, 1),
    JMP(inner),
    LABEL(tail),
    ISUB(n, n, 1),
    INEQ(f, n, 0),
    IPJMP2(f, HALT, outer)
TKERNEL_END2(s, c);

// A long START that goes four ways (one of them out), with registers it sets
// to literals, sets twice and leaves to later blocks.
template <std::unsigned_integral T>
TKERNEL2(started, a, b)
    IMOV(n, 3),
    IMOV(s, 7),
    IMOV(c, 0),
    IMOV(d, 1),
    ILSHFT(t, a, 13),
    IXOR(x, a, t),
    IRSHFT(t, x, 7),
    IXOR(x, x, t),
    ILSHFT(t, x, 17),
    IXOR(x, x, t),
    IMUL(y, b, 0x9E3779B9),
    IADD(y, y, x),
    IRSHFT(t, y, 11),
    IXOR(y, y, t),
    IMUL(y, y, 0x85EBCA6B),
    IRSHFT(t, y, 13),
    IXOR(y, y, t),
    ILSHFT(t, y, 3),
    IADD(y, y, t),
    IXOR(x, x, y),
    IRSHFT(t, x, 5),
    IADD(x, x, t),
    IADD(s, s, x),
    IMOV(d, 9),
    IBAND(k, y, 3),
    IPJMP4(k, spin, once, HALT, twice),
    LABEL(twice),
    IADD(n, n, 4),
    LABEL(spin),
    IMUL(s, s, 5),
    IADD(s, s, d),
    IADD(c, c, 1),
    ISUB(n, n, 1),
    IBAND(f, s, 64),
    ICMOV(n, f, 0, n),
    INEQ(f, n, 0),
    IPJMP2(f, once, spin),
    LABEL(once),
    IXOR(s, s, x),
    IADD(c, c, 100)
TKERNEL_END3(s, c, d);

// A long START with more words live after it than a pool may hold.
template <std::unsigned_integral T>
TKERNEL2(crowded, a, b)
    IBAND(n, a, 15),
    IMUL(r0, b, 2654435769),
    IXOR(r0, r0, a),
    IMUL(r1, r0, 2654435771),
    IXOR(r1, r1, a),
    IMUL(r2, r1, 2654435773),
    IXOR(r2, r2, a),
    IMUL(r3, r2, 2654435775),
    IXOR(r3, r3, a),
    IMUL(r4, r3, 2654435777),
    IXOR(r4, r4, a),
    IMUL(r5, r4, 2654435779),
    IXOR(r5, r5, a),
    IMUL(r6, r5, 2654435781),
    IXOR(r6, r6, a),
    IMUL(r7, r6, 2654435783),
    IXOR(r7, r7, a),
    IMUL(r8, r7, 2654435785),
    IXOR(r8, r8, a),
    IMUL(r9, r8, 2654435787),
    IXOR(r9, r9, a),
    IMUL(ra, r9, 2654435789),
    IXOR(ra, ra, a),
    IMUL(rb, ra, 2654435791),
    IXOR(rb, rb, a),
    LABEL(turn),
    IADD(r0, r0, r5),
    IADD(r1, r1, r6),
    IADD(r2, r2, r7),
    IADD(r3, r3, r8),
    IADD(r4, r4, r9),
    IADD(r5, r5, ra),
    IADD(r6, r6, rb),
    IADD(r7, r7, r0),
    IADD(r8, r8, r1),
    IADD(r9, r9, r2),
    IADD(ra, ra, r3),
    IADD(rb, rb, r4),
    ISUB(n, n, 1),
    IBAND(f, n, 15),
    IPJMP2(f, done, turn),
    LABEL(done),
    IXOR(r0, r0, r1),
    IXOR(r0, r0, r2),
    IXOR(r0, r0, r3),
    IXOR(r0, r0, r4),
    IXOR(r0, r0, r5),
    IXOR(r0, r0, r6),
    IXOR(r0, r0, r7),
    IXOR(r0, r0, r8),
    IXOR(r0, r0, r9),
    IXOR(r0, r0, ra),
    IXOR(r0, r0, rb)
TKERNEL_END2(r0, n);

// Integer op mix, straight-line: every binary integer operation of the
// contract on (a, b), folded into several outputs.
template <std::unsigned_integral T>
TKERNEL2(int_mix, a, b)
    TADD(s, a, b),
    TSUB(d, a, b),
    TMUL(m, a, b),
    TDIV(q, a, b),
    TMOD(r, a, b),
    IBAND(x1, a, b),
    IBOR(x2, a, b),
    IXOR(x3, a, b),
    IBNOT(x4, a),
    ILSHFT(l, a, b),
    IRSHFT(h, a, b),
    IMIN(mn, a, b),
    IMAX(mx, a, b),
    TNEG(ng, a),
    ILAND(la, a, b),
    ILOR(lo, a, b),
    ILNOT(ln, a),
    TLT(c1, a, b),
    TGE(c2, a, b),
    TNEQ(c3, a, b),
    ISCT4(sc, c1, 10, 0x20, 0b11, 4),
    IANDLT(p1, c2, a, b),
    IORGE(p2, c1, a, b),
    IXOR(x1, x1, x2),
    IXOR(x1, x1, x3),
    IXOR(x1, x1, x4),
    IADD(s, s, l),
    IADD(s, s, h),
    IADD(d, d, mn),
    IADD(d, d, mx),
    IADD(m, m, ng),
    IADD(q, q, r),
    IADD(la, la, lo),
    IADD(la, la, ln),
    IADD(la, la, c1),
    IADD(la, la, c2),
    IADD(la, la, c3),
    IADD(la, la, sc),
    IADD(la, la, p1),
    IADD(la, la, p2)
TKERNEL_END6(s, d, m, q, x1, la);

// Sine and cosine of x: the op contract's polynomials (the reference SIMD
// backends', simd.hpp:955-1100), valid on [-pi, pi].  Checked bit for bit
// against vectors evaluated in exact arithmetic from the reference's tables.
template <std::floating_point T>
TKERNEL1(sincos, x)
    TSIN(s, x),
    TCOS(c, x)
TKERNEL_END2(s, c);

// Square root and reciprocal square root, one of each per input: the
// correctly rounded results of the op contract over the whole input range
// (zeros, subnormals, infinities, NaN and negatives included).
template <std::floating_point T>
TKERNEL1(roots, x)
    TSQRT(s, x),
    TRSQRT(r, x)
TKERNEL_END2(s, r);

// Division by literals: powers of two (whose quotients the backend forms as
// products with the exact reciprocal) beside divisors that are not.
template <std::floating_point T>
TKERNEL1(literal_div, x)
    TDIV(q1, x, 0.5),
    TDIV(q2, x, 16777216),
    TDIV(q3, x, -0.125),
    TDIV(q4, x, 3),
    TDIV(q5, x, 0.1),
    TDIV(q6, 1, x)
TKERNEL_END6(q1, q2, q3, q4, q5, q6);

// Constant selection with indices inside and outside the constant list:
// sct(i, c0, ..., cN-1) is c_i for i < N and 0 otherwise (operators.hpp
// sct).  The backend reads a list of at least four 4-byte constants from a
// table in LDS and the others through compares and selects; this kernel has
// lists of both kinds.
template <std::floating_point T>
KERNEL(sct_range, IVAR(x))
    TSCT6(a, x, 1.5, -2.25, 3e3, 0.125, -7, 9.5),
    ISCT5(b, x, 7, 0xFFFF, 3, 0x12345678, 1),
    ISUB(y, x, 2),
    TSCT4(c, y, 0.5, 0.25, -1, 2),
    TSCT3(s3, x, 4, 5, 6)
KERNEL_END(TVAR(a), IVAR(b), TVAR(c), TVAR(s3));

// Float op mix, straight-line, exercising the floating-point contract:
// arithmetic, fused multiply-add/sub, sqrt/rsqrt, rounding, min/max,
// copysign, sin/cos polynomials, select, union register and conversions.
template <std::floating_point T>
TKERNEL2(fp_mix, x, y)
    TMUL(a, x, y),
    TADD(a, a, x),
    TDIV(b, x, y),
    TFMA(c, x, y, b),
    TFMS(d, x, y, a),
    TABS(g1, x),
    TSQRT(g1, g1),
    TRSQRT(g2, g1),
    TROUND(r1, b),
    TFLOOR(r2, b),
    TCEIL(r3, b),
    TTRUNC(r4, b),
    TADD(r1, r1, r2),
    TADD(r3, r3, r4),
    TMIN(mn, x, y),
    TMAX(mx, x, y),
    TCOPYSIGN(cs, x, y),
    TMUL(ang, x, 0.001),
    TSIN(sn, ang),
    TCOS(cn, ang),
    TLT(sel, x, y),
    TCMOV(pick, sel, mn, mx),
    TSCT3(k, sel, 0.5, 1.25, -3e2),
    TADD(a, a, c),
    TADD(a, a, d),
    TADD(b, b, g2),
    TADD(b, b, r1),
    TADD(b, b, r3),
    TADD(cs, cs, pick),
    TADD(cs, cs, k),
    TMUL(sn, sn, cn),
    MOV(IVAR(u), TVAR(x)),
    TMOV(sum, a),
    TADD(sum, sum, b)
KERNEL_END(TVAR(a), TVAR(b), TVAR(cs), TVAR(sn), IVAR(u), TVAR(sum));

// clang-format on
} // namespace loom_amd::programs
