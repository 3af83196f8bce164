#!/usr/bin/env python3
"""Generates constants.hip.h: every field constant the HIP kernels use, derived from p and r.

Fp (base field of BLS12-381 G1) is kept in registers as 13 signed limbs of 30 bits, Montgomery
radix R = 2^390 (fq.hip.h, the kernels), and as 14 limbs of 29 bits, radix 2^406 (fp.hip.h, the
element-wise operations and the host-side checks).  Fr (scalar field) is kept as 8 limbs of 32
bits, Montgomery radix 2^256.
Run: python3 gen_constants.py > constants.hip.h
"""

P = 0x1A0111EA397FE69A4B1BA7B6434BACD764774B84F38512BF6730D2A0F6B0F6241EABFFFEB153FFFFB9FEFFFFFFFFAAAB
R = 0x73EDA753299D7D483339D80809A1D80553BDA402FFFE5BFEFFFFFFFF00000001
# BLS12-381: curve y^2 = x^3 + 4; GLV endomorphism (x, y) -> (beta x, y) acts as lambda on G1
B = 4

FP_BITS, FP_N = 29, 14
FP_RBITS = FP_BITS * FP_N  # 406
FR_BITS, FR_N = 32, 8
FQ_BITS, FQ_N = 30, 13
FQ_RBITS = FQ_BITS * FQ_N  # 390


def limbs(v, bits, n):
    assert v < (1 << (bits * n))
    return [(v >> (bits * i)) & ((1 << bits) - 1) for i in range(n)]


def carr(name, vals, typ="uint32_t"):
    body = ", ".join("0x%08xu" % x for x in vals)
    return "static constexpr %s %s[%d] = {%s};" % (typ, name, len(vals), body)


def balanced(v, n=FQ_N, bits=FQ_BITS):
    """v as n digits of `bits` bits in [-2^(bits-1), 2^(bits-1)), the last one unbounded."""
    d = []
    for _ in range(n - 1):
        x = v & ((1 << bits) - 1)
        if x >> (bits - 1):
            x -= 1 << bits
        d.append(x)
        v = (v - x) >> bits
    return d + [v]


def centred(v):
    v %= P
    return v - P if v > P // 2 else v


def iarr(name, vals, typ="int32_t"):
    assert all(-(1 << 31) <= x < (1 << 31) for x in vals)
    return "static constexpr %s %s[%d] = {%s};" % (typ, name, len(vals), ", ".join("%d" % x for x in vals))


# The digit offsets of a product in the signed form (fq.hip.h): output digit k is taken as the
# low 30 bits of its column minus FQ_BETA[k], so it lies in [-BETA, 2^30 - BETA) with no carry
# to round, and the constant FQ_K0 added to the lowest column makes up for it:
#     K0 2^-390 = sum_k BETA[k] 2^(30k)  (mod p).
# Found as a short vector of the 14-dimensional lattice of such relations with K0 < 2^63,
# BETA[k] within 2^24.1 of 2^29 and BETA[12] < 2^16 (a value offset below p / 32); the relation
# itself is asserted here.
FQ_K0 = 6969937068335403541
FQ_BETA = [550457077, 529115271, 538425416, 540408362, 534947505, 530527195, 527739787, 553457329,
           541486612, 537384151, 545225655, 547666669, 37975]


def fq_constants():
    R = 1 << FQ_RBITS
    assert (FQ_K0 * pow(R, -1, P) - sum(b << (FQ_BITS * k) for k, b in enumerate(FQ_BETA))) % P == 0
    assert 0 < FQ_K0 < 1 << 63 and all(abs(b - (1 << 29)) < 1 << 25 for b in FQ_BETA[:12]) and FQ_BETA[12] < 1 << 16
    # -c p = -1 (mod 2^30) with the small c = p^-1 mod 2^30: with it as the Montgomery multiple a
    # quotient digit is the column's low 30 bits, no multiplication
    c = pow(P, -1, 1 << FQ_BITS)
    assert c < 1 << 18
    pt = balanced(-c * P, FQ_N + 1)
    assert pt[0] == -1
    out = ["// ---- Fp, signed form: 13 x 30-bit digits, Montgomery radix 2^390 ----",
           "static constexpr int FQ_N = %d;" % FQ_N,
           "static constexpr uint32_t FQ_MASK = 0x%08xu;" % ((1 << FQ_BITS) - 1),
           iarr("FQ_P", balanced(P)) + "  // p",
           iarr("FQ_PT", pt) + "  // -%d p: digit 0 is -1" % c,
           "// (-p^-1 mod 2^30) << 2: a low word times this, shifted right by 2, is the signed quotient digit",
           "static constexpr uint32_t FQ_PINV4 = 0x%08xu;" % (((-c) << 2) & 0xFFFFFFFF),
           "static constexpr int64_t FQ_K0 = %dll;" % FQ_K0,
           iarr("FQ_BETA", FQ_BETA) + "  // digit offsets of a product",
           iarr("FQ_ONE", balanced(centred(R))) + "  // R mod p",
           iarr("FQ_R2", balanced(centred(R * R))) + "  // R^2 mod p",
           iarr("FQ_R3", balanced(centred(R * R * R))) + "  // R^3 mod p"]
    beta = 0x1A0111EA397FE699EC02408663D4DE85AA0D857D89759AD4897D29650FB85F9B409427EB4F49FFFD8BFD00000000AAAC
    out += [iarr("FQ_GLV", balanced(centred(beta * R))) + "  // beta of the endomorphism (Montgomery)",
            iarr("FQ_GLV2", balanced(centred(beta * beta * R))) + "  // beta^2",
            iarr("FQ_4P", [((4 * P) >> (30 * i)) & ((1 << 30) - 1) for i in range(13)]) + "  // 4 p, non-negative digits",
            carr("FQ_FROM_FP", limbs(R % P, FP_BITS, FP_N)) + "  // 2^390 mod p: x 2^406 -> x 2^390",
            carr("FP_FROM_FQ", limbs(pow(2, 2 * FP_RBITS - FQ_RBITS, P), FP_BITS, FP_N)) + "  // 2^422 mod p: x 2^390 -> x 2^406",
            ""]
    return out


def main():
    out = []
    out.append("// Generated by gen_constants.py -- do not edit.")
    out.append("#pragma once")
    out.append("#include <stdint.h>")
    out.append("namespace fk20 {")
    out.append("")
    out.append("// ---- Fp: 14 x 29-bit limbs, Montgomery radix 2^406 ----")
    out.append("static constexpr int FP_N = %d;" % FP_N)
    out.append("static constexpr uint32_t FP_MASK = 0x%08xu;" % ((1 << FP_BITS) - 1))
    out.append(carr("FP_P", limbs(P, FP_BITS, FP_N)))
    out.append("static constexpr uint32_t FP_PINV = 0x%08xu;  // -p^-1 mod 2^29" % ((-pow(P, -1, 1 << FP_BITS)) % (1 << FP_BITS)))
    rm = (1 << FP_RBITS) % P
    out.append(carr("FP_R2", limbs(rm * rm % P, FP_BITS, FP_N)) + "  // R^2 mod p")
    out.append(carr("FP_ONE", limbs(rm, FP_BITS, FP_N)) + "  // R mod p")
    for k in (2, 4, 8, 16, 32, 64, 128):
        out.append(carr("FP_%dP" % k, limbs(k * P, FP_BITS, FP_N)) + "  // %d p" % k)
    # GLV endomorphism phi(x, y) = (beta x, y) acts on G1 as multiplication by
    # lambda = z^2 - 1 (z = -0xd201000000010000), with r = lambda^2 + lambda + 1.
    z = -0xD201000000010000
    lam = z * z - 1
    assert lam * lam + lam + 1 == R
    beta = 0x1A0111EA397FE699EC02408663D4DE85AA0D857D89759AD4897D29650FB85F9B409427EB4F49FFFD8BFD00000000AAAC
    assert pow(beta, 3, P) == 1 and beta != 1
    out.append("static constexpr uint64_t GLV_LAMBDA[2] = {0x%016xull, 0x%016xull};  // z^2 - 1"
               % (lam & (2**64 - 1), lam >> 64))
    out.append("")
    out += fq_constants()
    out.append("// p as 12 x 32-bit limbs (packed storage form)")
    out.append(carr("FP_P_PACKED", limbs(P, 32, 12)))
    out.append(carr("FP_HALF_PACKED", limbs((P - 1) // 2, 32, 12)) + "  // (p - 1) / 2: y above it is the larger root")
    out.append("// the 12 x 32-bit CIOS layout of the limb-layout probe (Montgomery radix 2^384)")
    out.append("static constexpr const uint32_t *FP32_P = FP_P_PACKED;")
    out.append("static constexpr uint32_t FP32_PINV = 0x%08xu;  // -p^-1 mod 2^32" % ((-pow(P, -1, 1 << 32)) % (1 << 32)))
    out.append("")
    out.append("// ---- Fr: 8 x 32-bit limbs, Montgomery radix 2^256 ----")
    out.append(carr("FR_R", limbs(R, 32, FR_N)))
    out.append("static constexpr uint32_t FR_RINV = 0x%08xu;  // -r^-1 mod 2^32" % ((-pow(R, -1, 1 << 32)) % (1 << 32)))
    rr = (1 << 256) % R
    out.append(carr("FR_R2", limbs(rr * rr % R, 32, FR_N)) + "  // 2^512 mod r")
    out.append(carr("FR_ONE", limbs(rr, 32, FR_N)) + "  // 2^256 mod r")
    out.append(carr("FR_RM2", limbs(R - 2, 32, FR_N)) + "  // r - 2 (Fermat inverse exponent)")
    # Fr of the transforms: 9 signed digits of 29 bits, radix 2^261
    rt = balanced(-R, 9, 29)
    assert rt[0] == -1
    out.append("// Fr of the transforms: 9 x 29-bit digits, Montgomery radix 2^261")
    out.append(iarr("FN_RT", rt) + "  // -r: digit 0 is -1")
    out.append(carr("FP_PM2", limbs(P - 2, 32, 12)) + "  // p - 2 (Fermat inverse exponent)")
    out.append("")
    out.append("}  // namespace fk20")
    print("\n".join(out))


if __name__ == "__main__":
    main()
