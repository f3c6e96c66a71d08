// The codes of one packed word as fp16 magic pairs: the unpack step that every kernel reading 4..7-bit rows shares.
// Plain integer arithmetic, compiled for the host too (its test runs every code at every position).
//
// A packed word holds 8 codes n = nibble + 16 h (value k: nibble k % 4 of the low or, for k >= 4, the high nibbles of W's
// bytes; high bits h at bit (B - 4) k of the word's high field).  The half with bits 0x6400 | n is 1024 + n, the half
// 0x5400 | 16 n (n < 64) is 64 + n, both exact, so one fp16 add of the bias below leaves the signed code exactly.
//
// The pairs come in the order (0, 2) (1, 3) (4, 6) (5, 7): values k and k + 2 sit 16 bits apart in W, so a pair's two
// nibbles are in place for both halves at once, and the second two pairs take theirs at bits 4..7 (the 0x5400 form)
// without a shift.  One AND-OR merges a pair's high bits with the magic and one its nibbles: 11 instructions for the 8
// codes of a 5-bit word, 14 for a 6-bit word and 5 for a 4-bit word, where masking nibbles and high bits into code
// bytes and permuting those into halves takes 17, 20 and 7.  Every contraction over the values (K Q^T) and every index
// of them (the output dims of P V) uses the same order, pair_at.  The 7-bit words go by code bytes all the same: their three
// high bits leave the 0x5400 form no room and no pair's bits in place, so the AND-OR form takes as many instructions and
// more registers (T = 4 on K 7 / V 6 bits, 40,000 positions: 127.9 us over four layers, by bytes 126.3; T = 2 on 7 / 7:
// 123.3, by bytes 120.0; one token on 7 / 6 at 9,001: 55.1 and 54.6).
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#define QKV_HD __host__ __device__ __forceinline__
#else
#define QKV_HD inline
#endif

namespace qkv {

// value index of element e (0, 1) of pair i of a word
QKV_HD constexpr int pair_at(int i, int e) { return 4 * (i >> 1) + (i & 1) + 2 * e; }

// magic + offset of pairs 0, 1 and of pairs 2, 3: half(p[i]) - bias = code - 2^(B-1)
template <int B>
struct CodeBias {
    static constexpr float lo = (float) (1024 + (1 << (B - 1))), hi = (float) ((B == 7 ? 1024 : 64) + (1 << (B - 1))); // (7 bits: byte_pairs)
};
template <>
struct CodeBias<8> { // q8 bytes: signed q -> q + 128 in the 0x6400 form
    static constexpr float lo = 1152.f, hi = 1152.f;
};

// (x & m) | c in one instruction, named: given the masks as constants the compiler regroups the merges below into two
// ANDs and an OR each.  m in a scalar register (SC) or in a VGPR.
template <bool SC>
QKV_HD uint32_t and_or(uint32_t x, uint32_t m, uint32_t c) {
#ifdef __HIP_DEVICE_COMPILE__
    uint32_t r;
    if constexpr (SC) asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "s"(m), "v"(c));
    else asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "v"(m), "v"(c));
    return r;
#else
    return (x & m) | c;
#endif
}

// the code bytes lo (values 0..3) and hi (values 4..7) as magic pairs
QKV_HD void byte_pairs(uint32_t lo, uint32_t hi, uint32_t (&p)[4]) {
#ifdef __HIP_DEVICE_COMPILE__
    p[0] = __builtin_amdgcn_perm(lo, 0x64646464u, 0x00060004u);
    p[1] = __builtin_amdgcn_perm(lo, 0x64646464u, 0x00070005u);
    p[2] = __builtin_amdgcn_perm(hi, 0x64646464u, 0x00060004u);
    p[3] = __builtin_amdgcn_perm(hi, 0x64646464u, 0x00070005u);
#else
    p[0] = (lo & 0x00ff00ffu) | 0x64006400u;
    p[1] = ((lo >> 8) & 0x00ff00ffu) | 0x64006400u;
    p[2] = (hi & 0x00ff00ffu) | 0x64006400u;
    p[3] = ((hi >> 8) & 0x00ff00ffu) | 0x64006400u;
#endif
}
// the 3-bit fields 0..3 of x (field k at bit 3 k) moved to bits 4..6 of byte k
QKV_HD uint32_t spread3(uint32_t x) {
    x &= 0xfffu;
    x = (x | (x << 10)) & 0x003f003fu;
    x = (x | (x << 5)) & 0x07070707u;
    return x << 4;
}

// the four pairs of word W.  The word's high field is part idx of hd: B = 5 byte idx (0..3), B = 6 half idx (0, 1),
// B = 7 the low 24 bits (idx unused, the bits above them ignored)
// SC: the high bits' masks in scalar registers.  The three-per-CU kernels have a few of each kind to spare: with 6-bit
// sides (two masks more) all-scalar masks spill scalars into the tile loop (5 + 6 bits: 2% slower), and with 5-bit sides
// alone masks in VGPRs spill those (5 + 5 bits: 2% slower).  The 16- and 24-row kernels have no VGPR to spare (5 + 6 bits,
// T = 4, masks in VGPRs: two more spilled; eight short sequences 144.8 us over four layers, in scalars 137.9)
template <int B, bool SC = true>
QKV_HD void code_pairs(uint32_t W, uint32_t hd, int idx, uint32_t (&p)[4]) {
    if constexpr (B == 7) {
        byte_pairs((W & 0x0f0f0f0fu) | spread3(hd), ((W >> 4) & 0x0f0f0f0fu) | spread3(hd >> 12), p);
        return;
    }
    constexpr uint32_t M64 = 0x64006400u, M54 = 0x54005400u, N0 = 0x000f000fu, N4 = 0x00f000f0u;
    const uint32_t W8 = W >> 8;
    uint32_t t0 = M64, t1 = M64, t2 = M54, t3 = M54; // magic and the pairs' high bits in place
    if constexpr (B == 5) {
        // bit k of H to bit 4 (k = 0, 1), 8 (k = 4, 5), and 16 further for k + 2; the odd k one bit higher
        const uint32_t Y = ((hd >> (8 * idx)) & 0xffu) * 0x00040010u, Z = Y >> 1;
        t0 = and_or<SC>(Y, 0x00100010u, t0);
        t1 = and_or<SC>(Z, 0x00100010u, t1);
        t2 = and_or<SC>(Y, 0x01000100u, t2);
        t3 = and_or<SC>(Z, 0x01000100u, t3);
    } else if constexpr (B == 6) {
        // the field's upper part 4 bits (two values) ahead: value k + 2 sits 16 bits above value k
        if (idx == 0) {
            const uint32_t X = (hd & 0x0000ffffu) | ((hd << 12) & 0xffff0000u);
            t0 = and_or<SC>(X << 4, 0x00300030u, t0);
            t1 = and_or<SC>(X << 2, 0x00300030u, t1);
            t2 = and_or<SC>(X, 0x03000300u, t2);
            t3 = and_or<SC>(X >> 2, 0x03000300u, t3);
        } else { // the lower part taken 4 bits up instead: the upper half stays where it is
            const uint32_t X = (hd & 0xffff0000u) | ((hd >> 12) & 0x0000ffffu);
            t0 = and_or<SC>(X, 0x00300030u, t0);
            t1 = and_or<SC>(X >> 2, 0x00300030u, t1);
            t2 = and_or<SC>(X >> 4, 0x03000300u, t2);
            t3 = and_or<SC>(X >> 6, 0x03000300u, t3);
        }
    }
    p[0] = and_or<true>(W, N0, t0);
    p[1] = and_or<true>(W8, N0, t1);
    p[2] = and_or<true>(W, N4, t2);
    p[3] = and_or<true>(W8, N4, t3);
}

} // namespace qkv
