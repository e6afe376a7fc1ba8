// Keccak-f[1600] and the FIPS 202 sponges (SHAKE-128, SHA3-256, SHA3-512),
// one state split across a pair of adjacent lanes: lane p = lane & 1 holds
// the low (p = 0) or high (p = 1) 32 bits of each of the 25 words.
//
// A 64-bit rotation by r then needs the partner's half, fetched with one DPP
// swap of adjacent lanes, and one v_alignbit: for 0 < r < 32 the new half is
// alignbit(own, partner, 32 - r) in both lanes, for r > 32 it is
// alignbit(partner, own, 64 - r).  With three-input XORs and chi in v_bitop3,
// a round is 119 VALU instructions per lane (122 instructions with the round
// constant's read and the loop), against 180 for a whole state in one lane, and a
// batch gets twice the waves.
//
// Round constants come from the rc(t) LFSR of FIPS 202 Algorithm 5, evaluated
// at compile time; the rho offsets of the (x, y) -> (y, 2x + 3y) walk of
// Algorithm 2 are the rotation operands of KF_ROUND.  Both lanes of a pair
// must execute every call together (the DPP swap reads the partner's
// register).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <utility>

namespace tmvp {
namespace keccak {

struct Tables {
    uint64_t rc[24];
};

constexpr int lfsr_bit(int t)
{
    int m = t % 255;
    if (m == 0) return 1;
    unsigned r = 1;
    for (int i = 0; i < m; i++) {
        r <<= 1;
        if (r & 0x100) r ^= 0x171;
    }
    return (int)(r & 1);
}

constexpr Tables make_tables()
{
    Tables T{};
    for (int ir = 0; ir < 24; ir++) {
        uint64_t rc = 0;
        for (int j = 0; j <= 6; j++)
            if (lfsr_bit(j + 7 * ir)) rc |= 1ull << ((1 << j) - 1);
        T.rc[ir] = rc;
    }
    return T;
}

constexpr Tables kT = make_tables();
static_assert(kT.rc[0] == 1ull, "rc(0)");

// The partner lane's value (DPP quad_perm [1, 0, 3, 2]).
__device__ __forceinline__ uint32_t partner(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xf, 0xf, false);
}

// A lane's place in its sponge: which half of every word it holds, and where
// the round constants' halves lie in LDS.
struct Half {
    int p;              // 0: the low 32 bits, 1: the high ones
    const uint32_t *rc; // fill_rc's table
    bool shared = false; // (a constant) several sponge waves share the SIMD: see f1600
    __device__ __forceinline__ operator int() const { return p; }
};

// The round constants as (low, high) dwords to LDS, from immediates (a copy of
// a constant table would put a memory latency before the first permutation).
// The caller synchronises before the first permutation.
constexpr int kRcDwords = 48;
template <int... Is> __device__ __forceinline__ void fill_rc_all(uint4 *t, std::integer_sequence<int, Is...>)
{
    ((t[Is] = make_uint4((uint32_t)kT.rc[2 * Is], (uint32_t)(kT.rc[2 * Is] >> 32), (uint32_t)kT.rc[2 * Is + 1],
                         (uint32_t)(kT.rc[2 * Is + 1] >> 32))),
     ...);
}
__device__ __forceinline__ void fill_rc(uint32_t (&t)[kRcDwords])
{
    fill_rc_all(reinterpret_cast<uint4 *>(t), std::make_integer_sequence<int, 12>{});
}

// The permutation, two rounds per loop iteration, as one block of assembly.
//
// What bounds it: a wave issues at most one instruction every four cycles,
// whatever its kind, and a KEM call keeps one sponge wave per SIMD, so a
// permutation's time is its instruction count (122 a round) times four cycles,
// if nothing stalls.  The compiler's code stalled twice: a loop whose
// eight-byte instructions happen to start at 4 mod 8 bytes (decided by
// whatever code comes before it) runs 15 % slower (595 against 519 cycles a
// round for the same instructions), and dependent pairs were scheduled next to
// each other (a result is ready after eight cycles; a DPP read must come at
// least two instructions after its register's write).  Here the loop starts
// on a cache line and holds only eight-byte instructions (or pairs of
// four-byte ones), and every operand is at least four instructions old.
// Cycles a round at one wave per SIMD: 502, against 605 for the compiled loop
// inside the one-launch KEM kernels.
//
// Several sponge waves on a SIMD: a SIMD takes a half-rate instruction (DPP,
// alignbit: 58 a round) every four cycles and a full-rate one (bitop3, xor)
// every two, from different waves at once.  Left alone, the oldest wave issues
// whenever it can and the others wait for its full-rate runs with a half-rate
// instruction at their front: two waves took 947 cycles a round, as if one
// after the other.  With `shared`, a wave raises its priority for its half-rate
// runs, so the waves fall into step, one wave's half-rate run under another's
// full-rate one: 623 cycles a round for two waves, 1123 for four (947 and
// 1813 without), 533 for a lone one (502), which therefore goes without.
//
// C: column parities; R = rotl(C, 1); A ^= C[x-1] ^ R[x+1]; B = rho and pi of A
// (word 0 stays in A); A = chi of B's rows, ^ the round constant, which is
// read from LDS at the top of the iteration.
#define KF_PAR3(C, I, J, K) "v_bitop3_b32 %[c" #C "], %[a" #I "], %[a" #J "], %[a" #K "] bitop3:0x96\n\t"
#define KF_PAR2(C, I, J) "v_bitop3_b32 %[c" #C "], %[c" #C "], %[a" #I "], %[a" #J "] bitop3:0x96\n\t"
#define KF_SWAP(D, V) "v_mov_b32_dpp %[" #D "], %[" #V "] quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
#define KF_R(X) "v_alignbit_b32 %[r" #X "], %[c" #X "], %[r" #X "], 31\n\t"
#define KF_ADD(I, C, R) "v_bitop3_b32 %[a" #I "], %[a" #I "], %[c" #C "], %[r" #R "] bitop3:0x96\n\t"
// b[D] holds the partner's half of a[I]; rotations by less / more than 32
#define KF_LO(D, I, N) "v_alignbit_b32 %[b" #D "], %[a" #I "], %[b" #D "], " #N "\n\t"
#define KF_HI(D, I, N) "v_alignbit_b32 %[b" #D "], %[b" #D "], %[a" #I "], " #N "\n\t"
// X ^ (~Y & Z)
#define KF_CHI(D, X, Y, Z) "v_bitop3_b32 %[a" #D "], %[" #X "], %[" #Y "], %[" #Z "] bitop3:0xd2\n\t"
#define KF_ROUND(RC, WAIT, HALF_RATE, FULL_RATE) \
    KF_PAR3(0, 0, 5, 10) KF_PAR3(1, 1, 6, 11) KF_PAR3(2, 2, 7, 12) KF_PAR3(3, 3, 8, 13) KF_PAR3(4, 4, 9, 14) \
    KF_PAR2(0, 15, 20) KF_PAR2(1, 16, 21) KF_PAR2(2, 17, 22) KF_PAR2(3, 18, 23) KF_PAR2(4, 19, 24) \
    HALF_RATE KF_SWAP(r0, c0) KF_SWAP(r1, c1) KF_SWAP(r2, c2) KF_SWAP(r3, c3) KF_SWAP(r4, c4) \
    KF_R(0) KF_R(1) KF_R(2) KF_R(3) KF_R(4) FULL_RATE \
    KF_ADD(0, 4, 1) KF_ADD(1, 0, 2) KF_ADD(2, 1, 3) KF_ADD(3, 2, 4) KF_ADD(4, 3, 0) \
    KF_ADD(5, 4, 1) KF_ADD(6, 0, 2) KF_ADD(7, 1, 3) KF_ADD(8, 2, 4) KF_ADD(9, 3, 0) \
    KF_ADD(10, 4, 1) KF_ADD(11, 0, 2) KF_ADD(12, 1, 3) KF_ADD(13, 2, 4) KF_ADD(14, 3, 0) \
    KF_ADD(15, 4, 1) KF_ADD(16, 0, 2) KF_ADD(17, 1, 3) KF_ADD(18, 2, 4) KF_ADD(19, 3, 0) \
    KF_ADD(20, 4, 1) KF_ADD(21, 0, 2) KF_ADD(22, 1, 3) KF_ADD(23, 2, 4) KF_ADD(24, 3, 0) \
    HALF_RATE \
    KF_SWAP(b10, a1) KF_SWAP(b20, a2) KF_SWAP(b5, a3) KF_SWAP(b15, a4) KF_SWAP(b16, a5) KF_SWAP(b1, a6) \
    KF_SWAP(b11, a7) KF_SWAP(b21, a8) KF_SWAP(b6, a9) KF_SWAP(b7, a10) KF_SWAP(b17, a11) KF_SWAP(b2, a12) \
    KF_SWAP(b12, a13) KF_SWAP(b22, a14) KF_SWAP(b23, a15) KF_SWAP(b8, a16) KF_SWAP(b18, a17) KF_SWAP(b3, a18) \
    KF_SWAP(b13, a19) KF_SWAP(b14, a20) KF_SWAP(b24, a21) KF_SWAP(b9, a22) KF_SWAP(b19, a23) KF_SWAP(b4, a24) \
    KF_LO(10, 1, 31) KF_HI(20, 2, 2) KF_LO(5, 3, 4) KF_LO(15, 4, 5) KF_HI(16, 5, 28) KF_HI(1, 6, 20) \
    KF_LO(11, 7, 26) KF_HI(21, 8, 9) KF_LO(6, 9, 12) KF_LO(7, 10, 29) KF_LO(17, 11, 22) KF_HI(2, 12, 21) \
    KF_LO(12, 13, 7) KF_HI(22, 14, 25) KF_HI(23, 15, 23) KF_HI(8, 16, 19) KF_LO(18, 17, 17) KF_LO(3, 18, 11) \
    KF_LO(13, 19, 24) KF_LO(14, 20, 14) KF_LO(24, 21, 30) KF_HI(9, 22, 3) KF_HI(19, 23, 8) KF_LO(4, 24, 18) \
    FULL_RATE \
    KF_CHI(3, b3, b4, a0) KF_CHI(4, b4, a0, b1) KF_CHI(0, a0, b1, b2) KF_CHI(1, b1, b2, b3) KF_CHI(2, b2, b3, b4) \
    KF_CHI(5, b5, b6, b7) KF_CHI(6, b6, b7, b8) KF_CHI(7, b7, b8, b9) KF_CHI(8, b8, b9, b5) KF_CHI(9, b9, b5, b6) \
    KF_CHI(10, b10, b11, b12) KF_CHI(11, b11, b12, b13) KF_CHI(12, b12, b13, b14) KF_CHI(13, b13, b14, b10) KF_CHI(14, b14, b10, b11) \
    KF_CHI(15, b15, b16, b17) KF_CHI(16, b16, b17, b18) KF_CHI(17, b17, b18, b19) KF_CHI(18, b18, b19, b15) KF_CHI(19, b19, b15, b16) \
    KF_CHI(20, b20, b21, b22) KF_CHI(21, b21, b22, b23) KF_CHI(22, b22, b23, b24) KF_CHI(23, b23, b24, b20) KF_CHI(24, b24, b20, b21) \
    WAIT "v_xor_b32_e64 %[a0], %[a0], %[" #RC "]\n\t"
#define KF_IO(i) [a##i] "+v"(A[i])
#define KF_B(i) [b##i] "=&v"(B[i])
#define KF_T(t) [t] "=&v"(t)

#define KF_PERMUTE(HALF_RATE, FULL_RATE) \
    "s_movk_i32 %[n], 11\n\t" \
    ".p2align 6\n" \
    "keccak%=:\n\t" \
    "ds_read_b32 %[k0], %[at]\n\t" \
    "ds_read_b32 %[k1], %[at] offset:8\n\t" \
    KF_ROUND(k0, "s_waitcnt lgkmcnt(0)\n\ts_nop 0\n\t", HALF_RATE, FULL_RATE) \
    KF_ROUND(k1, "", HALF_RATE, FULL_RATE) \
    "v_add_u32_e64 %[at], 16, %[at]\n\t" \
    "s_add_u32 %[n], %[n], -1\n\t" /* carries until n is 0 */ \
    "s_cbranch_scc1 keccak%=\n\t" \
    "s_nop 1\n" /* a DPP read of the results: two wait states */
#define KF_OUTS \
    KF_IO(0), KF_IO(1), KF_IO(2), KF_IO(3), KF_IO(4), KF_IO(5), KF_IO(6), \
    KF_IO(7), KF_IO(8), KF_IO(9), KF_IO(10), KF_IO(11), KF_IO(12), \
    KF_IO(13), KF_IO(14), KF_IO(15), KF_IO(16), KF_IO(17), KF_IO(18), \
    KF_IO(19), KF_IO(20), KF_IO(21), KF_IO(22), KF_IO(23), KF_IO(24), \
    KF_B(0), KF_B(1), KF_B(2), KF_B(3), KF_B(4), KF_B(5), KF_B(6), KF_B(7), \
    KF_B(8), KF_B(9), KF_B(10), KF_B(11), KF_B(12), KF_B(13), KF_B(14), \
    KF_B(15), KF_B(16), KF_B(17), KF_B(18), KF_B(19), KF_B(20), KF_B(21), \
    KF_B(22), KF_B(23), KF_B(24), \
    KF_T(c0), KF_T(c1), KF_T(c2), KF_T(c3), KF_T(c4), KF_T(r0), KF_T(r1), KF_T(r2), KF_T(r3), KF_T(r4), \
    KF_T(k0), KF_T(k1), [n] "=&s"(n), [at] "+v"(at)

__device__ __forceinline__ void f1600(uint32_t (&A)[25], Half p)
{
    uint32_t B[25], c0, c1, c2, c3, c4, r0, r1, r2, r3, r4, k0, k1;
    int n;
    uint32_t at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const uint32_t *)(p.rc + p.p);
    if (p.shared)
        asm volatile(KF_PERMUTE("s_setprio 2\n\ts_nop 0\n\t", "s_setprio 0\n\ts_nop 0\n\t")
                     : KF_OUTS
                     :
                     : "scc", "memory");
    else
        asm volatile(KF_PERMUTE("", "") : KF_OUTS : : "scc", "memory");
}
#undef KF_PERMUTE
#undef KF_OUTS
#undef KF_PAR3
#undef KF_PAR2
#undef KF_SWAP
#undef KF_R
#undef KF_ADD
#undef KF_LO
#undef KF_HI
#undef KF_CHI
#undef KF_ROUND
#undef KF_IO
#undef KF_B
#undef KF_T

constexpr int kShake128Rate = 168;
constexpr int kSha3_256Rate = 136;
constexpr int kSha3_512Rate = 72;
constexpr uint8_t kShakeDS = 0x1F;
constexpr uint8_t kSha3DS = 0x06;

// This lane's halves of the n 64-bit words at p_ (8-byte aligned).
template <int N> __device__ __forceinline__ void load_words(uint32_t (&m)[N], const uint8_t *src, Half p)
{
    const uint32_t *w = reinterpret_cast<const uint32_t *>(src);
#pragma unroll
    for (int i = 0; i < N; i++) m[i] = w[2 * i + p];
}
template <int N> __device__ __forceinline__ void store_words(uint8_t *dst, const uint32_t (&m)[N], Half p)
{
    uint32_t *w = reinterpret_cast<uint32_t *>(dst);
#pragma unroll
    for (int i = 0; i < N; i++) w[2 * i + p] = m[i];
}

// Absorb `len` bytes (8-byte aligned source) with rate RATE and domain byte
// `ds`, leaving the state ready for the first squeeze permutation.  The next
// block's words are loaded before the current block is permuted, so their
// latency hides behind the permutation (17 more VGPRs).  Every state index is
// a compile-time constant so the state stays in registers.
template <int RATE>
__device__ __forceinline__ void absorb(uint32_t (&A)[25], const uint8_t *in, int len, uint8_t ds, Half p)
{
    constexpr int RW = RATE / 8;
#pragma unroll
    for (int i = 0; i < 25; i++) A[i] = 0;
    const int blocks = len / RATE;
    const uint32_t *w = reinterpret_cast<const uint32_t *>(in) + p;
    uint32_t nxt[RW];
    if (blocks > 0) {
#pragma unroll
        for (int i = 0; i < RW; i++) nxt[i] = w[2 * i];
    }
    for (int b = 0; b < blocks; b++) {
#pragma unroll
        for (int i = 0; i < RW; i++) A[i] ^= nxt[i];
        w += 2 * RW;
        if (b + 1 < blocks) {
#pragma unroll
            for (int i = 0; i < RW; i++) nxt[i] = w[2 * i];
        }
        f1600(A, p);
    }
    // from the length alone, so that a constant length leaves no tests
    len -= blocks * RATE;
    const int full = len >> 3, rem = len & 7;
    uint64_t last = (uint64_t)ds << (8 * rem);
    const uint8_t *tail = reinterpret_cast<const uint8_t *>(w - p + 2 * full);
    for (int b = 0; b < rem; b++) last |= (uint64_t)tail[b] << (8 * b);
    const uint32_t lh = p ? (uint32_t)(last >> 32) : (uint32_t)last;
#pragma unroll
    for (int i = 0; i < RW; i++) {
        if (i < full) A[i] ^= w[2 * i];
        else if (i == full) A[i] ^= lh;
    }
    A[RW - 1] ^= p ? 0x80000000u : 0u;
}

// Absorption of a message whose bytes become available in pieces (another
// wave is still writing the rest): absorb_upto takes every whole rate block of
// in[done, avail) into A (zeroed by the caller before the first piece),
// advancing `done`; absorb_final then takes the len % RATE bytes left and the
// padding.  in is 8-byte aligned and done stays a multiple of RATE.
template <int RATE>
__device__ __forceinline__ void absorb_upto(uint32_t (&A)[25], const uint8_t *in, int &done, int avail, Half p)
{
    constexpr int RW = RATE / 8;
    uint32_t m[RW];
    auto load = [&] {
        const uint32_t *w = reinterpret_cast<const uint32_t *>(in + done) + p;
#pragma unroll
        for (int i = 0; i < RW; i++) m[i] = w[2 * i];
    };
    if (done + RATE <= avail) load();
    while (done + RATE <= avail) {
#pragma unroll
        for (int i = 0; i < RW; i++) A[i] ^= m[i];
        done += RATE;
        if (done + RATE <= avail) load(); // the next block, while this one is permuted
        f1600(A, p);
    }
}

template <int RATE>
__device__ __forceinline__ void absorb_final(uint32_t (&A)[25], const uint8_t *in, int len, uint8_t ds, Half p)
{
    constexpr int RW = RATE / 8;
    const int done = len / RATE * RATE;
    const int rest = len - done, full = rest >> 3, rem = rest & 7;
    const uint32_t *w = reinterpret_cast<const uint32_t *>(in + done) + p;
    uint64_t last = (uint64_t)ds << (8 * rem);
    const uint8_t *tail = in + done + 8 * full;
    for (int b = 0; b < rem; b++) last |= (uint64_t)tail[b] << (8 * b);
    const uint32_t lh = p ? (uint32_t)(last >> 32) : (uint32_t)last;
#pragma unroll
    for (int i = 0; i < RW; i++) {
        if (i < full) A[i] ^= w[2 * i];
        else if (i == full) A[i] ^= lh;
    }
    A[RW - 1] ^= p ? 0x80000000u : 0u;
}

// Absorb N words held in registers (N * 8 bytes < rate).
template <int N>
__device__ __forceinline__ void absorb_words(uint32_t (&A)[25], const uint32_t (&m)[N], int rate, uint8_t ds, Half p)
{
#pragma unroll
    for (int i = 0; i < 25; i++) A[i] = 0;
#pragma unroll
    for (int i = 0; i < N; i++) A[i] = m[i];
    A[N] ^= p ? 0u : (uint32_t)ds;
    if (rate == kShake128Rate) A[20] ^= p ? 0x80000000u : 0u;
    else if (rate == kSha3_256Rate) A[16] ^= p ? 0x80000000u : 0u;
    else A[8] ^= p ? 0x80000000u : 0u;
}

// SHA3-256 of an 8-byte-aligned buffer -> four words.
__device__ __forceinline__ void sha3_256(uint32_t (&out)[4], const uint8_t *in, int len, Half p)
{
    uint32_t A[25];
    absorb<kSha3_256Rate>(A, in, len, kSha3DS, p);
    f1600(A, p);
#pragma unroll
    for (int i = 0; i < 4; i++) out[i] = A[i];
}

template <int N> __device__ __forceinline__ void sha3_256_words(uint32_t (&out)[4], const uint32_t (&m)[N], Half p)
{
    uint32_t A[25];
    absorb_words(A, m, kSha3_256Rate, kSha3DS, p);
    f1600(A, p);
#pragma unroll
    for (int i = 0; i < 4; i++) out[i] = A[i];
}

__device__ __forceinline__ void sha3_512_words(uint32_t (&out)[8], const uint32_t (&m)[8], Half p)
{
    uint32_t A[25];
    absorb_words(A, m, kSha3_512Rate, kSha3DS, p);
    f1600(A, p);
#pragma unroll
    for (int i = 0; i < 8; i++) out[i] = A[i];
}

// Squeeze `nwords` 64-bit words of SHAKE-128 output (absorbed, not yet
// permuted state), calling f(k, half) with this lane's half of word k.  Only
// the last block tests each word for the end.
template <class F> __device__ __forceinline__ void squeeze_each(uint32_t (&A)[25], int nwords, Half p, F f)
{
    constexpr int RB = kShake128Rate / 8;
    for (int k = 0; k < nwords; k += RB) {
        f1600(A, p);
        if (k + RB <= nwords) {
#pragma unroll
            for (int i = 0; i < RB; i++) f(k + i, A[i]);
        } else {
#pragma unroll
            for (int i = 0; i < RB; i++)
                if (k + i < nwords) f(k + i, A[i]);
        }
    }
}

} // namespace keccak
} // namespace tmvp
