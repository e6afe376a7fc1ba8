// Keccak-f[1600] with one state on the sixteen lanes of a row: the short
// permutation, for calls whose instances do not fill the chip.
//
// On lane pairs (tmvp_keccak.h) a permutation is 122 instructions a round for
// each wave, at four cycles each: 502 cycles.  Here lane (h, i) of a row, h =
// lane bit 3, i = lane bits 0-2, holds the 32-bit halves h of the five words of
// column x = (i + 4) mod 5, so a round is 40 instructions, and 10 waits and
// no-ops.  Columns 0..4 are lanes i = 1..5; i = 0, 6 and 7 repeat columns 4, 0 and
// 1, so that theta's neighbours are one lane away (DPP row_shr / row_shl), and the
// other halves are eight lanes away (row_ror).  pi goes through LDS: every lane
// writes its five rotated words where the rows of the result keep them and reads
// its column and the next two, chi's operands.  The rotation's amount and the words'
// places depend on the lane and sit in registers; a rotation by 32 or more is
// one by 32 less whose result belongs to the other half's place.
//
// What bounds it: the LDS round trip (about 130 of the 304 cycles a round) and
// the instruction chain around it; the LDS itself carries four such waves on a
// CU at 308 cycles a round, eight at 504, where lane pairs are as fast.  A row
// holds one state where a row of lane pairs holds eight, so it pays where
// latency is all that counts.  In LDS a state's words y = 0..3 of a column and
// half are sixteen contiguous bytes and the words y = 4 follow, which avoids bank
// conflicts (columns at a stride of 64 bytes: 320 cycles alone, 404 for four
// waves), though not all: in the KEM kernels conflict cycles count 0.17 to 0.22 of
// the time of the CUs in use.
#pragma once

#include "tmvp_keccak.h"

namespace tmvp {
namespace keccak {

constexpr int kRowDwords = 52; // LDS of one state
constexpr int kRowRc = 52;     // round constants (fill_rc) and zeros behind them

__device__ __forceinline__ uint32_t lds_address(const uint32_t *p)
{
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const uint32_t *)p;
}

// A lane's place in its row and the row's LDS.
struct Row {
    int x, h, i;             // column, half, position
    uint32_t put[5];         // where word y goes
    uint32_t col[3], top[3]; // where columns x, x + 1, x + 2 are: words 0..3, word 4
    uint32_t turn[5];        // alignbit amounts
    uint32_t rc, rc_step;    // round constants of word 0's lanes, zeros for the others

    // state: the row's kRowDwords; rc_table: kRowRc dwords, zeros from kRcDwords on.
    __device__ __forceinline__ Row(const uint32_t *state, const uint32_t *rc_table)
    {
        const int lane = threadIdx.x & 63;
        h = (lane >> 3) & 1;
        i = lane & 7;
        x = i + 4 >= 10 ? i - 6 : i + 4 >= 5 ? i - 1 : i + 4;
        const uint32_t base = lds_address(state);
        // rho offsets of column x, six bits each, word y = 0 first
        constexpr uint32_t rho[5] = {0u | 36u << 6 | 3u << 12 | 41u << 18 | 18u << 24,
                                     1u | 44u << 6 | 10u << 12 | 45u << 18 | 2u << 24,
                                     62u | 6u << 6 | 43u << 12 | 15u << 18 | 61u << 24,
                                     28u | 55u << 6 | 25u << 12 | 21u << 18 | 56u << 24,
                                     27u | 20u << 6 | 39u << 12 | 8u << 18 | 14u << 24};
        const uint32_t mine = x == 0 ? rho[0] : x == 1 ? rho[1] : x == 2 ? rho[2] : x == 3 ? rho[3] : rho[4];
#pragma unroll
        for (int y = 0; y < 5; y++) {
            const int r = (mine >> (6 * y)) & 63, s = r & 31;
            turn[y] = (32 - s) & 31; // alignbit by 0 gives the other half: a word that stays goes there
            const int half = h ^ (int)((r >= 32) != (s == 0));
            const int to = (2 * x + 3 * y) % 5; // row of the result; its column is y
            put[y] = base + (to < 4 ? (half * 5 + y) * 16 + 4 * to : 160 + 4 * (half * 5 + y));
            if (!real()) put[y] = base + 200 + 4 * h; // repeated columns write nowhere
        }
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const int c = x + k >= 5 ? x + k - 5 : x + k;
            col[k] = base + (h * 5 + c) * 16;
            top[k] = base + 160 + 4 * (h * 5 + c);
        }
        rc = lds_address(rc_table) + (x == 0 ? 4 * h : 4 * kRcDwords);
        rc_step = x == 0 ? 8 : 0;
    }
    __device__ __forceinline__ bool real() const { return i >= 1 && i <= 5; }
    // This lane's half of word x + 5 y of a byte string, in dwords.
    __device__ __forceinline__ int at(int y) const { return 2 * (x + 5 * y) + h; }
};

#define KR_ROUND                                                                                                     \
    "v_bitop3_b32 %[c], %[a0], %[a1], %[a2] bitop3:0x96\n\t"                                                         \
    "ds_read_b32 %[k], %[at]\n\t"                                                                                    \
    "v_add_u32_e64 %[at], %[step], %[at]\n\t"                                                                        \
    "v_bitop3_b32 %[c], %[c], %[a3], %[a4] bitop3:0x96\n\t"                                                          \
    "s_nop 1\n\ts_nop 0\n\t"                                                                                         \
    "v_mov_b32_dpp %[p], %[c] row_ror:8 row_mask:0xf bank_mask:0xf\n\t"                                              \
    "v_mov_b32_dpp %[m], %[c] row_shr:1 row_mask:0xf bank_mask:0xf\n\t"                                              \
    "v_alignbit_b32 %[r], %[c], %[p], 31\n\t"                                                                        \
    "s_nop 1\n\ts_nop 0\n\t"                                                                                         \
    "v_mov_b32_dpp %[p], %[r] row_shl:1 row_mask:0xf bank_mask:0xf\n\t"                                              \
    "s_nop 0\n\ts_nop 0\n\t"                                                                                         \
    KR_5("v_bitop3_b32 %[a", "], %[a", "], %[m], %[p] bitop3:0x96\n\t")                                              \
    "v_mov_b32_dpp v96, %[a0] row_ror:8 row_mask:0xf bank_mask:0xf\n\t"                                              \
    "v_mov_b32_dpp v97, %[a1] row_ror:8 row_mask:0xf bank_mask:0xf\n\t"                                              \
    "v_mov_b32_dpp v98, %[a2] row_ror:8 row_mask:0xf bank_mask:0xf\n\t"                                              \
    "v_mov_b32_dpp v99, %[a3] row_ror:8 row_mask:0xf bank_mask:0xf\n\t"                                              \
    "v_mov_b32_dpp v100, %[a4] row_ror:8 row_mask:0xf bank_mask:0xf\n\t"                                             \
    "v_alignbit_b32 %[a0], %[a0], v96, %[t0]\n\t"                                                                    \
    "v_alignbit_b32 %[a1], %[a1], v97, %[t1]\n\t"                                                                    \
    "v_alignbit_b32 %[a2], %[a2], v98, %[t2]\n\t"                                                                    \
    "v_alignbit_b32 %[a3], %[a3], v99, %[t3]\n\t"                                                                    \
    "v_alignbit_b32 %[a4], %[a4], v100, %[t4]\n\t"                                                                   \
    KR_5("ds_write_b32 %[w", "], %[a", "]\n\t")                                                                      \
    "ds_read_b128 v[96:99], %[d0]\n\t"                                                                               \
    "ds_read_b128 v[102:105], %[d1]\n\t"                                                                             \
    "ds_read_b128 v[108:111], %[d2]\n\t"                                                                             \
    "ds_read_b32 v100, %[e0]\n\t"                                                                                    \
    "ds_read_b32 v106, %[e1]\n\t"                                                                                    \
    "ds_read_b32 v112, %[e2]\n\t"                                                                                    \
    "s_waitcnt lgkmcnt(3)\n\ts_nop 0\n\t"                                                                            \
    "v_bitop3_b32 %[a0], v96, v102, v108 bitop3:0xd2\n\t"                                                            \
    "v_bitop3_b32 %[a1], v97, v103, v109 bitop3:0xd2\n\t"                                                            \
    "v_bitop3_b32 %[a2], v98, v104, v110 bitop3:0xd2\n\t"                                                            \
    "v_bitop3_b32 %[a3], v99, v105, v111 bitop3:0xd2\n\t"                                                            \
    "v_xor_b32_e64 %[a0], %[a0], %[k]\n\t"                                                                           \
    "s_waitcnt lgkmcnt(0)\n\ts_nop 0\n\t"                                                                            \
    "v_bitop3_b32 %[a4], v100, v106, v112 bitop3:0xd2\n\t"
#define KR_5(a, b, c) a "0" b "0" c a "1" b "1" c a "2" b "2" c a "3" b "3" c a "4" b "4" c

// A[y]: this lane's half of word x + 5 y.  Every lane of the row takes part.
__device__ __forceinline__ void f1600(uint32_t (&A)[5], const Row &L)
{
    uint32_t c, p, m, r, k, at = L.rc;
    int n;
    asm volatile("s_movk_i32 %[n], 11\n\t"
                 ".p2align 6\n"
                 "keccak_row%=:\n\t"
                 KR_ROUND KR_ROUND
                 "s_add_u32 %[n], %[n], -1\n\t"
                 "s_cbranch_scc1 keccak_row%=\n\t"
                 "s_nop 1\n"
                 : [a0] "+v"(A[0]), [a1] "+v"(A[1]), [a2] "+v"(A[2]), [a3] "+v"(A[3]), [a4] "+v"(A[4]), [c] "=&v"(c),
                   [p] "=&v"(p), [m] "=&v"(m), [r] "=&v"(r), [k] "=&v"(k), [at] "+v"(at), [n] "=&s"(n)
                 : [step] "v"(L.rc_step), [t0] "v"(L.turn[0]), [t1] "v"(L.turn[1]), [t2] "v"(L.turn[2]),
                   [t3] "v"(L.turn[3]), [t4] "v"(L.turn[4]), [w0] "v"(L.put[0]), [w1] "v"(L.put[1]),
                   [w2] "v"(L.put[2]), [w3] "v"(L.put[3]), [w4] "v"(L.put[4]), [d0] "v"(L.col[0]), [d1] "v"(L.col[1]),
                   [d2] "v"(L.col[2]), [e0] "v"(L.top[0]), [e1] "v"(L.top[1]), [e2] "v"(L.top[2])
                 : "scc", "memory", "v96", "v97", "v98", "v99", "v100", "v102", "v103", "v104", "v105", "v106", "v108",
                   "v109", "v110", "v111", "v112");
}
#undef KR_ROUND
#undef KR_5

__device__ __forceinline__ void row_zero(uint32_t (&A)[5])
{
#pragma unroll
    for (int y = 0; y < 5; y++) A[y] = 0;
}

// This lane's halves of the first N words at src (global memory or LDS); 0 beyond them.
template <int N> __device__ __forceinline__ void row_load(uint32_t (&m)[5], const uint32_t *src, const Row &L)
{
#pragma unroll
    for (int y = 0; y < 5; y++) {
        m[y] = 0;
        if (5 * y < N && (5 * y + 5 <= N || L.x + 5 * y < N)) m[y] = src[L.at(y)];
    }
}

template <int N> __device__ __forceinline__ void row_store(uint32_t *dst, const uint32_t (&A)[5], const Row &L)
{
    if (!L.real()) return;
#pragma unroll
    for (int y = 0; y < 5; y++)
        if (5 * y < N && (5 * y + 5 <= N || L.x + 5 * y < N)) dst[L.at(y)] = A[y];
}

// Domain byte at word N (the message is N words into its last block) and the
// rate's final bit.
template <int N, int RATE> __device__ __forceinline__ void row_pad(uint32_t (&A)[5], uint8_t ds, const Row &L)
{
    constexpr int last = RATE / 8 - 1;
#pragma unroll
    for (int y = 0; y < 5; y++) {
        if (y == N / 5 && L.x == N % 5 && L.h == 0) A[y] ^= ds;
        if (y == last / 5 && L.x == last % 5 && L.h == 1) A[y] ^= 0x80000000u;
    }
}

// The sponge of one block: N words at src, permuted.
template <int N, int RATE>
__device__ __forceinline__ void row_hash(uint32_t (&A)[5], const uint32_t *src, uint8_t ds, const Row &L)
{
    row_load<N>(A, src, L);
    row_pad<N, RATE>(A, ds, L);
    f1600(A, L);
}

// SHA3-256 blocks [from, to) of the message at in, the next block loaded while
// one is permuted; A holds the blocks before them.
__device__ __forceinline__ void row_absorb(uint32_t (&A)[5], const uint8_t *in, int from, int to, const Row &L)
{
    constexpr int RW = kSha3_256Rate / 8;
    const uint32_t *w = reinterpret_cast<const uint32_t *>(in) + 2 * RW * from;
    uint32_t m[5];
    if (from < to) row_load<RW>(m, w, L);
    for (int b = from; b < to; b++) {
#pragma unroll
        for (int y = 0; y < 5; y++) A[y] ^= m[y];
        w += 2 * RW;
        if (b + 1 < to) row_load<RW>(m, w, L);
        f1600(A, L);
    }
}

// The last block of a message of LEN bytes (a multiple of 8), permuted.
template <int LEN> __device__ __forceinline__ void row_absorb_last(uint32_t (&A)[5], const uint8_t *in, const Row &L)
{
    constexpr int RW = kSha3_256Rate / 8, N = LEN / 8 % RW;
    static_assert(LEN % 8 == 0, "words");
    if constexpr (N > 0) {
        uint32_t m[5];
        row_load<N>(m, reinterpret_cast<const uint32_t *>(in) + 2 * (LEN / 8 - N), L);
#pragma unroll
        for (int y = 0; y < 5; y++) A[y] ^= m[y];
    }
    row_pad<N, kSha3_256Rate>(A, kSha3DS, L);
    f1600(A, L);
}

} // namespace keccak
} // namespace tmvp
