// Batched Saber/Sable KEM on the GPU: sampling (SHAKE-128 GenMatrix and
// centred-binomial GenSecret), codecs, the Fujisaki-Okamoto hashes, and the
// host-side launch chains for key generation, encapsulation and
// decapsulation.  The products and rounding run in the MatrixVectorMul /
// InnerProd kernels (launch_mfma / launch_valu).
//
// Step order follows saber_enc / saber_dec (S/src/cuda_kernel.cu:114-186,
// :341-450) and SABLE_enc / SABLE_dec (SB/src/SABLE_indcpa.cu:133-233,
// :422-563); the decapsulation replaces the pre-key with z before the final
// hash when the re-encryption differs (Saber round 3), which the reference's
// verify_gpu / cmov_gpu (S/src/pack.cu:225-255) never do.  Key generation is
// absent from the reference and follows Saber round 3 (seed_A is hashed with
// SHAKE-128, b = round(A^T s)).
//
// Sponges run on a pair of lanes per instance (state in registers, split in
// 32-bit halves), or, in the one-launch kernels of small batches, on a row of
// sixteen (tmvp_keccak_row.h).  In the chains of kernels they write their
// results in the form the products read: A (through a buffer in LDS), s, b of the
// public key and the message bits; in the one-launch kernels they write the
// raw stream, and the products read it packed (tmvp_rows.h).  The sponges' lanes
// also pack the secret into the sk (key generation) and the ciphertext before
// hashing it (encapsulation); the other codecs run one thread per 64
// coefficients.
#include <string.h>

#include <type_traits>
#include <utility>

#include "tmvp_internal.h"
#include "tmvp_keccak.h"
#include "tmvp_keccak_row.h"
#include "tmvp_kem.h"
#include "tmvp_kem_form.h"
#include "tmvp_rows.h"

namespace tmvp {

using namespace keccak;

// ---------------------------------------------------------------- sampling
//
// Every sponge runs on a pair of adjacent lanes (tmvp_keccak.h): thread g of a
// sponge kernel works on pair t = g >> 1, half p = g & 1, and both lanes of a
// pair always take the same branch.

// The compile-time shape of a parameter set's sampling: EQ (matrix bits), MU
// (CBD width) and EP (bits of b).  Each sponge kernel is instantiated per
// shape, so it holds only its own set's code paths (a kernel holding every
// set's variants measured 19 us slower on Saber encapsulation).
template <int EQ_, int MU_, int EP_> struct Shape {
    static constexpr int EQ = EQ_, MU = MU_, EP = EP_;
};

// SHARED: the kernel's launch puts several of its one-wave workgroups on a SIMD
// (by_load), see keccak::f1600.
#define TMVP_PAIR(t0, SHARED)                                                                                        \
    const int64_t t = (((int64_t)blockIdx.x * 64 + threadIdx.x) >> 1) + (t0);                                       \
    __shared__ __attribute__((aligned(16))) uint32_t rc_lds[kRcDwords];                                              \
    fill_rc(rc_lds);                                                                                                 \
    __syncthreads();                                                                                                 \
    const Half p{(int)(threadIdx.x & 1), rc_lds, SHARED}

// GenMatrix (S/src/pack.cu:145-153 with the 13-bit unpacking of :51-65;
// SB/src/pack.cu:22-50, 11 bits): the SHAKE-128(seed) stream read as EQ-bit
// little-endian coefficients, in the order of A[i][j][k].  64 coefficients
// are exactly EQ 64-bit words of the stream, so the squeezed words go through
// a buffer in LDS (per instance; the pair's lanes write the low and high
// dwords of each word) and every group of EQ words the stream has completed is
// unpacked at once, lane p taking coefficients 32p..32p+31 of it, which are
// exactly its EQ dwords.  The words of the unfinished group (at most EQ - 1)
// are written again at the buffer's front, and the next block goes right
// behind them: a block's 21 writes have one address and constant offsets.
// (A ring instead tested every word for the stream's end and the ring's wrap:
// 42 branches a block, about 2600 cycles between permutations of 14500.)
// kTailWords words before the front take the rewritten words that are not
// left over.  The buffer's instance stride (90 dwords) keeps the 64 lanes'
// reads and writes in distinct banks.
constexpr int kTailWords = 12;                              // groups have at most 13 words
constexpr int kRingDwords = 2 * (2 * kTailWords + kShake128Rate / 8); // per instance

// The 32 W-bit coefficients packed LSB-first in d[0..W) to dst (16-byte
// aligned), one dword of two coefficients at a time.  The bits of a 16-bit
// element above W are left as they come: every product takes its operands
// modulo 2^W (the matrix-core form masks them as it splits the limbs).
template <int W> __device__ __forceinline__ void unpack32(const uint32_t (&d)[W], uint16_t *dst)
{
    uint32_t o[16];
#pragma unroll
    for (int j = 0; j < 16; j++) {
        const int bit = 2 * W * j, i = bit >> 5, sh = bit & 31;
        const uint32_t t = sh + 2 * W <= 32 ? (d[i] >> sh) : __builtin_amdgcn_alignbit(d[i + 1 < W ? i + 1 : i], d[i], sh);
        o[j] = __builtin_amdgcn_bitop3_b32(0xffff0000u, t << (16 - W), t, 0xca); // high half of the shift, low half of t
    }
    uint4 *q4 = reinterpret_cast<uint4 *>(dst);
#pragma unroll
    for (int q = 0; q < 4; q++) q4[q] = make_uint4(o[4 * q], o[4 * q + 1], o[4 * q + 2], o[4 * q + 3]);
}

// A packed W-bit vector of ncoef coefficients (ncoef a multiple of 256) at
// src, unpacked to dst by a lane pair: 64 coefficients are W 64-bit words, and
// lane p takes coefficients 32p..32p+31 of each group, its W dwords.  Four
// groups' loads are issued before their stores (stores in flight hold up the
// next loads' wait).
template <int W> __device__ __forceinline__ void unpack_pair(const uint8_t *src, uint16_t *dst, int ncoef, Half p)
{
    for (int g0 = 0; g0 < ncoef / 64; g0 += 4) {
        uint32_t d[4][W];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const uint32_t *s = reinterpret_cast<const uint32_t *>(src + 8 * W * (g0 + u)) + W * p;
#pragma unroll
            for (int i = 0; i < W; i++) d[u][i] = s[i];
        }
#pragma unroll
        for (int u = 0; u < 4; u++) unpack32<W>(d[u], dst + 64 * (g0 + u) + 32 * p);
    }
}

// The vector b of a public key (its first pvc bytes, EP bits per coefficient).
template <int EP> __device__ __forceinline__ void unpack_b(const KemParams &P, const uint8_t *pk, uint16_t *dst, Half p)
{
    unpack_pair<EP>(pk, dst, P.l * kN, p);
}

// The message bits as one 0/1 coefficient each (bit k of m is coefficient k):
// this lane's halves of the four words cover coefficients 64w + 32p + j.
__device__ __forceinline__ void message_bits(const uint32_t (&m)[4], uint16_t *dst, Half p)
{
#pragma unroll
    for (int w = 0; w < 4; w++) {
        uint32_t o[16];
#pragma unroll
        for (int q = 0; q < 16; q++) o[q] = ((m[w] >> (2 * q)) & 1u) | (((m[w] >> (2 * q + 1)) & 1u) << 16);
        uint4 *q4 = reinterpret_cast<uint4 *>(dst + 64 * w + 32 * p);
#pragma unroll
        for (int q = 0; q < 4; q++) q4[q] = make_uint4(o[4 * q], o[4 * q + 1], o[4 * q + 2], o[4 * q + 3]);
    }
}

// The SHAKE-128(seed) stream of nwords words (a multiple of G), handed to
// f(g, d) one group of G words at a time: d holds this lane's G dwords of
// group g (dwords G p .. G p + G - 1 of the group's 2G).  buf is the
// instance's kRingDwords in LDS.
template <int G, class F>
__device__ __forceinline__ void stream_groups(const uint32_t (&seed)[4], int nwords, uint32_t *buf, Half p, F f)
{
    constexpr int RB = kShake128Rate / 8;
    static_assert(G - 1 <= kTailWords, "buffer size");
    uint32_t st[25];
    absorb_words(st, seed, kShake128Rate, kShakeDS, p);
    uint32_t *const front = buf + 2 * kTailWords;
    const int groups = nwords / G;
    int g = 0;  // next group to hand over
    int lo = 0; // words of it already at the front
    while (g < groups) {
        f1600(st, p);
        uint32_t *w = front + 2 * lo + p;
#pragma unroll
        for (int i = 0; i < RB; i++) w[2 * i] = st[i];
        // The pair's writes above are read by both lanes below; the wave's LDS
        // operations execute in order, so only code motion must be stopped.
        __builtin_amdgcn_wave_barrier();
        lo += RB;
        const uint32_t *src = front + G * p;
        for (; lo >= G; lo -= G, src += 2 * G) {
            if (g < groups) { // the last block may hold more words than the stream needs
                uint32_t d[G];
#pragma unroll
                for (int i = 0; i < G; i++) d[i] = src[i];
                f(g, d);
                g++;
            }
        }
        __builtin_amdgcn_wave_barrier();
        uint32_t *v = front + 2 * (lo - RB) + p; // the block's last lo words come to the front
#pragma unroll
        for (int i = RB - (G - 1); i < RB; i++) v[2 * i] = st[i];
    }
}

// GenMatrix: 64 coefficients of EQ bits are exactly EQ words of the stream.
template <int EQ>
__device__ __forceinline__ void matrix_to_a(const uint32_t (&seed)[4], uint16_t *arow, int nwords, uint32_t *ring,
                                            Half p)
{
    stream_groups<EQ>(seed, nwords, ring, p,
                         [&](int g, const uint32_t(&d)[EQ]) { unpack32<EQ>(d, arow + 64 * g + 32 * p); });
}

// A[t] from the 32-byte seed; `ring` is the instance's kRingDwords in LDS.
template <int EQ>
__device__ __forceinline__ void gen_matrix(const KemParams &P, const uint32_t (&seed)[4], uint16_t *arow,
                                           uint32_t *ring, Half p)
{
    matrix_to_a<EQ>(seed, arow, P.araw / 8, ring, p);
}

#define TMVP_RING                                                                                                    \
    __shared__ uint32_t ring_lds[32 * kRingDwords];                                                                  \
    uint32_t *const ring = ring_lds + (threadIdx.x >> 1) * kRingDwords

// CBD_mu (S/src/poly.cu:836-916, SB/src/fips202.cu:625-651): coefficient c
// is the popcount of stream bits [c mu, c mu + mu/2) minus that of the next
// mu/2 bits, stored as int16 (Saber) or masked mod q (Sable) by qmask.  For
// mu = 8 and mu = 2 every coefficient lies inside one 32-bit half of a word
// (bit i of this lane's half of word k is stream bit 64k + 32p + i) and is
// sampled straight from the squeeze; for mu = 6 and 10 the coefficients
// straddle the halves, and 64 of them are exactly mu words, so they go through
// the LDS ring.  S is the instance's row of L * 256 coefficients.

// The samplers give each coefficient plus kCbdBias as a byte.
constexpr uint32_t kCbdBias = 8;

// mu = 8: the four coefficients in h.
__device__ __forceinline__ uint32_t cbd8(uint32_t h)
{
    uint32_t x = h - ((h >> 1) & 0x55555555u);
    x = (x & 0x33333333u) + ((x >> 2) & 0x33333333u); // popcount of every nibble
    return (x & 0x0f0f0f0fu) + kCbdBias * 0x01010101u - ((x >> 4) & 0x0f0f0f0fu);
}

// mu = 2: the four coefficients in the low byte of h.
__device__ __forceinline__ uint32_t cbd2(uint32_t h)
{
    uint32_t y = h & 0xffu;
    y = (y | (y << 12)) & 0x000f000fu;
    y = (y | (y << 6)) & 0x03030303u;
    return (y & 0x01010101u) + kCbdBias * 0x01010101u - ((y >> 1) & 0x01010101u);
}

// mu = 6 and 10: the 32 coefficients whose MU-bit fields are packed LSB-first
// in d, four to a dword.  The popcounts of the MU/2-bit fields of 24 (four
// coefficients) or 20 bits (two) are summed bit by bit, all fields at once.
template <int MU> __device__ __forceinline__ void cbd32(const uint32_t (&d)[MU], uint32_t (&o)[8])
{
    constexpr int H = MU / 2, C = MU == 6 ? 4 : 2; // coefficients per piece
    constexpr uint32_t ones = MU == 6 ? 0x249249u : 0x08421u;    // bit 0 of every H-bit field
    constexpr uint32_t bias = MU == 6 ? 0x041041u : 0x00401u;    // bit 0 of every coefficient
    constexpr uint32_t count = bias * ((1u << H) - 1u);          // the first field of every coefficient
#pragma unroll
    for (int q = 0; q < 32 / C; q++) {
        const int bit = MU * C * q, i = bit >> 5, sh = bit & 31;
        const uint32_t t = sh + MU * C <= 32 ? (d[i] >> sh) : __builtin_amdgcn_alignbit(d[i + 1 < MU ? i + 1 : i], d[i], sh);
        uint32_t c = t & ones;
#pragma unroll
        for (int b = 1; b < H; b++) c += (t >> b) & ones;
        const uint32_t e = (c & count) + kCbdBias * bias - ((c >> H) & count); // MU-bit fields
        if constexpr (MU == 6) {
            o[q] = (e & 0x3fu) | ((e << 2) & 0x3f00u) | ((e << 4) & 0x3f0000u) | ((e << 6) & 0x3f000000u);
        } else {
            const uint32_t two = (e & 0x3ffu) | ((e << 6) & 0x3ff0000u); // halfwords
            const uint32_t b2 = (two & 0xffu) | ((two >> 8) & 0xff00u);
            o[q >> 1] = q & 1 ? o[q >> 1] | (b2 << 16) : b2;
        }
    }
}

// Four samples as int8.
__device__ __forceinline__ uint32_t cbd_int8(uint32_t e) { return ((e | 0x80808080u) - kCbdBias * 0x01010101u) ^ 0x80808080u; }

// Four samples as halfwords, masked by qmask.
__device__ __forceinline__ uint2 cbd_int16(uint32_t e, uint32_t qmask)
{
    auto widen = [&](uint32_t sel) { // selector 0x0c: a zero byte
        return sub16x2(__builtin_amdgcn_perm(0u, e, sel), kCbdBias * 0x00010001u) & (qmask * 0x00010001u);
    };
    return make_uint2(widen(0x0c010c00u), widen(0x0c030c02u));
}

// The secret of one instance from its 32-byte seed: the samples of four
// consecutive coefficients 4 i .. 4 i + 3 go to put(i, biased bytes).
template <int MU, class F>
__device__ __forceinline__ void sample_secret(const uint32_t (&seed)[4], int nwords, uint32_t *buf, Half p, F put)
{
    if constexpr (MU == 8 || MU == 2) {
        uint32_t A[25];
        absorb_words(A, seed, kShake128Rate, kShakeDS, p);
        squeeze_each(A, nwords, p, [&](int k, uint32_t h) {
            if constexpr (MU == 8) {
                put(2 * k + p, cbd8(h));
            } else {
#pragma unroll
                for (int q = 0; q < 4; q++) put(8 * k + 4 * p + q, cbd2(h >> (8 * q)));
            }
        });
    } else {
        static_assert(MU == 6 || MU == 10, "CBD width");
        stream_groups<MU>(seed, nwords, buf, p, [&](int g, const uint32_t(&d)[MU]) {
            uint32_t o[8];
            cbd32<MU>(d, o);
#pragma unroll
            for (int q = 0; q < 8; q++) put(16 * g + 8 * p + q, o[q]);
        });
    }
}

// As halfwords, two's complement (Saber) or masked mod q (Sable), to S.
template <int MU>
__device__ __forceinline__ void secret_stream(const KemParams &P, const uint32_t (&seed)[4], uint16_t *S,
                                              uint32_t *buf, Half p)
{
    constexpr uint32_t qmask = MU == 2 ? 0x7ffu : 0xffffu; // the Sable sets: mu = 2, q = 2^11
    uint2 *dst = reinterpret_cast<uint2 *>(S);
    sample_secret<MU>(seed, P.sraw / 8, buf, p, [&](int i, uint32_t e) { dst[i] = cbd_int16(e, qmask); });
}

// As int8 to s (the one-launch kernels).
template <class S>
__device__ __forceinline__ void secret_bytes(const uint32_t (&seed)[4], uint8_t *s, uint32_t *buf, Half p)
{
    uint32_t *dst = reinterpret_cast<uint32_t *>(s);
    sample_secret<S::MU>(seed, S::L * S::MU * 4, buf, p, [&](int i, uint32_t e) { dst[i] = cbd_int8(e); });
}

// One instance's polynomials packed by its lane pair (the codecs of
// S/src/pack.cu:1-213 and SB/src/pack.cu:182-467): chunk c of 64 coefficients
// is W 64-bit words of the LSB-first W-bit code, and lane p's 32 coefficients
// 32p..32p+31 of it are exactly dwords pW..pW+W-1.  SK2: the Sable secret
// code s & 3 (SB/src/pack.cu:366-377).
//
// Callers order these accesses against the pair's other ones with a
// workgroup-scope fence (the workgroup is this one wave): one after the stores
// that wrote the source, one before loads of what was packed.  An agent-scope
// fence would also write back the L2, which made key generation 24 us slower.
__device__ __forceinline__ void wave_fence_global()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

template <int W, bool SK2>
__device__ __forceinline__ void pack_half(const uint16_t *S, uint8_t *dst, int nchunks, Half p, uint8_t *dst2 = nullptr)
{
    constexpr uint32_t mask = SK2 ? 3u : (1u << W) - 1u;
    constexpr int G = 4; // chunks whose loads are in flight together (nchunks is a multiple of 4)
    for (int c0 = 0; c0 < nchunks; c0 += G) {
        uint4 v[G][4];
#pragma unroll
        for (int g = 0; g < G; g++) {
            const uint4 *src = reinterpret_cast<const uint4 *>(S + 64 * (c0 + g) + 32 * p);
#pragma unroll
            for (int q = 0; q < 4; q++) v[g][q] = src[q];
        }
#pragma unroll
        for (int g = 0; g < G; g++) {
            uint32_t e[32];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const uint32_t h[4] = {v[g][q].x, v[g][q].y, v[g][q].z, v[g][q].w};
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    e[8 * q + 2 * k] = h[k] & mask;
                    e[8 * q + 2 * k + 1] = (h[k] >> 16) & mask;
                }
            }
            uint32_t w[W];
#pragma unroll
            for (int i = 0; i < W; i++) w[i] = 0;
#pragma unroll
            for (int j = 0; j < 32; j++) {
                const int bit = W * j, i = bit >> 5, o = bit & 31;
                w[i] |= e[j] << o;
                if (o + W > 32) w[i + 1] |= e[j] >> (32 - o);
            }
            uint32_t *d = reinterpret_cast<uint32_t *>(dst + (int64_t)(c0 + g) * W * 8) + p * W;
#pragma unroll
            for (int i = 0; i < W; i++) d[i] = w[i];
            if (dst2) {
                uint32_t *d2 = reinterpret_cast<uint32_t *>(dst2 + (int64_t)(c0 + g) * W * 8) + p * W;
#pragma unroll
                for (int i = 0; i < W; i++) d2[i] = w[i];
            }
        }
    }
}

// 32 int8 secret coefficients as the secret key holds them: W-bit two's
// complement (W = 2: the Sable code s & 3).
template <int W> __device__ __forceinline__ void pack_int8(const uint32_t (&v)[8], uint32_t (&w)[W])
{
#pragma unroll
    for (int i = 0; i < W; i++) w[i] = 0;
#pragma unroll
    for (int j = 0; j < 32; j++) {
        const uint32_t e = (uint32_t)((int32_t)(v[j >> 2] << (24 - 8 * (j & 3))) >> 24) & ((1u << W) - 1u);
        const int bit = W * j, i = bit >> 5, o = bit & 31;
        w[i] |= e << o;
        if (o + W > 32) w[i + 1] |= e >> (32 - o);
    }
}

// An int8 secret (secret_bytes) into the secret key.  A lane packs half of
// every chunk, as in pack_half.
template <class S> __device__ __forceinline__ void pack_secret(const uint8_t *s, uint8_t *sk, Half p)
{
    constexpr int W = S::kSable ? 2 : S::EQ;
    wave_fence_global(); // the sampling wrote s with the pair's lanes interleaved
    for (int c = 0; c < 4 * S::L; c++) {
        const uint4 *src = reinterpret_cast<const uint4 *>(s + 64 * c + 32 * p);
        const uint4 a = src[0], b = src[1];
        const uint32_t v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        uint32_t w[W];
        pack_int8<W>(v, w);
        uint32_t *d = reinterpret_cast<uint32_t *>(sk + c * W * 8) + p * W;
#pragma unroll
        for (int i = 0; i < W; i++) d[i] = w[i];
    }
}

// 32 halfword coefficients at S as W-bit codes.
template <int W> __device__ __forceinline__ void pack_coefficients(const uint16_t *S, uint32_t (&w)[W])
{
    constexpr uint32_t mask = (1u << W) - 1u;
    const uint4 *src = reinterpret_cast<const uint4 *>(S);
    uint4 v[4];
#pragma unroll
    for (int q = 0; q < 4; q++) v[q] = src[q];
#pragma unroll
    for (int i = 0; i < W; i++) w[i] = 0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const uint32_t h[4] = {v[q].x, v[q].y, v[q].z, v[q].w};
#pragma unroll
        for (int e2 = 0; e2 < 8; e2++) {
            const int j = 8 * q + e2;
            const uint32_t e = (e2 & 1 ? h[e2 >> 1] >> 16 : h[e2 >> 1]) & mask;
            const int bit = W * j, i = bit >> 5, o = bit & 31;
            w[i] |= e << o;
            if (o + W > 32) w[i + 1] |= e >> (32 - o);
        }
    }
}

// pack_half's code of one instance's polynomials, compared with the bytes at
// dst instead of written there: nonzero when they differ (this lane's half).
template <int W>
__device__ __forceinline__ uint32_t pack_compare_half(const uint16_t *S, const uint8_t *dst, int nchunks, Half p)
{
    uint32_t x = 0;
    for (int c = 0; c < nchunks; c++) {
        const uint32_t *d = reinterpret_cast<const uint32_t *>(dst + (int64_t)c * W * 8) + p * W;
        uint32_t w[W], have[W];
#pragma unroll
        for (int i = 0; i < W; i++) have[i] = d[i];
        pack_coefficients<W>(S + 64 * c + 32 * p, w);
#pragma unroll
        for (int i = 0; i < W; i++) x |= w[i] ^ have[i];
    }
    return x;
}

// G(m | H(pk)) -> buf = m | H(pk), kr; returns the coins kr[32:64]; the
// shared first step of encapsulation and of the re-encryption in
// decapsulation (S/src/cuda_kernel.cu:116-118, :378-379).
__device__ __forceinline__ void hash_g(const uint32_t (&m)[4], const uint32_t (&hpk)[4], uint8_t *buf, uint8_t *kr,
                                       uint32_t (&coins)[4], Half p)
{
    uint32_t b[8], k[8];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        b[i] = m[i];
        b[4 + i] = hpk[i];
    }
    sha3_512_words(k, b, p);
    store_words(buf, b, p);
    store_words(kr, k, p);
#pragma unroll
    for (int i = 0; i < 4; i++) coins[i] = k[4 + i];
}

// The front kernels run the long matrix sponge (23 permutations for Saber;
// pairs [0, B)) beside the rest of the instance's hashing and its secret
// stream (pairs [B, 2B)), one wave per SIMD at B = 16384: a sponge wave alone
// is latency-bound, and separate launches of the two roles share SIMDs and
// slow the matrix sponge down.  A kernel starting at pair t0 = B skips the
// matrix.

// Key generation: seeds[t] = seed_A | seed_s | z.  Matrix role: seed_A' =
// SHAKE-128(seed_A) goes to the pk tail (and the sk's copy of it) and seeds
// GenMatrix.  Secret role: seed_s seeds the secret, which goes to S and,
// packed, to the head of the sk; z goes to the sk tail.
template <class SH>
__device__ __forceinline__ void kp_matrix_role(const KemParams &P, const uint8_t *seeds, uint8_t *pk, uint8_t *sk,
                                               uint16_t *A, int64_t t, uint32_t *ring, Half p)
{
    uint32_t m[4], st[25];
    load_words(m, seeds + t * 96, p);
    absorb_words(st, m, kShake128Rate, kShakeDS, p);
    f1600(st, p);
    const uint32_t sa[4] = {st[0], st[1], st[2], st[3]};
    store_words(pk + t * P.pk + P.pvc, sa, p);
    store_words(sk + t * P.sk + P.indcpa_sk + P.pvc, sa, p);
    gen_matrix<SH::EQ>(P, sa, A + t * P.l * P.l * kN, ring, p);
}

template <class SH>
__device__ __forceinline__ void kp_secret_role(const KemParams &P, const uint8_t *seeds, uint8_t *sk, uint16_t *S,
                                               int64_t t, uint32_t *ring, Half p)
{
    uint32_t m[4];
    load_words(m, seeds + t * 96 + 32, p);
    secret_stream<SH::MU>(P, m, S + t * P.l * kN, ring, p);
    wave_fence_global(); // the sampling wrote S with the pair's lanes interleaved
    if constexpr (SH::MU == 2) pack_half<2, true>(S + t * P.l * kN, sk + t * P.sk, 4 * P.l, p);
    else pack_half<SH::EQ, false>(S + t * P.l * kN, sk + t * P.sk, 4 * P.l, p);
    load_words(m, seeds + t * 96 + 64, p);
    store_words(sk + t * P.sk + P.sk - 32, m, p);
}

// Encapsulation.  Matrix role: GenMatrix from the pk tail.  Secret role:
// m = H(rnd), kr = G(m | H(pk)), the secret from kr[32:64], and the InnerProd
// operands: b of the pk to V and m's bits to bits.  hpk (if not null) holds
// H(pk) per instance.
template <class SH>
__device__ __forceinline__ void enc_matrix_role(const KemParams &P, const uint8_t *pk, uint16_t *A, int64_t t,
                                                uint32_t *ring, Half p)
{
    uint32_t m[4];
    load_words(m, pk + t * P.pk + P.pvc, p);
    gen_matrix<SH::EQ>(P, m, A + t * P.l * P.l * kN, ring, p);
}

template <class SH>
__device__ __forceinline__ void enc_secret_role(const KemParams &P, const uint8_t *rnd, const uint8_t *pk,
                                                const uint8_t *hpk, uint8_t *buf, uint8_t *kr, uint16_t *S,
                                                uint16_t *V, uint16_t *bits, int64_t t, int64_t kt, uint32_t *ring,
                                                Half p)
{
    // t: the instance; kt: its row of pk / hpk (a key id when they are a key store)
    uint32_t r[4], m[4], h[4], coins[4];
    load_words(r, rnd + t * 32, p);
    sha3_256_words<4>(m, r, p);
    if (hpk) load_words(h, hpk + kt * 32, p);
    else sha3_256(h, pk + kt * P.pk, P.pk, p);
    hash_g(m, h, buf + t * 64, kr + t * 64, coins, p);
    secret_stream<SH::MU>(P, coins, S + t * P.l * kN, ring, p);
    message_bits(m, bits + t * kN, p);
    unpack_b<SH::EP>(P, pk + kt * P.pk, V + t * P.l * kN, p);
}

template <class SH, bool SHARED>
__global__ __launch_bounds__(64) void kp_front_kernel(KemParams P, const uint8_t *seeds, uint8_t *pk, uint8_t *sk,
                                                      uint16_t *A, uint16_t *S, int64_t B)
{
    TMVP_PAIR(0, SHARED);
    TMVP_RING;
    if (t >= 2 * B) return;
    if (t < B) kp_matrix_role<SH>(P, seeds, pk, sk, A, t, ring, p);
    else kp_secret_role<SH>(P, seeds, sk, S, t - B, ring, p);
}

// KEYED (A resident, t0 = B): pk and hpk are key stores, read at keys[i].  A
// template flag rather than a null test of keys: with the runtime select the
// non-keyed Saber kernel measured 176 us at B = 16384 against 159 us without.
template <class SH, bool KEYED, bool SHARED>
__global__ __launch_bounds__(64) void enc_front_kernel(KemParams P, const uint8_t *rnd, const uint8_t *pk,
                                                       const uint8_t *hpk, uint8_t *buf, uint8_t *kr, uint16_t *A,
                                                       uint16_t *S, uint16_t *V, uint16_t *bits,
                                                       int64_t B, int64_t t0, const int32_t *keys)
{
    TMVP_PAIR(t0, SHARED);
    TMVP_RING;
    if (t >= 2 * B) return;
    if (t < B) {
        enc_matrix_role<SH>(P, pk, A, t, ring, p);
    } else {
        const int64_t i = t - B;
        enc_secret_role<SH>(P, rnd, pk, hpk, buf, kr, S, V, bits, i, KEYED ? (int64_t)keys[i] : i, ring, p);
    }
}

// Decapsulation, before the decryption and beside it (on the auxiliary
// stream): the matrix stream from the pk inside the sk (pairs [0, B)) and
// H(ct) (pairs [B, 2B)).
template <class SH, bool SHARED>
__global__ __launch_bounds__(64) void dec_pre_kernel(KemParams P, const uint8_t *ct, const uint8_t *sk, uint16_t *A,
                                                     uint8_t *hct, int64_t B)
{
    TMVP_PAIR(0, SHARED);
    TMVP_RING;
    if (t >= 2 * B) return;
    if (t < B) {
        uint32_t m[4];
        load_words(m, sk + t * P.sk + P.indcpa_sk + P.pvc, p);
        gen_matrix<SH::EQ>(P, m, A + t * P.l * P.l * kN, ring, p);
    } else {
        const int64_t i = t - B;
        uint32_t h[4];
        sha3_256(h, ct + i * P.ct, P.ct, p);
        store_words(hct + i * 32, h, p);
    }
}

// Decapsulation, after the decryption: m' from its bits, kr = G(m' | H(pk))
// with H(pk) from the sk, secret from kr[32:64], b of the pk inside the sk to
// V for the re-encryption, and the instance's mismatch flag cleared (pairs
// [0, B)).  With hct set, pairs [B, 2B) compute H(ct) beside it (the
// decapsulation of keys whose A is resident has no matrix sponge to run it
// next to).  With skey set, instance t's sk is row skey[t] of sk.
template <class SH, bool SHARED>
__global__ __launch_bounds__(64) void dec_front_kernel(KemParams P, const uint16_t *mbits, const uint8_t *sk,
                                                       uint8_t *buf, uint8_t *kr, uint16_t *S, uint16_t *V,
                                                       uint32_t *diff, int64_t B, const uint8_t *ct, uint8_t *hct,
                                                       const int32_t *skey)
{
    TMVP_PAIR(0, SHARED);
    TMVP_RING;
    if (t >= (hct ? 2 * B : B)) return;
    if (t >= B) {
        const int64_t i = t - B;
        uint32_t h[4];
        sha3_256(h, ct + i * P.ct, P.ct, p);
        store_words(hct + i * 32, h, p);
        return;
    }
    if (p == 0) diff[t] = 0; // set by the re-encryption's compare-packs below
    uint32_t m[4];
    // this lane's 32 bits of each message word: bits 64w + 32p + j
    const uint32_t *mb = reinterpret_cast<const uint32_t *>(mbits + t * kN + 32 * p); // bit k in uint16 k
#pragma unroll
    for (int w = 0; w < 4; w++) {
        uint32_t x = 0;
#pragma unroll
        for (int j = 0; j < 16; j++) {
            const uint32_t two = mb[32 * w + j];
            x |= ((two & 1u) << (2 * j)) | (((two >> 16) & 1u) << (2 * j + 1));
        }
        m[w] = x;
    }
    uint32_t h[4], coins[4];
    const uint8_t *skt = sk + (skey ? (int64_t)skey[t] : t) * P.sk;
    load_words(h, skt + P.sk - 64, p);
    hash_g(m, h, buf + t * 64, kr + t * 64, coins, p);
    secret_stream<SH::MU>(P, coins, S + t * P.l * kN, ring, p);
    unpack_b<SH::EP>(P, skt + P.indcpa_sk, V + t * P.l * kN, p);
}

// ---------------------------------------------------------------- codecs

// One thread per (instance, chunk of 64 coefficients), which is exactly W
// 64-bit words of a W-bit little-endian bit stream (LSB first, as every
// reference codec: S/src/pack.cu:1-213, SB/src/pack.cu:182-467).  W is a
// template argument so every shift and word index is a constant.
// kXfSk2 is the Sable secret-key code on unpacking, ((x ^ 2) - 2)
// (SB/src/pack.cu:366-377).
enum Xf : int { kXfNone = 0, kXfSk2 = 1 };

// One chunk: 64 coefficients at s -> W 64-bit words.
template <int W> __device__ __forceinline__ void pack_chunk(const uint4 *s, uint64_t (&words)[W])
{
    constexpr uint32_t mask = (1u << W) - 1u;
#pragma unroll
    for (int k = 0; k < W; k++) words[k] = 0;
#pragma unroll
    for (int q = 0; q < 8; q++) {
        const uint4 v = s[q];
        const uint32_t e[8] = {v.x & 0xffffu, v.x >> 16, v.y & 0xffffu, v.y >> 16,
                               v.z & 0xffffu, v.z >> 16, v.w & 0xffffu, v.w >> 16};
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int bit = (8 * q + j) * W, wi = bit >> 6, o = bit & 63;
            const uint64_t x = e[j] & mask;
            words[wi] |= x << o;
            if (o + W > 64) words[wi + 1] |= x >> (64 - o);
        }
    }
}

// With diff set, nothing is written: the packed words are compared with those
// already at dst, and a mismatch sets diff[t] to 1 (decapsulation's check of
// the re-encryption against the ciphertext).
template <int W>
__global__ __launch_bounds__(256) void pack_kernel(const uint16_t *src, int64_t src_stride, uint8_t *dst,
                                                   int64_t dst_stride, int dst_off, int chunks, int64_t B,
                                                   uint32_t *diff)
{
    const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (gid >= B * chunks) return;
    const int64_t t = gid / chunks;
    const int c = (int)(gid - t * chunks);
    uint64_t words[W];
    pack_chunk<W>(reinterpret_cast<const uint4 *>(src + t * src_stride + c * 64), words);
    uint64_t *d = reinterpret_cast<uint64_t *>(dst + t * dst_stride + dst_off + (int64_t)c * W * 8);
    if (diff) {
        uint64_t x = 0;
#pragma unroll
        for (int k = 0; k < W; k++) x |= d[k] ^ words[k];
        if (x) atomicOr(diff + t, 1u);
        return;
    }
#pragma unroll
    for (int k = 0; k < W; k++) d[k] = words[k];
}

// Decapsulation's check of the whole re-encryption in one launch: 4L chunks
// of b' (bp, EP bits) against ct[0, pvc) and 4 chunks of v' (vp, ET bits)
// against ct[pvc, ...); a mismatch sets diff[t] (S/src/cuda_kernel.cu:414,
// :442, :445).
template <int EP, int ET>
__global__ __launch_bounds__(256) void dec_compare_kernel(const uint16_t *bp, const uint16_t *vp, const uint8_t *ct,
                                                          int64_t ct_stride, int pvc, uint32_t *diff, int l, int64_t B)
{
    const int cv = 4 * l;
    const int chunks = cv + 4;
    const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (gid >= B * chunks) return;
    const int64_t t = gid / chunks;
    const int c = (int)(gid - t * chunks);
    uint64_t x = 0;
    if (c < cv) {
        uint64_t w[EP];
        pack_chunk<EP>(reinterpret_cast<const uint4 *>(bp + (t * cv + c) * 64), w);
        const uint64_t *d = reinterpret_cast<const uint64_t *>(ct + t * ct_stride + (int64_t)c * EP * 8);
#pragma unroll
        for (int k = 0; k < EP; k++) x |= d[k] ^ w[k];
    } else {
        uint64_t w[ET];
        pack_chunk<ET>(reinterpret_cast<const uint4 *>(vp + t * kN + (c - cv) * 64), w);
        const uint64_t *d = reinterpret_cast<const uint64_t *>(ct + t * ct_stride + pvc + (int64_t)(c - cv) * ET * 8);
#pragma unroll
        for (int k = 0; k < ET; k++) x |= d[k] ^ w[k];
    }
    if (x) atomicOr(diff + t, 1u);
}

// One chunk: W 64-bit words at s -> 64 coefficients at d.
template <int W, int XF> __device__ __forceinline__ void unpack_chunk(const uint64_t *s, uint4 *d)
{
    constexpr uint32_t mask = (1u << W) - 1u;
    uint64_t words[W];
#pragma unroll
    for (int k = 0; k < W; k++) words[k] = s[k];
#pragma unroll
    for (int q = 0; q < 8; q++) {
        uint32_t e[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int bit = (8 * q + j) * W, wi = bit >> 6, o = bit & 63;
            uint64_t x = words[wi] >> o;
            if (o + W > 64) x |= words[wi + 1] << (64 - o);
            uint32_t v = (uint32_t)x & mask;
            if (XF == kXfSk2) v = ((v ^ 2u) - 2u) & 0xffffu;
            e[j] = v;
        }
        d[q] = make_uint4(e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16), e[6] | (e[7] << 16));
    }
}

template <int W, int XF>
__global__ __launch_bounds__(256) void unpack_kernel(const uint8_t *src, int64_t src_stride, int src_off,
                                                     uint16_t *dst, int64_t dst_stride, int chunks, int64_t B)
{
    const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (gid >= B * chunks) return;
    const int64_t t = gid / chunks;
    const int c = (int)(gid - t * chunks);
    unpack_chunk<W, XF>(reinterpret_cast<const uint64_t *>(src + t * src_stride + src_off + (int64_t)c * W * 8),
                        reinterpret_cast<uint4 *>(dst + t * dst_stride + c * 64));
}

// Decapsulation's three decodes in one launch (S/src/cuda_kernel.cu:341-352;
// SB/src/SABLE_indcpa.cu:422-440): per instance 4L chunks of s from the sk (WS
// bits, or the Sable 2-bit code), 4L chunks of b' (WB bits) and 4 chunks of
// c_m (WC bits) from the ct.  Used where nothing runs beside the decryption
// (A resident); beside the matrix sponge, three launches measured faster.
// With skey set, instance t's sk is row skey[t] of sk (a key store).
template <int WS, int XS, int WB, int WC>
__global__ __launch_bounds__(256) void dec_unpack_kernel(const uint8_t *sk, int64_t sk_stride, const uint8_t *ct,
                                                         int64_t ct_stride, int pvc, uint16_t *S, uint16_t *Bp,
                                                         uint16_t *Cm, int l, int64_t B, const int32_t *skey)
{
    const int cv = 4 * l; // chunks of one polynomial vector
    const int chunks = 2 * cv + 4;
    const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (gid >= B * chunks) return;
    const int64_t t = gid / chunks;
    const int c = (int)(gid - t * chunks);
    if (c < cv)
        unpack_chunk<WS, XS>(reinterpret_cast<const uint64_t *>(sk + (skey ? (int64_t)skey[t] : t) * sk_stride +
                                                                (int64_t)c * WS * 8),
                             reinterpret_cast<uint4 *>(S + (t * cv + c) * 64));
    else if (c < 2 * cv)
        unpack_chunk<WB, kXfNone>(reinterpret_cast<const uint64_t *>(ct + t * ct_stride + (int64_t)(c - cv) * WB * 8),
                                  reinterpret_cast<uint4 *>(Bp + (t * cv + c - cv) * 64));
    else
        unpack_chunk<WC, kXfNone>(
            reinterpret_cast<const uint64_t *>(ct + t * ct_stride + pvc + (int64_t)(c - 2 * cv) * WC * 8),
            reinterpret_cast<uint4 *>(Cm + t * kN + (c - 2 * cv) * 64));
}

// Up to three gathers of one batch in one launch: segment g copies words[g]
// 8-byte words per instance, dst[g] + t * dst_stride[g] <- src[g] +
// keys[t] * src_stride[g] (key ids checked by the caller).  Unused segments
// have zero words.
struct GatherSet {
    const uint8_t *src[3];
    int64_t src_stride[3];
    uint8_t *dst[3];
    int64_t dst_stride[3];
    int words[3];
};

__global__ __launch_bounds__(256) void gather_kernel(GatherSet G, const int32_t *keys, int64_t B)
{
    const int total = G.words[0] + G.words[1] + G.words[2];
    const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (gid >= B * total) return;
    const int64_t t = gid / total;
    int k = (int)(gid - t * total);
    const uint8_t *src;
    uint8_t *dst;
    const int64_t key = keys[t];
    if (k < G.words[0]) {
        src = G.src[0] + key * G.src_stride[0];
        dst = G.dst[0] + t * G.dst_stride[0];
    } else if (k < G.words[0] + G.words[1]) {
        k -= G.words[0];
        src = G.src[1] + key * G.src_stride[1];
        dst = G.dst[1] + t * G.dst_stride[1];
    } else {
        k -= G.words[0] + G.words[1];
        src = G.src[2] + key * G.src_stride[2];
        dst = G.dst[2] + t * G.dst_stride[2];
    }
    reinterpret_cast<uint64_t *>(dst)[k] = reinterpret_cast<const uint64_t *>(src)[k];
}

// ---------------------------------------------------------------- hashing steps (one lane pair per instance)

// H(pk) of each public key (for a key store).
__global__ __launch_bounds__(64) void hash_pk_kernel(KemParams P, const uint8_t *pk, uint8_t *hpk, int64_t B)
{
    TMVP_PAIR(0, false);
    if (t >= B) return;
    uint32_t h[4];
    sha3_256(h, pk + t * P.pk, P.pk, p);
    store_words(hpk + t * 32, h, p);
}

// GenMatrix from the 32-byte seed at seed + t * stride (for a key store).
template <class SH>
__global__ __launch_bounds__(64) void matrix_kernel(KemParams P, const uint8_t *seed, int64_t stride, uint16_t *A,
                                                    int64_t B)
{
    TMVP_PAIR(0, false);
    TMVP_RING;
    if (t >= B) return;
    uint32_t m[4];
    load_words(m, seed + t * stride, p);
    gen_matrix<SH::EQ>(P, m, A + t * P.l * P.l * kN, ring, p);
}

// Key generation, last step: b (bp, EP bits) packed into the pk and the sk's
// copy of it, then H(pk) into the sk.
template <int EP, bool SHARED>
__global__ __launch_bounds__(64) void kp_hash_kernel(KemParams P, uint8_t *pk, uint8_t *sk, int64_t B,
                                                     const uint16_t *bp)
{
    TMVP_PAIR(0, SHARED);
    if (t >= B) return;
    pack_half<EP, false>(bp + t * P.l * kN, pk + t * P.pk, 4 * P.l, p, sk + t * P.sk + P.indcpa_sk);
    wave_fence_global(); // H(pk) reads both lanes' words
    uint32_t h[4];
    sha3_256(h, pk + t * P.pk, P.pk, p);
    store_words(sk + t * P.sk + P.sk - 64, h, p);
}

// Encapsulation, last step: with EP > 0 the ciphertext is first packed from
// b' (bp, EP bits) and v' (vp, ET bits) (S/src/cuda_kernel.cu:133, :178);
// then kr[32:] = H(ct), ss = H(kr) (:185-186).
template <int EP, int ET, bool SHARED>
__global__ __launch_bounds__(64) void enc_hash2_kernel(KemParams P, uint8_t *ct, uint8_t *kr, uint8_t *ss, int64_t B,
                                                       const uint16_t *bp, const uint16_t *vp)
{
    TMVP_PAIR(0, SHARED);
    if (t >= B) return;
    if constexpr (EP > 0) {
        pack_half<EP, false>(bp + t * P.l * kN, ct + t * P.ct, 4 * P.l, p);
        pack_half<ET, false>(vp + t * kN, ct + t * P.ct + P.pvc, 4, p);
        wave_fence_global(); // H(ct) reads both lanes' words
    }
    uint32_t h[4], k[8], s[4], k0[4];
    sha3_256(h, ct + t * P.ct, P.ct, p);
    load_words(k0, kr + t * 64, p);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        k[i] = k0[i];
        k[4 + i] = h[i];
    }
    sha3_256_words<8>(s, k, p);
    store_words(ss + t * 32, s, p);
}

// Decapsulation, last step: diff[t] is the outcome of comparing ct with the
// re-encryption (set while packing it), kr[32:] = H(ct) (computed
// beforehand); replace kr[0:32] by z on mismatch, ss = H(kr).  fail[t]
// records the outcome.  KEYED: instance t's sk is row skey[t] of sk (a template
// flag, as in enc_front_kernel: the runtime test cost the non-keyed kernel
// 0.7 us at 16384 instances).
template <bool KEYED, bool SHARED>
__global__ __launch_bounds__(64) void dec_fin_kernel(KemParams P, const uint32_t *diff, const uint8_t *sk,
                                                     const uint8_t *hct, const uint8_t *kr, uint8_t *ss, uint8_t *fail,
                                                     int64_t B, const int32_t *skey)
{
    TMVP_PAIR(0, SHARED);
    if (t >= B) return;
    const uint32_t mask = 0u - (uint32_t)(diff[t] != 0); // all ones on mismatch, in both lanes
    uint32_t h[4], k[8], s[4], k0[4], z[4];
    load_words(h, hct + t * 32, p);
    load_words(k0, kr + t * 64, p);
    load_words(z, sk + (KEYED ? (int64_t)skey[t] : t) * P.sk + P.sk - 32, p);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        k[i] = k0[i] ^ (mask & (k0[i] ^ z[i]));
        k[4 + i] = h[i];
    }
    sha3_256_words<8>(s, k, p);
    store_words(ss + t * 32, s, p);
    if (fail && p == 0) fail[t] = (uint8_t)(mask & 1u);
}

// ---------------------------------------------------------------- one-launch key generation, encapsulation and decapsulation
//
// The MFMA backend runs each operation as ONE launch in which the products and
// the hashes overlap the matrix sponge.  A workgroup of 16 waves holds up to 32
// instances in each of G = 2 or 4 groups (fused_launch below; G = 2 here; the
// waves go round-robin over the CU's four SIMDs, so each SIMD holds one sponge
// wave and three MFMA waves):
//   waves 0, 1   the matrix sponges (GenMatrix) of instances 0-31 and 32-63;
//   waves 2, 3   the rest of those instances' hashing: the secret, and at the
//                end the hash over the packed output (H(pk) / H(ct)),
//                absorbed row by row as the products finish the rows;
//   waves 4-15   the products on the matrix cores, in jobs of one to three
//                output rows (rows_body), each as soon as its polynomials and
//                the secret exist.  In encapsulation waves 6 and 7, which
//                share their SIMDs with the secret waves rather than the
//                matrix sponges, first hash the public keys.
// Small batches run the kernels further down (tmvp_kem_form.h).
// A row's polynomials come out of the matrix stream in order (encapsulation,
// A s': row i is A[i][0..L); key generation, A^T s: row j is A[0..L)[j], so
// the rows finish with the stream's last L polynomials), and the hash over
// the output starts with the first finished row while the stream still runs.
//
// What bounds a call: the chain of permutations of one instance (encapsulation
// of Saber: 23 of the matrix stream, then 6 over the last row and the shared
// key, at about 5.3 us each), and beside it the products, which get the issue
// slots the sponges leave.  A sponge wave issues an instruction whenever it
// can, so waves that the critical path waits for raise their priority
// (s_setprio).
//
// The matrix goes through memory as the raw stream (a workgroup's share is
// 234 KB for Saber against 160 KB of LDS, and in encapsulation most of it
// exists before the secret that multiplies it); the products spread its
// coefficients as they stage them, and are the only readers, from the L2 or
// the MALL soon after.
//
// Progress goes through LDS counters, each raised by one wave or counted up
// by the MFMA waves (wait_for / publish / fused_leave).  Every wait is on a
// counter raised by waves that do not themselves wait on the waiter, and
// every wave raises its counters to their final values even when it has no
// instances, so every wait ends; a bound on each wait (about 0.2 s) sets the
// status word instead of hanging if that ever failed.
constexpr int kFusedThreads = 1024; // 16 waves: G matrix waves, G secret waves, then the MFMA waves
template <int G> constexpr int kFusedInst = kGroupInst * G; // instances of a workgroup at most
template <int G> constexpr int kFusedMfma = 16 - 2 * G;
constexpr int kMaxGroups = 4;
constexpr int kSpinLimit = 1 << 22;
constexpr int kDone = 1 << 20; // a counter's value when its wave has no instances

constexpr int kFusedJobs = 10; // product jobs: at most those of key generation, L = 4
constexpr int kFusedGrab = 2; // instances an MFMA wave takes from a job at a time

struct FusedSync {
    int mat[kMaxGroups];          // polynomials of A written by matrix wave w (published at the milestones below)
    int sec[kMaxGroups];          // secret wave w: 1 once the secret and the message are written
    int hpk[kMaxGroups];          // encapsulation: 1 once H(pk) of group w's instances is in LDS
    int next[kFusedJobs];  // next unclaimed instance of each product job
    int done[kFusedJobs];  // MFMA waves that have left each job (all its instances finished at kFusedMfma)
};

__device__ __forceinline__ int peek(const int *f)
{
    return __hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ __forceinline__ void wait_for(const int *f, int v, int *status)
{
    int n = 0;
    while (peek(f) < v) {
        __builtin_amdgcn_s_sleep(2);
        if (++n == kSpinLimit) {
            *status = 1;
            break;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

__device__ __forceinline__ void publish(int *f, int v)
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __hip_atomic_store(f, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// The matrix stream of one instance to raw (S::kMatrix bytes), squeezed words
// as they come; publishes `flag`, the number of whole polynomials written, at
// every count some job waits for: both need every i L (key generation's term
// i - 1 of all rows, encapsulation's row i - 1), and key generation's row r ends
// with polynomial (L - 1) L + r.
template <class S, bool KEYGEN> __device__ __forceinline__ bool is_milestone(int polys, int now)
{
    constexpr int L = S::L;
    return now / L > polys / L || (KEYGEN && now > polys && now >= (L - 1) * L);
}

template <class S, bool KEYGEN>
__device__ __forceinline__ void fused_matrix(const uint32_t (&seed)[4], uint8_t *raw, Half p, int *flag)
{
    constexpr int L = S::L, RB = kShake128Rate / 8, PW = S::kPoly / 8, NW = L * L * PW;
    uint32_t st[25];
    absorb_words(st, seed, kShake128Rate, kShakeDS, p);
    uint32_t *w = reinterpret_cast<uint32_t *>(raw) + p;
    int polys = 0;
    for (int k = 0; k < NW / RB; k++) {
        f1600(st, p);
#pragma unroll
        for (int i = 0; i < RB; i++) w[2 * i] = st[i];
        w += 2 * RB;
        const int now = (k + 1) * RB / PW;
        if (is_milestone<S, KEYGEN>(polys, now)) publish(flag, now);
        polys = now;
    }
    if constexpr (NW % RB != 0) {
        f1600(st, p);
#pragma unroll
        for (int i = 0; i < NW % RB; i++) w[2 * i] = st[i];
    }
    publish(flag, L * L);
}

// One product job over the workgroup's instances.  The MFMA waves claim
// kFusedGrab instances at a time, so waves sharing a SIMD with a busy sponge
// take fewer; a wave that finds nothing left counts itself out of the job
// (fused_leave), and the job is finished when all kFusedMfma have.
__device__ __forceinline__ void fused_leave(FusedSync &sy, int job)
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    if ((threadIdx.x & 63) == 0) __hip_atomic_fetch_add(&sy.done[job], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <class S, int NT, int NR, bool B, bool TR, RowOp OP, SecretForm SF>
__device__ __forceinline__ void fused_job(FusedSync &sy, int job, int nloc, const RowJob &J, int row0, int term0,
                                          uint8_t *slices)
{
    for (;;) {
        int i = 0;
        if ((threadIdx.x & 63) == 0)
            i = __hip_atomic_fetch_add(&sy.next[job], kFusedGrab, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        i = __builtin_amdgcn_readfirstlane(i);
        if (i >= nloc) break;
        rows_body<S, NT, NR, B, TR, OP, SF>(J, row0, term0, i, 1, i + kFusedGrab < nloc ? i + kFusedGrab : nloc, slices);
    }
    fused_leave(sy, job);
}

// A product job that the hashing waits for, such as the last, which starts when
// the matrix sponges have ended: an even split without claims, so that each
// wave loads its next instance while it multiplies the current one.  The priority
// stays: what a wave does afterwards is poll for the next such job (lowered again
// after each, all sets and sizes from 1537 on took within 0.3 % of the same).
template <class S, int G, int NT, int NR, bool B, bool TR, RowOp OP, SecretForm SF>
__device__ __forceinline__ void fused_even(FusedSync &sy, int job, int nloc, const RowJob &J, int row0, int term0,
                                           uint8_t *slices, int k)
{
    __builtin_amdgcn_s_setprio(3);
    rows_body<S, NT, NR, B, TR, OP, SF>(J, row0, term0, k, kFusedMfma<G>, nloc, slices);
    fused_leave(sy, job);
}

// The LDS of a workgroup.
template <class S, int G> struct FusedLds {
    FusedSync sync;
    __attribute__((aligned(16))) uint32_t rc[kRcDwords];     // round constants (fill_rc)
    uint32_t hpk[kFusedInst<G> * 8];                            // H(pk) per local instance (encapsulation)
    uint32_t msg[kFusedInst<G> * 8];                            // the message per local instance
    uint32_t buf[G][(S::MU == 6 || S::MU == 10) ? 32 * kRingDwords : 1]; // secret waves' stream buffers
    __attribute__((aligned(16))) uint8_t mfma[kFusedMfma<G>][2 * kRowSlice<3>]; // MFMA waves' slices
};

// The counters, the message words and the round constants, before the roles start.
template <class S, int G> __device__ __forceinline__ void fused_init(FusedLds<S, G> &M, int wave)
{
    if (threadIdx.x < sizeof(FusedSync) / 4) reinterpret_cast<int *>(&M.sync)[threadIdx.x] = 0;
    if (threadIdx.x < kFusedInst<G> * 8) M.msg[threadIdx.x] = 0;
    if (wave == 0) fill_rc(M.rc);
    __syncthreads();
}

// Key generation's jobs: the heads, terms i .. i + kTerms - 1 of rows h kRows ..
// + kRows - 1 (i + kTerms < L), then the tails, the rows' last terms.
template <int L, int G> struct KeygenJobs {
    static constexpr int kHalves = L == 4 ? 2 : 1, kRows = L / kHalves, kTerms = G == 2 ? 1 : L - 1;
    static __device__ __forceinline__ constexpr int head(int i, int h) { return i / kTerms * kHalves + h; }
    static __device__ __forceinline__ constexpr int tail(int r) { return (L - 1) / kTerms * kHalves + r; }
};
static_assert(3 * 2 + 4 <= kFusedJobs, "jobs of L = 4");

template <class S, int G>
__global__ __launch_bounds__(kFusedThreads) void kp_fused_kernel(const uint8_t *seeds, uint8_t *pk, uint8_t *sk,
                                                                 KemWorkspace W, int64_t B, int per, int *status)
{
    constexpr int L = S::L, EP = S::EP;
    __shared__ FusedLds<S, G> M;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int64_t base = (int64_t)blockIdx.x * per;
    const int nloc = (int)(B - base < per ? B - base : per);
    fused_init(M, wave);
    const Half p{lane & 1, M.rc, G > 2};
    uint8_t *const raw = reinterpret_cast<uint8_t *>(W.A), *const sec = reinterpret_cast<uint8_t *>(W.s);
    if (wave < 2 * G) {
        const int grp = wave & (G - 1), li = 32 * grp + (lane >> 1);
        const int64_t t = base + li;
        if (32 * grp >= nloc) {
            publish(wave < G ? &M.sync.mat[grp] : &M.sync.sec[grp], kDone);
            return;
        }
        if (li >= nloc) return; // lane 0 of the wave has an instance and publishes
        uint8_t *pkt = pk + t * S::kPk, *skt = sk + t * S::kSk;
        if (wave < G) {
            // seed_A' = SHAKE-128(seed_A) to the pk tail and the sk's copy of the pk, then GenMatrix
            uint32_t m[4], st[25];
            load_words(m, seeds + t * 96, p);
            absorb_words(st, m, kShake128Rate, kShakeDS, p);
            f1600(st, p);
            const uint32_t sa[4] = {st[0], st[1], st[2], st[3]};
            store_words(pkt + S::kPvc, sa, p);
            store_words(skt + S::kSec + S::kPvc, sa, p);
            fused_matrix<S, true>(sa, raw + t * S::kMatrix, p, &M.sync.mat[grp]);
            return;
        }
        // the secret, packed into the sk, and z
        uint32_t m[4];
        load_words(m, seeds + t * 96 + 32, p);
        uint8_t *s = sec + t * L * kN;
        secret_bytes<S>(m, s, M.buf[grp] + (lane >> 1) * kRingDwords, p);
        publish(&M.sync.sec[grp], 1);
        pack_secret<S>(s, skt, p);
        load_words(m, seeds + t * 96 + 64, p);
        store_words(skt + S::kSk - 32, m, p);
        // b row by row into the pk and the sk's copy, and H(pk) over it as it grows
        uint32_t st[25];
#pragma unroll
        for (int i = 0; i < 25; i++) st[i] = 0;
        int done = 0;
        for (int r = 0; r < L; r++) {
            wait_for(&M.sync.done[KeygenJobs<L, G>::tail(r)], kFusedMfma<G>, status);
            pack_half<EP, false>(W.v1 + (t * L + r) * kN, pkt + r * EP * 32, 4, p, skt + S::kSec + r * EP * 32);
            wave_fence_global();
            absorb_upto<kSha3_256Rate>(st, pkt, done, (r + 1) * EP * 32, p);
        }
        // the pk tail (seed_A') was written by the matrix wave before the rows' products began
        absorb_upto<kSha3_256Rate>(st, pkt, done, S::kPk, p);
        absorb_final<kSha3_256Rate>(st, pkt, S::kPk, kSha3DS, p);
        f1600(st, p);
        const uint32_t h[4] = {st[0], st[1], st[2], st[3]};
        store_words(skt + S::kSk - 64, h, p);
        return;
    }
    // Products: b = round(A^T s).  Term i of every row comes with the stream's
    // polynomials i L .. i L + L - 1, so the first terms go ahead as heads (of all
    // rows at once, for L = 4 two of two rows), which sum into the rows' outputs,
    // and each row's tail adds its last term and rounds.  With two groups a head
    // is one term, so that it ends while the next term's polynomials are being
    // squeezed, a row ends soon after its last polynomial, and H(pk) takes the
    // first rows while the stream runs; the tails are split evenly, since claims
    // of two one-term instances wait for their loads each time.  (Heads of L - 1
    // terms started with the stream's last row, and every row ended after the
    // stream: Saber, 8192 instances 190 -> 185 us, 16384 198 -> 190; FireSaber 298 ->
    // 285, 304 -> 300; 33 instances a workgroup 176 -> 163 and 276 -> 256.)  With four groups, whose
    // sponges leave the products less, the second pass over the sums costs more
    // than the wait: 32768 FireSaber instances 482 us, 514 term by term.
    const int k = wave - 2 * G;
    RowJob J{};
    J.a = raw + base * S::kMatrix;
    J.s = sec + base * L * kN;
    J.out = W.v1 + base * L * kN;
    J.status = status;
    using Jobs = KeygenJobs<L, G>;
    constexpr int R = Jobs::kRows, T = Jobs::kTerms;
    for (int g = 0; g < G; g++) wait_for(&M.sync.sec[g], 1, status);
    for (int i = 0; i < L - 1; i += T) {
        for (int g = 0; g < G; g++) wait_for(&M.sync.mat[g], (i + T) * L, status);
        for (int h = 0; h < Jobs::kHalves; h++) {
            const int job = Jobs::head(i, h);
            if (i == 0) {
                fused_job<S, T, R, false, true, kRowSum, kSecBytes>(M.sync, job, nloc, J, h * R, 0, M.mfma[k]);
            } else {
                wait_for(&M.sync.done[Jobs::head(i - 1, h)], kFusedMfma<G>, status);
                fused_job<S, T, R, false, true, kRowAdd, kSecBytes>(M.sync, job, nloc, J, h * R, i, M.mfma[k]);
            }
        }
    }
    for (int r = 0; r < L; r++) {
        for (int g = 0; g < G; g++) wait_for(&M.sync.mat[g], (L - 1) * L + r + 1, status);
        wait_for(&M.sync.done[Jobs::head(L - 1 - T, r / R)], kFusedMfma<G>, status); // the row's sum, by whichever waves
        if (G > 2 && r < L - 1)
            fused_job<S, 1, 1, false, true, kRowAddRound, kSecBytes>(M.sync, Jobs::tail(r), nloc, J, r, L - 1, M.mfma[k]);
        else
            fused_even<S, G, 1, 1, false, true, kRowAddRound, kSecBytes>(M.sync, Jobs::tail(r), nloc, J, r, L - 1, M.mfma[k], k);
    }
}

// The encryption's products, jobs job0..: the first R rows (one or two) of A s'
// with v' = b . s', then the other rows.
template <int R> __device__ __forceinline__ constexpr int enc_job_of(int row) { return row < R ? 0 : row - R + 1; }

template <class S, int G, int R>
__device__ __forceinline__ void enc_products(FusedSync &sy, int job0, int nloc, const RowJob &J, uint8_t *slices, int k,
                                             int *status)
{
    // The rows from kEven on are split evenly and go before the sponges on their
    // SIMDs.  Beside the last row, with three rows and two groups also the one
    // before it, whose hashing ends just before the last row needs it (16384
    // Saber encapsulations 194 -> 189 us, Sable type 2 168 -> 161); with four rows
    // it would hold up the matrix sponges (FireSaber 269 -> 282).
    constexpr int L = S::L, kEven = G == 2 && L == 3 ? L - 2 : L - 1;
    for (int g = 0; g < G; g++) wait_for(&sy.sec[g], 1, status);
    for (int g = 0; g < G; g++) wait_for(&sy.mat[g], R * L, status);
    fused_job<S, L, R + 1, true, false, kRowRound, kSecBytes>(sy, job0, nloc, J, 0, 0, slices);
    for (int r = R; r < L; r++) {
        for (int g = 0; g < G; g++) wait_for(&sy.mat[g], (r + 1) * L, status);
        if (r < kEven)
            fused_job<S, L, 1, false, false, kRowRound, kSecBytes>(sy, job0 + enc_job_of<R>(r), nloc, J, r, 0, slices);
        else
            fused_even<S, G, L, 1, false, false, kRowRound, kSecBytes>(sy, job0 + enc_job_of<R>(r), nloc, J, r, 0, slices, k);
    }
}

template <class S, int G>
__global__ __launch_bounds__(kFusedThreads) void enc_fused_kernel(const uint8_t *pk, const uint8_t *rnd, uint8_t *ct,
                                                                  uint8_t *ss, KemWorkspace W, int64_t B, int per, int *status)
{
    constexpr int L = S::L, EP = S::EP, ET = S::ET;
    __shared__ FusedLds<S, G> M;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int64_t base = (int64_t)blockIdx.x * per;
    const int nloc = (int)(B - base < per ? B - base : per);
    fused_init(M, wave);
    const Half p{lane & 1, M.rc, G > 2};
    uint8_t *const raw = reinterpret_cast<uint8_t *>(W.A), *const sec = reinterpret_cast<uint8_t *>(W.s);
    if (wave < 2 * G) {
        const int grp = wave & (G - 1), li = 32 * grp + (lane >> 1);
        const int64_t t = base + li;
        if (32 * grp >= nloc) {
            publish(wave < G ? &M.sync.mat[grp] : &M.sync.sec[grp], kDone);
            return;
        }
        if (li >= nloc) return; // lane 0 of the wave has an instance and publishes
        if (wave < G) {
            uint32_t m[4];
            load_words(m, pk + t * S::kPk + S::kPvc, p);
            fused_matrix<S, false>(m, raw + t * S::kMatrix, p, &M.sync.mat[grp]);
            return;
        }
        // m = H(rnd), (K, r) = G(m | H(pk)), the secret from r
        uint32_t r[4], m[4], kb[8], kk[8];
        load_words(r, rnd + t * 32, p);
        sha3_256_words<4>(m, r, p);
#pragma unroll
        for (int i = 0; i < 4; i++) M.msg[li * 8 + 2 * i + p] = m[i];
        wait_for(&M.sync.hpk[grp], 1, status);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            kb[i] = m[i];
            kb[4 + i] = M.hpk[li * 8 + 2 * i + p];
        }
        sha3_512_words(kk, kb, p);
        const uint32_t coins[4] = {kk[4], kk[5], kk[6], kk[7]};
        secret_bytes<S>(coins, sec + t * L * kN, M.buf[grp] + (lane >> 1) * kRingDwords, p);
        publish(&M.sync.sec[grp], 1);
        // the ciphertext row by row, and H(ct) over it as it grows
        uint8_t *c = ct + t * S::kCt;
        uint32_t st[25];
#pragma unroll
        for (int i = 0; i < 25; i++) st[i] = 0;
        int done = 0;
        for (int row = 0; row < L; row++) {
            wait_for(&M.sync.done[enc_job_of<1>(row)], kFusedMfma<G>, status);
            pack_half<EP, false>(W.v1 + (t * L + row) * kN, c + row * EP * 32, 4, p);
            if (row == L - 1) pack_half<ET, false>(W.poly + t * kN, c + S::kPvc, 4, p); // v' came with row 0
            wave_fence_global();
            absorb_upto<kSha3_256Rate>(st, c, done, row == L - 1 ? S::kCt : (row + 1) * EP * 32, p);
        }
        absorb_final<kSha3_256Rate>(st, c, S::kCt, kSha3DS, p);
        f1600(st, p);
        // ss = H(K | H(ct))
#pragma unroll
        for (int i = 0; i < 4; i++) kb[4 + i] = st[i];
#pragma unroll
        for (int i = 0; i < 4; i++) kb[i] = kk[i];
        uint32_t sv[4];
        sha3_256_words<8>(sv, kb, p);
        store_words(ss + t * 32, sv, p);
        return;
    }
    const int k = wave - 2 * G;
    constexpr int kHash0 = G == 2 ? 2 : 0;
    if (k >= kHash0 && k < kHash0 + G) {
        // H(pk) of group k - kHash0's instances, for the secret waves.  With two
        // groups waves 6 and 7 share their SIMDs with the secret waves (waves go
        // round-robin over the four SIMDs), which wait for this, rather than
        // with the matrix sponges, and go before them; with four the permutation sets
        // the priority itself (f1600's `shared`).
        const int li = 32 * (k - kHash0) + (lane >> 1);
        if (li < nloc) {
            if constexpr (G == 2) __builtin_amdgcn_s_setprio(3);
            uint32_t h[4];
            sha3_256(h, pk + (base + li) * S::kPk, S::kPk, p);
#pragma unroll
            for (int i = 0; i < 4; i++) M.hpk[li * 8 + 2 * i + p] = h[i];
            if constexpr (G == 2) __builtin_amdgcn_s_setprio(0);
        }
        publish(&M.sync.hpk[k - kHash0], 1);
    }
    RowJob J{};
    J.a = raw + base * S::kMatrix;
    J.b = pk + base * S::kPk;
    J.bstride = S::kPk;
    J.s = sec + base * L * kN;
    J.out = W.v1 + base * L * kN;
    J.out2 = W.poly + base * kN;
    J.msg = M.msg;
    J.status = status;
    enc_products<S, G, 1>(M.sync, 0, nloc, J, M.mfma[k], k, status);
}

// Decapsulation in one launch.  The MFMA waves run the decryption (job 0: m' =
// dec(b' . s, c_m), from the packed sk and ct), and after the secret waves
// have turned m' into the re-encryption's secret s'', its products: rows 0 and
// 1 of A s'' with v'' = b . s'' (job 1; m' folded in) and the later rows.  The
// secret waves hash the ciphertext, as far as they get before m' is there and
// the rest while the products run, compare each finished row with the
// ciphertext (packing it in registers), and the final hash takes K' or z by
// the outcome.  The sk's pk supplies the matrix seed and b.
template <class S, int G>
__global__ __launch_bounds__(kFusedThreads) void dec_fused_kernel(const uint8_t *ct, const uint8_t *sk, uint8_t *ss,
                                                                  uint8_t *fail, KemWorkspace W, int64_t B, int per, int *status)
{
    constexpr int L = S::L, EP = S::EP, ET = S::ET;
    __shared__ FusedLds<S, G> M;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int64_t base = (int64_t)blockIdx.x * per;
    const int nloc = (int)(B - base < per ? B - base : per);
    fused_init(M, wave);
    const Half p{lane & 1, M.rc, G > 2};
    uint8_t *const raw = reinterpret_cast<uint8_t *>(W.A), *const sec = reinterpret_cast<uint8_t *>(W.s);
    if (wave < 2 * G) {
        const int grp = wave & (G - 1), li = 32 * grp + (lane >> 1);
        const int64_t t = base + li;
        if (32 * grp >= nloc) {
            publish(wave < G ? &M.sync.mat[grp] : &M.sync.sec[grp], kDone);
            return;
        }
        if (li >= nloc) return; // lane 0 of the wave has an instance and publishes
        const uint8_t *skt = sk + t * S::kSk;
        if (wave < G) {
            uint32_t m[4];
            load_words(m, skt + S::kSec + S::kPvc, p);
            fused_matrix<S, false>(m, raw + t * S::kMatrix, p, &M.sync.mat[grp]);
            return;
        }
        // H(ct) up to the decryption's end
        const uint8_t *c = ct + t * S::kCt;
        uint32_t st[25];
#pragma unroll
        for (int i = 0; i < 25; i++) st[i] = 0;
        int done = 0;
        while (done + kSha3_256Rate <= S::kCt && __builtin_amdgcn_readfirstlane(peek(&M.sync.done[0])) < kFusedMfma<G>)
            absorb_upto<kSha3_256Rate>(st, c, done, done + kSha3_256Rate, p);
        wait_for(&M.sync.done[0], kFusedMfma<G>, status);
        // (K', r') = G(m' | H(pk)), the secret s'' from r'
        uint32_t hpk[4], kb[8], kk[8];
        load_words(hpk, skt + S::kSk - 64, p);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            kb[i] = M.msg[li * 8 + 2 * i + p];
            kb[4 + i] = hpk[i];
        }
        sha3_512_words(kk, kb, p);
        const uint32_t coins[4] = {kk[4], kk[5], kk[6], kk[7]};
        secret_bytes<S>(coins, sec + t * L * kN, M.buf[grp] + (lane >> 1) * kRingDwords, p);
        publish(&M.sync.sec[grp], 1);
        absorb_upto<kSha3_256Rate>(st, c, done, S::kCt, p);
        absorb_final<kSha3_256Rate>(st, c, S::kCt, kSha3DS, p);
        f1600(st, p);
        // the re-encryption against the ciphertext, row by row
        uint32_t diff = 0;
        for (int row = 0; row < L; row++) {
            wait_for(&M.sync.done[1 + enc_job_of<2>(row)], kFusedMfma<G>, status);
            diff |= pack_compare_half<EP>(W.v1 + (t * L + row) * kN, c + row * EP * 32, 4, p);
        }
        diff |= pack_compare_half<ET>(W.poly + t * kN, c + S::kPvc, 4, p);
        diff |= partner(diff);
        // ss = H(K | H(ct)) with K = K' on a match, z otherwise (constant time)
        uint32_t z[4], sv[4];
        load_words(z, skt + S::kSk - 32, p);
        const uint32_t mask = 0u - (uint32_t)(diff != 0);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            kb[i] = kk[i] ^ (mask & (kk[i] ^ z[i]));
            kb[4 + i] = st[i];
        }
        sha3_256_words<8>(sv, kb, p);
        store_words(ss + t * 32, sv, p);
        if (fail && p == 0) fail[t] = (uint8_t)(mask & 1u);
        return;
    }
    const int k = wave - 2 * G;
    RowJob J{};
    J.a = ct + base * S::kCt;
    J.s = sk + base * S::kSk;
    J.cm = ct + base * S::kCt + S::kPvc;
    J.msg = M.msg;
    J.status = status;
    // the decryption, which everything else of this wave's work waits for,
    // before the hash waves on its SIMD
    if (G != 2 || (wave & 2)) __builtin_amdgcn_s_setprio(2);
    fused_job<S, L, 1, false, false, kRowDecrypt, kSecKey>(M.sync, 0, nloc, J, 0, 0, M.mfma[k]);
    __builtin_amdgcn_s_setprio(0);
    // the re-encryption
    J.a = raw + base * S::kMatrix;
    J.b = sk + base * S::kSk + S::kSec;
    J.bstride = S::kSk;
    J.s = sec + base * L * kN;
    J.out = W.v1 + base * L * kN;
    J.out2 = W.poly + base * kN;
    enc_products<S, G, 2>(M.sync, 1, nloc, J, M.mfma[k], k, status);
}

// ---------------------------------------------------------------- the same for small batches
//
// Up to kSmallBatch instances, a workgroup of eight waves takes eight of them,
// with a state on a row of sixteen lanes (tmvp_keccak_row.h), four states a
// wave, so the chain of permutations, which bounds such calls, is 0.6 of its
// length on lane pairs:
//   waves 0, 1   the matrix sponges of instances 0-3 and 4-7;
//   waves 2, 3   their secrets and output hashes;
//   waves 4-7    the products, split evenly; in encapsulation waves 4 and 5
//                first hash the public keys.
// Progress and waits are those of the kernels above.  What passes between
// lanes (the hashes' inputs, the secret's stream, the packed output) goes
// through LDS.
//
// Saber, 512 instances: key generation 105 us (lane pairs 159), encapsulation
// 109 (148), decapsulation 92 (139); one instance: 95, 99 and 85 us (decapsulation
// 130 on lane pairs).  Four product waves measured best (eight: 1 us more, and
// their registers and LDS slices keep a second workgroup off the CU).
constexpr int kSmallMfma = 4;
constexpr int kSmallThreads = 64 * (4 + kSmallMfma);

template <class S> struct SmallLds {
    FusedSync sync;
    __attribute__((aligned(16))) uint32_t rc[kRowRc];
    __attribute__((aligned(16))) uint32_t state[6][4][kRowDwords]; // matrix, secret and H(pk) waves' rows
    uint32_t msg[kSmallInst * 8];                                  // the message per instance
    uint32_t in[kSmallInst][16];                                   // m | H(pk), later K | H(ct)
    uint32_t kr[kSmallInst][16];                                   // K | coins
    uint32_t stream[kSmallInst][S::L * S::MU * 8 + 42];            // the secret's stream, in whole blocks
    uint32_t ct[kSmallInst][S::kCt / 4];                           // the packed output being hashed (a pk is shorter)
    __attribute__((aligned(16))) uint8_t mfma[kSmallMfma][2 * kRowSlice<3>];
    static_assert(S::kCt >= S::kPk, "output buffer");
};

// LDS written by some lanes of the wave, read by others: the wave's LDS
// operations execute in order, so only code motion must be stopped.
__device__ __forceinline__ void row_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <class S> __device__ __forceinline__ void small_init(SmallLds<S> &M, int wave)
{
    if (threadIdx.x < sizeof(FusedSync) / 4) reinterpret_cast<int *>(&M.sync)[threadIdx.x] = 0;
    if (threadIdx.x < kSmallInst * 8) M.msg[threadIdx.x] = 0;
    if (wave == 0) {
        fill_rc(*reinterpret_cast<uint32_t(*)[kRcDwords]>(M.rc));
        if (threadIdx.x < kRowRc - kRcDwords) M.rc[kRcDwords + threadIdx.x] = 0;
    }
    __syncthreads();
}

// fused_matrix on rows: A is the absorbed, unpermuted state.
template <class S, bool KEYGEN>
__device__ __forceinline__ void small_matrix(uint32_t (&A)[5], uint8_t *raw, const Row &row, int *flag)
{
    constexpr int L = S::L, RB = kShake128Rate / 8, PW = S::kPoly / 8, NW = L * L * PW;
    uint32_t *w = reinterpret_cast<uint32_t *>(raw);
    int polys = 0;
    for (int k = 0; k < NW / RB; k++) {
        f1600(A, row);
        row_store<RB>(w, A, row);
        w += 2 * RB;
        const int now = (k + 1) * RB / PW;
        if (is_milestone<S, KEYGEN>(polys, now)) publish(flag, now);
        polys = now;
    }
    if constexpr (NW % RB != 0) {
        f1600(A, row);
        row_store<NW % RB>(w, A, row);
    }
    publish(flag, L * L);
}

// The secret from the absorbed state A: its stream to LDS, then 32
// coefficients a lane (MU dwords of the stream) as int8 to s and, with a key
// to write, packed to sk.
template <class S, bool KEYGEN>
__device__ __forceinline__ void small_secret(uint32_t (&A)[5], uint32_t *stream, uint8_t *s, uint8_t *sk, int sub,
                                             const Row &row)
{
    constexpr int RB = kShake128Rate / 8, NW = S::L * S::MU * 4;
    for (int k = 0; k < NW; k += RB) {
        f1600(A, row);
        row_store<RB>(stream + 2 * k, A, row);
    }
    row_fence();
    for (int u = sub; u < 8 * S::L; u += 16) {
        uint32_t d[S::MU], o[8];
#pragma unroll
        for (int i = 0; i < S::MU; i++) d[i] = stream[u * S::MU + i];
        if constexpr (S::MU == 8) {
#pragma unroll
            for (int q = 0; q < 8; q++) o[q] = cbd8(d[q]);
        } else if constexpr (S::MU == 2) {
#pragma unroll
            for (int q = 0; q < 8; q++) o[q] = cbd2(d[q >> 2] >> (8 * (q & 3)));
        } else {
            cbd32<S::MU>(d, o);
        }
#pragma unroll
        for (int q = 0; q < 8; q++) o[q] = cbd_int8(o[q]);
        uint4 *q4 = reinterpret_cast<uint4 *>(s + 32 * u);
        q4[0] = make_uint4(o[0], o[1], o[2], o[3]);
        q4[1] = make_uint4(o[4], o[5], o[6], o[7]);
        if constexpr (KEYGEN) {
            constexpr int W = S::kSable ? 2 : S::EQ;
            uint32_t w[W];
            pack_int8<W>(o, w);
            uint32_t *dst = reinterpret_cast<uint32_t *>(sk) + u * W;
#pragma unroll
            for (int i = 0; i < W; i++) dst[i] = w[i];
        }
    }
}

// One polynomial of W-bit coefficients at S packed to dst, its LDS copy and
// (not null) dst2, 32 coefficients a lane on eight lanes.
template <int W>
__device__ __forceinline__ void small_pack(const uint16_t *S, uint8_t *dst, uint32_t *copy, uint8_t *dst2, int sub)
{
    if (sub >= 8) return;
    uint32_t w[W];
    pack_coefficients<W>(S + 32 * sub, w);
    uint32_t *d = reinterpret_cast<uint32_t *>(dst) + sub * W, *d2 = reinterpret_cast<uint32_t *>(dst2) + sub * W;
#pragma unroll
    for (int i = 0; i < W; i++) {
        d[i] = w[i];
        copy[sub * W + i] = w[i];
        if (dst2) d2[i] = w[i];
    }
}

// Nonzero where the polynomial at S, packed, differs from the bytes at c.
template <int W> __device__ __forceinline__ uint32_t small_compare(const uint16_t *S, const uint8_t *c, int sub)
{
    if (sub >= 8) return 0;
    uint32_t w[W], x = 0;
    pack_coefficients<W>(S + 32 * sub, w);
    const uint32_t *d = reinterpret_cast<const uint32_t *>(c) + sub * W;
#pragma unroll
    for (int i = 0; i < W; i++) x |= d[i] ^ w[i];
    return x;
}

template <class S, int NT, int NR, bool B, bool TR, RowOp OP, SecretForm SF>
__device__ __forceinline__ void small_job(FusedSync &sy, int job, int nloc, const RowJob &J, int row0, int term0,
                                          uint8_t *slices, int k)
{
    rows_body<S, NT, NR, B, TR, OP, SF>(J, row0, term0, k, kSmallMfma, nloc, slices);
    fused_leave(sy, job);
}

// The encryption's products: the first R rows with v', then the other rows (jobs as in enc_products).
template <class S, int R>
__device__ __forceinline__ void small_products(FusedSync &sy, int job0, int nloc, const RowJob &J, uint8_t *slices, int k,
                                               int *status)
{
    constexpr int L = S::L;
    for (int g = 0; g < 2; g++) wait_for(&sy.sec[g], 1, status);
    for (int g = 0; g < 2; g++) wait_for(&sy.mat[g], R * L, status);
    small_job<S, L, R + 1, true, false, kRowRound, kSecBytes>(sy, job0, nloc, J, 0, 0, slices, k);
    for (int r = R; r < L; r++) {
        for (int g = 0; g < 2; g++) wait_for(&sy.mat[g], (r + 1) * L, status);
        small_job<S, L, 1, false, false, kRowRound, kSecBytes>(sy, job0 + enc_job_of<R>(r), nloc, J, r, 0, slices, k);
    }
}

#define TMVP_SMALL                                                                                                   \
    constexpr int L = S::L, EP = S::EP;                                                                              \
    __shared__ SmallLds<S> M;                                                                                        \
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);                                               \
    const int64_t base = (int64_t)blockIdx.x * kSmallInst;                                                           \
    const int nloc = (int)(B - base < kSmallInst ? B - base : kSmallInst);                                           \
    small_init(M, wave);                                                                                             \
    uint8_t *const raw = reinterpret_cast<uint8_t *>(W.A), *const sec = reinterpret_cast<uint8_t *>(W.s);            \
    const int grp = wave & 1;                                                                                        \
    if (wave < 4 && 4 * grp >= nloc) {                                                                               \
        publish(wave < 2 ? &M.sync.mat[grp] : &M.sync.sec[grp], kDone);                                              \
        return;                                                                                                      \
    }                                                                                                                \
    /* a row past the last instance repeats it: every row of a wave permutes, and the copies write the same bytes */ \
    const int li = 4 * grp + ((threadIdx.x & 63) >> 4) < nloc ? 4 * grp + ((threadIdx.x & 63) >> 4) : nloc - 1;      \
    const int sub = threadIdx.x & 15;                                                                                \
    const int64_t t = base + li

template <class S>
__global__ __launch_bounds__(kSmallThreads) __attribute__((amdgpu_waves_per_eu(4))) void kp_small_kernel(
    const uint8_t *seeds, uint8_t *pk, uint8_t *sk, KemWorkspace W, int64_t B, int *status)
{
    TMVP_SMALL;
    if (wave < 4) {
        const Row row(M.state[wave][(threadIdx.x & 63) >> 4], M.rc);
        uint8_t *pkt = pk + t * S::kPk, *skt = sk + t * S::kSk;
        const uint32_t *seed = reinterpret_cast<const uint32_t *>(seeds + t * 96);
        uint32_t A[5];
        if (wave < 2) {
            // seed_A' = SHAKE-128(seed_A) to the pk tail and the sk's copy of the pk, then GenMatrix
            row_hash<4, kShake128Rate>(A, seed, kShakeDS, row);
            row_store<4>(reinterpret_cast<uint32_t *>(pkt + S::kPvc), A, row);
            row_store<4>(reinterpret_cast<uint32_t *>(skt + S::kSec + S::kPvc), A, row);
            A[0] = row.x < 4 ? A[0] : 0u; // words 0..3 are the seed
#pragma unroll
            for (int y = 1; y < 5; y++) A[y] = 0;
            row_pad<4, kShake128Rate>(A, kShakeDS, row);
            small_matrix<S, true>(A, raw + t * S::kMatrix, row, &M.sync.mat[grp]);
            return;
        }
        row_load<4>(A, seed + 8, row);
        row_pad<4, kShake128Rate>(A, kShakeDS, row);
        small_secret<S, true>(A, M.stream[li], sec + t * L * kN, skt, sub, row);
        publish(&M.sync.sec[grp], 1);
        uint32_t m[5];
        row_load<4>(m, seed + 16, row);
        row_store<4>(reinterpret_cast<uint32_t *>(skt + S::kSk - 32), m, row);
        // b row by row into the pk and the sk's copy, and H(pk) over it as it grows
        row_zero(A);
        int done = 0;
        for (int r = 0; r < L; r++) {
            wait_for(&M.sync.done[2 + r], kSmallMfma, status);
            small_pack<EP>(W.v1 + (t * L + r) * kN, pkt + r * EP * 32, M.ct[li] + r * EP * 8,
                           skt + S::kSec + r * EP * 32, sub);
            if (r == L - 1 && sub < 8) // seed_A', written by the matrix wave before the rows' products began
                M.ct[li][S::kPvc / 4 + sub] = reinterpret_cast<const uint32_t *>(pkt + S::kPvc)[sub];
            row_fence();
            const int whole = (r == L - 1 ? S::kPk : (r + 1) * EP * 32) / kSha3_256Rate;
            row_absorb(A, reinterpret_cast<const uint8_t *>(M.ct[li]), done, whole, row);
            done = whole;
        }
        row_absorb_last<S::kPk>(A, reinterpret_cast<const uint8_t *>(M.ct[li]), row);
        row_store<4>(reinterpret_cast<uint32_t *>(skt + S::kSk - 64), A, row);
        return;
    }
    // products: heads and tails as in kp_fused_kernel
    const int k = wave - 4;
    RowJob J{};
    J.a = raw + base * S::kMatrix;
    J.s = sec + base * L * kN;
    J.out = W.v1 + base * L * kN;
    J.status = status;
    constexpr int kHeads = L == 4 ? 2 : 1, kHeadRows = L / kHeads;
    for (int g = 0; g < 2; g++) wait_for(&M.sync.sec[g], 1, status);
    for (int g = 0; g < 2; g++) wait_for(&M.sync.mat[g], (L - 1) * L, status);
    for (int h = 0; h < kHeads; h++)
        small_job<S, L - 1, kHeadRows, false, true, kRowSum, kSecBytes>(M.sync, h, nloc, J, h * kHeadRows, 0, M.mfma[k], k);
    for (int r = 0; r < L; r++) {
        for (int g = 0; g < 2; g++) wait_for(&M.sync.mat[g], (L - 1) * L + r + 1, status);
        wait_for(&M.sync.done[r / kHeadRows], kSmallMfma, status);
        small_job<S, 1, 1, false, true, kRowAddRound, kSecBytes>(M.sync, 2 + r, nloc, J, r, L - 1, M.mfma[k], k);
    }
}

template <class S>
__global__ __launch_bounds__(kSmallThreads) __attribute__((amdgpu_waves_per_eu(4))) void enc_small_kernel(
    const uint8_t *pk, const uint8_t *rnd, uint8_t *ct, uint8_t *ss, KemWorkspace W, int64_t B, int *status)
{
    constexpr int ET = S::ET;
    TMVP_SMALL;
    if (wave < 4) {
        const Row row(M.state[wave][(threadIdx.x & 63) >> 4], M.rc);
        const uint8_t *pkt = pk + t * S::kPk;
        uint32_t A[5];
        if (wave < 2) {
            row_load<4>(A, reinterpret_cast<const uint32_t *>(pkt + S::kPvc), row);
            row_pad<4, kShake128Rate>(A, kShakeDS, row);
            small_matrix<S, false>(A, raw + t * S::kMatrix, row, &M.sync.mat[grp]);
            return;
        }
        // m = H(rnd), (K, r) = G(m | H(pk)), the secret from r
        row_hash<4, kSha3_256Rate>(A, reinterpret_cast<const uint32_t *>(rnd + t * 32), kSha3DS, row);
        row_store<4>(M.msg + li * 8, A, row);
        row_store<4>(M.in[li], A, row);
        wait_for(&M.sync.hpk[grp], 1, status);
        row_fence();
        row_hash<8, kSha3_512Rate>(A, M.in[li], kSha3DS, row);
        row_store<8>(M.kr[li], A, row);
        row_fence();
        row_load<4>(A, M.kr[li] + 8, row);
        row_pad<4, kShake128Rate>(A, kShakeDS, row);
        small_secret<S, false>(A, M.stream[li], sec + t * L * kN, nullptr, sub, row);
        publish(&M.sync.sec[grp], 1);
        // the ciphertext row by row, and H(ct) over it as it grows
        uint8_t *c = ct + t * S::kCt;
        row_zero(A);
        int done = 0;
        for (int r = 0; r < L; r++) {
            wait_for(&M.sync.done[enc_job_of<1>(r)], kSmallMfma, status);
            small_pack<EP>(W.v1 + (t * L + r) * kN, c + r * EP * 32, M.ct[li] + r * EP * 8, nullptr, sub);
            if (r == L - 1) small_pack<ET>(W.poly + t * kN, c + S::kPvc, M.ct[li] + S::kPvc / 4, nullptr, sub);
            row_fence();
            const int whole = (r == L - 1 ? S::kCt : (r + 1) * EP * 32) / kSha3_256Rate;
            row_absorb(A, reinterpret_cast<const uint8_t *>(M.ct[li]), done, whole, row);
            done = whole;
        }
        row_absorb_last<S::kCt>(A, reinterpret_cast<const uint8_t *>(M.ct[li]), row);
        // ss = H(K | H(ct))
        row_store<4>(M.in[li] + 8, A, row);
        row_load<4>(A, M.kr[li], row);
        row_store<4>(M.in[li], A, row);
        row_fence();
        row_hash<8, kSha3_256Rate>(A, M.in[li], kSha3DS, row);
        row_store<4>(reinterpret_cast<uint32_t *>(ss + t * 32), A, row);
        return;
    }
    const int k = wave - 4;
    if (k < 2) {
        // H(pk) of group k's instances
        if (4 * k < nloc) {
            const Row row(M.state[4 + k][(threadIdx.x & 63) >> 4], M.rc);
            const uint8_t *pkt = pk + t * S::kPk;
            uint32_t A[5];
            row_zero(A);
            row_absorb(A, pkt, 0, S::kPk / kSha3_256Rate, row);
            row_absorb_last<S::kPk>(A, pkt, row);
            row_store<4>(M.in[li] + 8, A, row);
        }
        publish(&M.sync.hpk[k], 1);
    }
    RowJob J{};
    J.a = raw + base * S::kMatrix;
    J.b = pk + base * S::kPk;
    J.bstride = S::kPk;
    J.s = sec + base * L * kN;
    J.out = W.v1 + base * L * kN;
    J.out2 = W.poly + base * kN;
    J.msg = M.msg;
    J.status = status;
    small_products<S, 1>(M.sync, 0, nloc, J, M.mfma[k], k, status);
}

template <class S>
__global__ __launch_bounds__(kSmallThreads) __attribute__((amdgpu_waves_per_eu(4))) void dec_small_kernel(
    const uint8_t *ct, const uint8_t *sk, uint8_t *ss, uint8_t *fail, KemWorkspace W, int64_t B, int *status)
{
    constexpr int ET = S::ET;
    TMVP_SMALL;
    if (wave < 4) {
        const Row row(M.state[wave][(threadIdx.x & 63) >> 4], M.rc);
        const uint8_t *skt = sk + t * S::kSk, *c = ct + t * S::kCt;
        uint32_t A[5];
        if (wave < 2) {
            row_load<4>(A, reinterpret_cast<const uint32_t *>(skt + S::kSec + S::kPvc), row);
            row_pad<4, kShake128Rate>(A, kShakeDS, row);
            small_matrix<S, false>(A, raw + t * S::kMatrix, row, &M.sync.mat[grp]);
            return;
        }
        // (K', r') = G(m' | H(pk)), the secret s'' from r', once m' is there
        uint32_t H[5];
        row_load<4>(H, reinterpret_cast<const uint32_t *>(skt + S::kSk - 64), row);
        row_store<4>(M.in[li] + 8, H, row);
        wait_for(&M.sync.done[0], kSmallMfma, status);
        row_load<4>(A, M.msg + li * 8, row);
        row_store<4>(M.in[li], A, row);
        row_fence();
        row_hash<8, kSha3_512Rate>(A, M.in[li], kSha3DS, row);
        row_store<8>(M.kr[li], A, row);
        row_fence();
        row_load<4>(A, M.kr[li] + 8, row);
        row_pad<4, kShake128Rate>(A, kShakeDS, row);
        small_secret<S, false>(A, M.stream[li], sec + t * L * kN, nullptr, sub, row);
        publish(&M.sync.sec[grp], 1);
        // H(ct) while the products run
        row_zero(A);
        row_absorb(A, c, 0, S::kCt / kSha3_256Rate, row);
        row_absorb_last<S::kCt>(A, c, row);
        // the re-encryption against the ciphertext, row by row
        uint32_t diff = 0;
        for (int r = 0; r < L; r++) {
            wait_for(&M.sync.done[1 + enc_job_of<2>(r)], kSmallMfma, status);
            diff |= small_compare<EP>(W.v1 + (t * L + r) * kN, c + r * EP * 32, sub);
        }
        diff |= small_compare<ET>(W.poly + t * kN, c + S::kPvc, sub);
#pragma unroll
        for (int d = 1; d < 16; d <<= 1) diff |= (uint32_t)__shfl_xor((int)diff, d, 16);
        // ss = H(K | H(ct)) with K = K' on a match, z otherwise (constant time)
        uint32_t z[5], K[5];
        row_load<4>(z, reinterpret_cast<const uint32_t *>(skt + S::kSk - 32), row);
        row_load<4>(K, M.kr[li], row);
        const uint32_t mask = 0u - (uint32_t)(diff != 0);
        K[0] ^= mask & (K[0] ^ z[0]);
        row_store<4>(M.in[li] + 8, A, row);
        row_store<4>(M.in[li], K, row);
        row_fence();
        row_hash<8, kSha3_256Rate>(A, M.in[li], kSha3DS, row);
        row_store<4>(reinterpret_cast<uint32_t *>(ss + t * 32), A, row);
        if (fail && sub == 0) fail[t] = (uint8_t)(mask & 1u);
        return;
    }
    const int k = wave - 4;
    RowJob J{};
    J.a = ct + base * S::kCt;
    J.s = sk + base * S::kSk;
    J.cm = ct + base * S::kCt + S::kPvc;
    J.msg = M.msg;
    J.status = status;
    small_job<S, L, 1, false, false, kRowDecrypt, kSecKey>(M.sync, 0, nloc, J, 0, 0, M.mfma[k], k);
    J.a = raw + base * S::kMatrix;
    J.b = sk + base * S::kSk + S::kSec;
    J.bstride = S::kSk;
    J.s = sec + base * L * kN;
    J.out = W.v1 + base * L * kN;
    J.out2 = W.poly + base * kN;
    small_products<S, 2>(M.sync, 1, nloc, J, M.mfma[k], k, status);
}

#undef TMVP_SMALL

template <class F> static hipError_t by_set(const KemParams &P, F f)
{
    auto is = [&](auto s) {
        using S = decltype(s);
        return P.l == S::L && P.eq == S::EQ && P.mu == S::MU && P.ep == S::EP && P.et == S::ET;
    };
    const auto light = KemSet<2, 13, 10, 3, 10>{};
    const auto saber = KemSet<3, 13, 10, 4, 8>{};
    const auto fire = KemSet<4, 13, 10, 6, 6>{};
    const auto sable1 = KemSet<2, 11, 9, 3, 2>{};
    const auto sable2 = KemSet<3, 11, 9, 5, 2>{};
    const auto sable3 = KemSet<4, 11, 10, 3, 2>{};
    if (is(light)) return f(light);
    if (is(saber)) return f(saber);
    if (is(fire)) return f(fire);
    if (is(sable1)) return f(sable1);
    if (is(sable2)) return f(sable2);
    if (is(sable3)) return f(sable3);
    return hipErrorInvalidValue;
}

// ---------------------------------------------------------------- host chains

static inline unsigned blocks_for(int64_t n, int per) { return (unsigned)((n + per - 1) / per); }

// The one-launch kernel for B instances in its form (tmvp_kem_form.h): pairs(groups,
// instances per workgroup, workgroups) or rows(workgroups).
template <class F, class G> static hipError_t fused_launch(int64_t B, F pairs, G rows)
{
    const KemForm f = kem_form(B);
    if (f.groups == 0) rows((unsigned)f.blocks);
    else if (f.groups == 2) pairs(std::integral_constant<int, 2>{}, f.per, (unsigned)f.blocks);
    else pairs(std::integral_constant<int, 4>{}, f.per, (unsigned)f.blocks);
    return hipGetLastError();
}

static Job make_job(const KemParams &P, int mode, int epi, uint16_t *out, const uint16_t *a, const uint16_t *s,
                    const uint16_t *aux, int64_t B, int *status)
{
    Job J;
    memset(&J, 0, sizeof(J));
    J.out = out;
    J.a = a;
    J.s = s;
    J.aux = aux;
    J.status = status;
    J.batch = B;
    J.eq = P.eq;
    J.ep = P.ep;
    J.et = P.et;
    J.epi = epi;
    J.w = (mode == kInner) ? P.ep : P.eq;
    J.h = (epi == kEpiDec) ? P.h2 : P.h1;
    return J;
}

static hipError_t product(const KemParams &P, int backend, int mode, int epi, uint16_t *out, const uint16_t *a,
                          const uint16_t *s, const uint16_t *aux, int64_t B, int *status, hipStream_t st)
{
    const Job J = make_job(P, mode, epi, out, a, s, aux, B, status);
    return backend == 0 ? launch_mfma(J, mode, P.l, st) : launch_valu(J, mode, P.l, st);
}

#define TRY(x)                                                                                                       \
    do {                                                                                                             \
        hipError_t e_ = (x);                                                                                         \
        if (e_ != hipSuccess) return e_;                                                                             \
        e_ = hipGetLastError();                                                                                      \
        if (e_ != hipSuccess) return e_;                                                                             \
    } while (0)

// Codec launch for a run-time width: finds the instantiation with W == w.
template <int W>
static hipError_t pack_w(const uint16_t *src, int64_t src_stride, uint8_t *dst, int64_t dst_stride, int dst_off, int w,
                         int chunks, int64_t B, hipStream_t st, uint32_t *diff)
{
    if constexpr (W > 13) {
        return hipErrorInvalidValue;
    } else {
        if (w != W) return pack_w<W + 1>(src, src_stride, dst, dst_stride, dst_off, w, chunks, B, st, diff);
        hipLaunchKernelGGL((pack_kernel<W>), dim3(blocks_for(B * chunks, 256)), dim3(256), 0, st, src, src_stride,
                           dst, dst_stride, dst_off, chunks, B, diff);
        return hipGetLastError();
    }
}

template <int W>
static hipError_t unpack_w(const uint8_t *src, int64_t src_stride, int src_off, uint16_t *dst, int64_t dst_stride,
                           int w, int chunks, int xf, int64_t B, hipStream_t st)
{
    if constexpr (W > 13) {
        return hipErrorInvalidValue;
    } else {
        if (w != W) return unpack_w<W + 1>(src, src_stride, src_off, dst, dst_stride, w, chunks, xf, B, st);
        const dim3 grid(blocks_for(B * chunks, 256));
        if (xf == kXfSk2)
            hipLaunchKernelGGL((unpack_kernel<W, kXfSk2>), grid, dim3(256), 0, st, src, src_stride, src_off, dst,
                               dst_stride, chunks, B);
        else
            hipLaunchKernelGGL((unpack_kernel<W, kXfNone>), grid, dim3(256), 0, st, src, src_stride, src_off, dst,
                               dst_stride, chunks, B);
        return hipGetLastError();
    }
}

// ncoef is a multiple of 64; byte offsets and strides are multiples of 8.
static hipError_t pack(const uint16_t *src, int64_t src_stride, uint8_t *dst, int64_t dst_stride, int dst_off, int w,
                       int ncoef, int64_t B, hipStream_t st, uint32_t *diff = nullptr)
{
    return pack_w<1>(src, src_stride, dst, dst_stride, dst_off, w, ncoef / 64, B, st, diff);
}

static hipError_t unpack(const uint8_t *src, int64_t src_stride, int src_off, uint16_t *dst, int64_t dst_stride,
                         int w, int ncoef, int xf, int64_t B, hipStream_t st)
{
    return unpack_w<1>(src, src_stride, src_off, dst, dst_stride, w, ncoef / 64, xf, B, st);
}

template <int WS, int XS, int WB, int WC>
static hipError_t dec_unpack_w(const KemParams &P, const uint8_t *sk, const uint8_t *ct, uint16_t *S, uint16_t *Bp,
                               uint16_t *Cm, int64_t B, hipStream_t st, const int32_t *skey)
{
    hipLaunchKernelGGL((dec_unpack_kernel<WS, XS, WB, WC>), dim3(blocks_for(B * (8 * P.l + 4), 256)), dim3(256), 0,
                       st, sk, (int64_t)P.sk, ct, (int64_t)P.ct, P.pvc, S, Bp, Cm, P.l, B, skey);
    return hipGetLastError();
}

template <int EP, int ET>
static hipError_t dec_compare_w(const KemParams &P, const uint16_t *bp, const uint16_t *vp, const uint8_t *ct,
                                uint32_t *diff, int64_t B, hipStream_t st)
{
    hipLaunchKernelGGL((dec_compare_kernel<EP, ET>), dim3(blocks_for(B * (4 * P.l + 4), 256)), dim3(256), 0, st, bp, vp,
                       ct, (int64_t)P.ct, P.pvc, diff, P.l, B);
    return hipGetLastError();
}

// The re-encryption (b' and v') against ct in one launch.
static hipError_t dec_compare(const KemParams &P, const uint16_t *bp, const uint16_t *vp, const uint8_t *ct,
                              uint32_t *diff, int64_t B, hipStream_t st)
{
    if (P.ep == 10 && P.et == 3) return dec_compare_w<10, 3>(P, bp, vp, ct, diff, B, st);
    if (P.ep == 10 && P.et == 4) return dec_compare_w<10, 4>(P, bp, vp, ct, diff, B, st);
    if (P.ep == 10 && P.et == 6) return dec_compare_w<10, 6>(P, bp, vp, ct, diff, B, st);
    if (P.ep == 9 && P.et == 3) return dec_compare_w<9, 3>(P, bp, vp, ct, diff, B, st);
    if (P.ep == 9 && P.et == 5) return dec_compare_w<9, 5>(P, bp, vp, ct, diff, B, st);
    return hipErrorInvalidValue;
}

// s (from the sk), b' and c_m (from the ct) of a decapsulation in one launch,
// for the six parameter sets' widths.
static hipError_t dec_unpack(const KemParams &P, const uint8_t *sk, const uint8_t *ct, uint16_t *S, uint16_t *Bp,
                             uint16_t *Cm, int64_t B, hipStream_t st, const int32_t *skey)
{
    if (!P.sable && P.eq == 13 && P.ep == 10) {
        if (P.et == 3) return dec_unpack_w<13, kXfNone, 10, 3>(P, sk, ct, S, Bp, Cm, B, st, skey);
        if (P.et == 4) return dec_unpack_w<13, kXfNone, 10, 4>(P, sk, ct, S, Bp, Cm, B, st, skey);
        if (P.et == 6) return dec_unpack_w<13, kXfNone, 10, 6>(P, sk, ct, S, Bp, Cm, B, st, skey);
    }
    if (P.sable) {
        if (P.ep == 9 && P.et == 3) return dec_unpack_w<2, kXfSk2, 9, 3>(P, sk, ct, S, Bp, Cm, B, st, skey);
        if (P.ep == 9 && P.et == 5) return dec_unpack_w<2, kXfSk2, 9, 5>(P, sk, ct, S, Bp, Cm, B, st, skey);
        if (P.ep == 10 && P.et == 3) return dec_unpack_w<2, kXfSk2, 10, 3>(P, sk, ct, S, Bp, Cm, B, st, skey);
    }
    return hipErrorInvalidValue;
}

// Calls f(Shape<EQ, MU, EP>{}) for the parameter set's sampling shape.
template <class F> static hipError_t by_shape(const KemParams &P, F f)
{
    if (P.eq == 13 && P.ep == 10) {
        if (P.mu == 8) return f(Shape<13, 8, 10>{});
        if (P.mu == 10) return f(Shape<13, 10, 10>{});
        if (P.mu == 6) return f(Shape<13, 6, 10>{});
    } else if (P.eq == 11 && P.mu == 2) {
        if (P.ep == 9) return f(Shape<11, 2, 9>{});
        if (P.ep == 10) return f(Shape<11, 2, 10>{});
    }
    return hipErrorInvalidValue;
}

// Threads for n lane pairs.
static inline unsigned pair_blocks(int64_t n) { return blocks_for(2 * n, 64); }

// Launches a sponge kernel of one-wave workgroups in the form for its load:
// f(shared, grid).  Beyond a workgroup per SIMD the waves share SIMDs, and the
// permutation falls into step (VALU backend, Saber encapsulation of 20000, 40000
// and 65536 instances 571 -> 515, 1103 -> 966 and 1773 -> 1585 us; with a sponge
// compiled from C++ 590, 1099 and 1698).  Key generation's front kernel starts there
// at `most` = 2 workgroups per SIMD: up to that a SIMD's second wave is the short
// secret sponge (24576 instances of Sable type 1: 224 us, in step 230).  As a
// run-time test in the kernels it cost calls of up to 16384 instances 1.5 to 2 %.
template <class F> static hipError_t by_load(int64_t pairs, F f, unsigned most = 1)
{
    const dim3 grid(pair_blocks(pairs));
    if (grid.x > most * 4 * kCus) f(std::true_type{}, grid);
    else f(std::false_type{}, grid);
    return hipGetLastError();
}

// IND-CPA encryption (S/src/cuda_kernel.cu:124-178) in two halves.  The
// InnerProd half needs s', b of the pk (unpacked in W.v2) and the message's
// bits (W.bits, one per coefficient: S/src/pack.cu:86-99), all written by the
// front kernels, and writes pack_ET(round(b . s' - m)) to the ct tail; the
// MatrixVectorMul half needs A and writes pack_EP(round(A s')) to the ct head.
// With diff set (decapsulation's re-encryption), the halves compare with the
// ciphertext at ct instead of writing it.
static hipError_t enc_inner_half(const KemParams &P, const KemWorkspace &W, int backend, uint8_t *ct,
                                 uint32_t *diff, int64_t B, int *status, hipStream_t st)
{
    TRY(product(P, backend, kInner, kEpiEnc, W.poly, W.v2, W.s, W.bits, B, status, st));
    TRY(pack(W.poly, kN, ct, P.ct, P.pvc, P.et, kN, B, st, diff));
    return hipSuccess;
}

static hipError_t enc_matvec_half(const KemParams &P, const KemWorkspace &W, int backend, uint8_t *ct,
                                  uint32_t *diff, int64_t B, int *status, hipStream_t st)
{
    const int L = P.l;
    TRY(product(P, backend, kMatVec, kEpiQ2P, W.v1, W.A, W.s, nullptr, B, status, st));
    TRY(pack(W.v1, L * kN, ct, P.ct, 0, P.ep, L * kN, B, st, diff));
    return hipSuccess;
}

// Encryption's products and the final hashes.  MFMA: A s' and b . s' as one
// product, and the ciphertext packed inside the hash kernel; VALU: the two
// halves, each packing its part, then the hash kernel.
// A / akey: where the MFMA product reads each instance's matrix (default:
// W.A, instance i at i; keyed calls: the key store at the key id).
static hipError_t enc_finish(const KemParams &P, const KemWorkspace &W, int backend, uint8_t *ct, uint8_t *ss,
                             int64_t B, int *status, hipStream_t st, const uint16_t *A = nullptr,
                             const int32_t *akey = nullptr)
{
    if (backend != 0) {
        TRY(enc_matvec_half(P, W, backend, ct, nullptr, B, status, st));
        TRY(enc_inner_half(P, W, backend, ct, nullptr, B, status, st));
        return by_load(B, [&](auto shared, dim3 grid) {
            hipLaunchKernelGGL((enc_hash2_kernel<0, 0, shared.value>), grid, dim3(64), 0, st, P, ct, W.kr, ss, B, nullptr,
                               nullptr);
        });
    }
    Job J = make_job(P, kMatVec, kEpiQ2P, W.v1, A ? A : W.A, W.s, W.bits, B, status);
    J.b = W.v2;
    J.out2 = W.poly;
    J.akey = akey;
    TRY(launch_mfma(J, kEnc, P.l, st));
    auto go = [&](auto k) {
        constexpr int EP = decltype(k)::first_type::value, ET = decltype(k)::second_type::value;
        return by_load(B, [&](auto shared, dim3 grid) {
            hipLaunchKernelGGL((enc_hash2_kernel<EP, ET, shared.value>), grid, dim3(64), 0, st, P, ct, W.kr, ss, B, W.v1,
                               W.poly);
        });
    };
    using std::integral_constant;
    using std::pair;
    if (P.ep == 10 && P.et == 3) return go(pair<integral_constant<int, 10>, integral_constant<int, 3>>{});
    if (P.ep == 10 && P.et == 4) return go(pair<integral_constant<int, 10>, integral_constant<int, 4>>{});
    if (P.ep == 10 && P.et == 6) return go(pair<integral_constant<int, 10>, integral_constant<int, 6>>{});
    if (P.ep == 9 && P.et == 3) return go(pair<integral_constant<int, 9>, integral_constant<int, 3>>{});
    if (P.ep == 9 && P.et == 5) return go(pair<integral_constant<int, 9>, integral_constant<int, 5>>{});
    return hipErrorInvalidValue;
}

// Key generation and encapsulation run on one stream: the front kernel keeps
// one sponge wave per SIMD, and the steps after it are short and mostly
// bandwidth-bound, so running them beside each other gains less than the
// event waits cost.
hipError_t kem_keypair(const KemParams &P, const KemWorkspace &W, int backend, const uint8_t *seeds, uint8_t *pk,
                       uint8_t *sk, int64_t B, int *status, hipStream_t st)
{
    if (B <= 0) return hipSuccess;
    if (backend == 0) {
        // one launch (the one-launch section above)
        return by_set(P, [&](auto set) {
            return fused_launch(B, [&](auto groups, int per, unsigned blocks) {
                constexpr int G = decltype(groups)::value;
                hipLaunchKernelGGL((kp_fused_kernel<decltype(set), G>), dim3(blocks), dim3(kFusedThreads), 0,
                                   st, seeds, pk, sk, W, B, per, status);
            }, [&](unsigned blocks) {
                hipLaunchKernelGGL(kp_small_kernel<decltype(set)>, dim3(blocks), dim3(kSmallThreads), 0, st, seeds, pk, sk, W, B,
                                   status);
            });
        });
    }
    TRY(by_shape(P, [&](auto sh) {
        return by_load(2 * B, [&](auto shared, dim3 grid) {
            hipLaunchKernelGGL((kp_front_kernel<decltype(sh), shared.value>), grid, dim3(64), 0, st, P, seeds, pk, sk, W.A,
                               W.s, B);
        }, 2);
    }));
    TRY(product(P, backend, kMatVecT, kEpiQ2P, W.v1, W.A, W.s, nullptr, B, status, st));
    // the front kernel packed s into the sk; the hash kernel packs b into the
    // pk and the sk's copy of it, then hashes the pk
    auto hash = [&](auto ep) {
        return by_load(B, [&](auto shared, dim3 grid) {
            hipLaunchKernelGGL((kp_hash_kernel<ep.value, shared.value>), grid, dim3(64), 0, st, P, pk, sk, B, W.v1);
        });
    };
    if (P.ep == 10) return hash(std::integral_constant<int, 10>{});
    if (P.ep == 9) return hash(std::integral_constant<int, 9>{});
    return hipErrorInvalidValue;
}

hipError_t kem_encaps(const KemParams &P, const KemWorkspace &W, int backend, const uint8_t *pk, const uint8_t *rnd,
                      uint8_t *ct, uint8_t *ss, int64_t B, int *status, hipStream_t st)
{
    if (B <= 0) return hipSuccess;
    if (backend == 0) {
        return by_set(P, [&](auto set) {
            return fused_launch(B, [&](auto groups, int per, unsigned blocks) {
                constexpr int G = decltype(groups)::value;
                hipLaunchKernelGGL((enc_fused_kernel<decltype(set), G>), dim3(blocks), dim3(kFusedThreads), 0,
                                   st, pk, rnd, ct, ss, W, B, per, status);
            }, [&](unsigned blocks) {
                hipLaunchKernelGGL(enc_small_kernel<decltype(set)>, dim3(blocks), dim3(kSmallThreads), 0, st, pk, rnd, ct, ss, W, B,
                                   status);
            });
        });
    }
    TRY(by_shape(P, [&](auto sh) {
        return by_load(2 * B, [&](auto shared, dim3 grid) {
            hipLaunchKernelGGL((enc_front_kernel<decltype(sh), false, shared.value>), grid, dim3(64), 0, st, P, rnd, pk,
                               nullptr, W.buf, W.kr, W.A, W.s, W.v2, W.bits, B, (int64_t)0, nullptr);
        });
    }));
    return enc_finish(P, W, backend, ct, ss, B, status, st);
}

// Decapsulation; with `resident` set, the matrix A of every instance is
// already in W.A and is not generated again.  The matrix stream (and its
// unpacking) and H(ct) depend only on the inputs and run on W.aux beside the
// decryption and the InnerProd half of the re-encryption.
// resident: A is already in place (W.A, or the key store A at akey[i] for the
// MFMA backend), so the matrix sponge is skipped; skey (resident only): instance
// i's sk is row skey[i] of sk (a key store).
static hipError_t decaps_chain(const KemParams &P, const KemWorkspace &W, int backend, const uint8_t *ct,
                               const uint8_t *sk, uint8_t *ss, uint8_t *fail, int64_t B, int *status, hipStream_t st,
                               bool resident, const uint16_t *A = nullptr, const int32_t *akey = nullptr,
                               const int32_t *skey = nullptr)
{
    const int L = P.l;
    // Without resident A, the matrix sponge and H(ct) (dec_pre_kernel) run on
    // the side stream beside the decryption; with it, H(ct) runs inside the
    // re-encryption's front kernel and the call stays on one stream.
    if (!resident) {
        TRY(hipEventRecord(W.fork, st));
        TRY(hipStreamWaitEvent(W.aux, W.fork, 0));
        TRY(by_shape(P, [&](auto sh) {
            return by_load(2 * B, [&](auto shared, dim3 grid) {
                hipLaunchKernelGGL((dec_pre_kernel<decltype(sh), shared.value>), grid, dim3(64), 0, W.aux, P, ct, sk, W.A,
                                   W.hct, B);
            });
        }));
        TRY(hipEventRecord(W.join, W.aux));
    }
    // IND-CPA decryption (S/src/cuda_kernel.cu:341-370; SB/src/SABLE_indcpa.cu:422-463)
    if (resident) {
        TRY(dec_unpack(P, sk, ct, W.s, W.v2, W.poly, B, st, skey));
    } else {
        if (P.sable)
            TRY(unpack(sk, P.sk, 0, W.s, L * kN, 2, L * kN, kXfSk2, B, st));
        else
            TRY(unpack(sk, P.sk, 0, W.s, L * kN, P.eq, L * kN, kXfNone, B, st));
        TRY(unpack(ct, P.ct, 0, W.v2, L * kN, P.ep, L * kN, kXfNone, B, st));
        TRY(unpack(ct, P.ct, P.pvc, W.poly, kN, P.et, kN, kXfNone, B, st));
    }
    // m' bits to W.bits, where the re-encryption's InnerProd reads them
    TRY(product(P, backend, kInner, kEpiDec, W.bits, W.v2, W.s, W.poly, B, status, st));
    // re-encryption of m' under the pk stored in the sk
    TRY(by_shape(P, [&](auto sh) {
        return by_load(resident ? 2 * B : B, [&](auto shared, dim3 grid) {
            hipLaunchKernelGGL((dec_front_kernel<decltype(sh), shared.value>), grid, dim3(64), 0, st, P, W.bits, sk, W.buf,
                               W.kr, W.s, W.v2, W.diff, B, ct, resident ? W.hct : nullptr, skey);
        });
    }));
    // ct is only read: the compare-packs never write through it
    uint8_t *ctc = const_cast<uint8_t *>(ct);
    if (resident && backend == 0) {
        // A is there from the start: both products of the re-encryption as
        // one L + 1 row product (as in encapsulation), then both compares
        Job J = make_job(P, kMatVec, kEpiQ2P, W.v1, A ? A : W.A, W.s, W.bits, B, status);
        J.b = W.v2;
        J.out2 = W.poly;
        J.akey = akey;
        TRY(launch_mfma(J, kEnc, L, st));
        TRY(dec_compare(P, W.v1, W.poly, ct, W.diff, B, st));
    } else {
        TRY(enc_inner_half(P, W, backend, ctc, W.diff, B, status, st));
        if (!resident) TRY(hipStreamWaitEvent(st, W.join, 0));
        TRY(enc_matvec_half(P, W, backend, ctc, W.diff, B, status, st));
    }
    return by_load(B, [&](auto shared, dim3 grid) {
        if (skey)
            hipLaunchKernelGGL((dec_fin_kernel<true, shared.value>), grid, dim3(64), 0, st, P, W.diff, sk, W.hct, W.kr, ss,
                               fail, B, skey);
        else
            hipLaunchKernelGGL((dec_fin_kernel<false, shared.value>), grid, dim3(64), 0, st, P, W.diff, sk, W.hct, W.kr, ss,
                               fail, B, skey);
    });
}

hipError_t kem_decaps(const KemParams &P, const KemWorkspace &W, int backend, const uint8_t *ct, const uint8_t *sk,
                      uint8_t *ss, uint8_t *fail, int64_t B, int *status, hipStream_t st)
{
    if (B <= 0) return hipSuccess;
    if (backend == 0) {
        return by_set(P, [&](auto set) {
            return fused_launch(B, [&](auto groups, int per, unsigned blocks) {
                constexpr int G = decltype(groups)::value;
                hipLaunchKernelGGL((dec_fused_kernel<decltype(set), G>), dim3(blocks), dim3(kFusedThreads), 0,
                                   st, ct, sk, ss, fail, W, B, per, status);
            }, [&](unsigned blocks) {
                hipLaunchKernelGGL(dec_small_kernel<decltype(set)>, dim3(blocks), dim3(kSmallThreads), 0, st, ct, sk, ss, fail, W, B,
                                   status);
            });
        });
    }
    return decaps_chain(P, W, backend, ct, sk, ss, fail, B, status, st, false);
}

// One launch for the gathers in G (bytes per row given in words[] as bytes,
// multiples of 8).
static hipError_t gather(GatherSet G, const int32_t *keys, int64_t B, hipStream_t st)
{
    for (int g = 0; g < 3; g++) G.words[g] /= 8;
    const int total = G.words[0] + G.words[1] + G.words[2];
    hipLaunchKernelGGL(gather_kernel, dim3(blocks_for(B * total, 256)), dim3(256), 0, st, G, keys, B);
    return hipGetLastError();
}
hipError_t kem_encaps_keyed(const KemParams &P, const KemWorkspace &W, int backend, const KeyStore &K,
                            const int32_t *keys, const uint8_t *rnd, uint8_t *ct, uint8_t *ss, int64_t B, int *status,
                            hipStream_t st)
{
    if (B <= 0) return hipSuccess;
    // The front kernel reads pk and H(pk) from the key store at the key id,
    // and the MFMA product reads A there too; the VALU backend gets a
    // gathered copy of A.
    if (backend != 0) {
        const int abytes = P.l * P.l * kN * 2;
        TRY(gather(GatherSet{{reinterpret_cast<const uint8_t *>(K.A), nullptr, nullptr},
                             {abytes, 0, 0},
                             {reinterpret_cast<uint8_t *>(W.A), nullptr, nullptr},
                             {abytes, 0, 0},
                             {abytes, 0, 0}},
                   keys, B, st));
    }
    TRY(by_shape(P, [&](auto sh) {
        return by_load(B, [&](auto shared, dim3 grid) {
            hipLaunchKernelGGL((enc_front_kernel<decltype(sh), true, shared.value>), grid, dim3(64), 0, st, P, rnd, K.pk,
                               K.hpk, W.buf, W.kr, W.A, W.s, W.v2, W.bits, B, B, keys);
        });
    }));
    if (backend == 0) return enc_finish(P, W, backend, ct, ss, B, status, st, K.A, keys);
    return enc_finish(P, W, backend, ct, ss, B, status, st);
}

hipError_t kem_decaps_keyed(const KemParams &P, const KemWorkspace &W, int backend, const KeyStore &K,
                            const int32_t *keys, const uint8_t *ct, uint8_t *ss, uint8_t *fail, int64_t B,
                            int *status, hipStream_t st)
{
    if (B <= 0) return hipSuccess;
    // The decode, front and final kernels read the sk from the key store at
    // the key id; as in kem_encaps_keyed, the MFMA product reads A there too
    // and the VALU backend gets a gathered copy of A.
    if (backend != 0) {
        const int abytes = P.l * P.l * kN * 2;
        TRY(gather(GatherSet{{reinterpret_cast<const uint8_t *>(K.A), nullptr, nullptr},
                             {abytes, 0, 0},
                             {reinterpret_cast<uint8_t *>(W.A), nullptr, nullptr},
                             {abytes, 0, 0},
                             {abytes, 0, 0}},
                   keys, B, st));
        return decaps_chain(P, W, backend, ct, K.sk, ss, fail, B, status, st, true, nullptr, nullptr, keys);
    }
    return decaps_chain(P, W, backend, ct, K.sk, ss, fail, B, status, st, true, K.A, keys, keys);
}

hipError_t kem_store_derive(const KemParams &P, const uint8_t *pk, int64_t n, uint16_t *A, uint8_t *hpk,
                            hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    TRY(by_shape(P, [&](auto sh) {
        hipLaunchKernelGGL(matrix_kernel<decltype(sh)>, dim3(pair_blocks(n)), dim3(64), 0, st, P, pk + P.pvc,
                           (int64_t)P.pk, A, n);
        return hipGetLastError();
    }));
    hipLaunchKernelGGL(hash_pk_kernel, dim3(pair_blocks(n)), dim3(64), 0, st, P, pk, hpk, n);
    return hipGetLastError();
}

// The matrix A is the last piece, so a workspace without it (keyed MFMA
// calls read A from the key store) is the same layout cut short.
size_t kem_workspace_bytes(const KemParams &P, int64_t B, bool with_A)
{
    const size_t L = (size_t)P.l, n = (size_t)B;
    size_t b = 0;
    b += n * L * kN * 2;     // s
    b += n * L * kN * 2;     // v1
    b += n * L * kN * 2;     // v2
    b += n * kN * 2;         // bits
    b += n * kN * 2;         // poly
    b += n * 64;             // buf
    b += n * 64;             // kr
    b += n * 4;              // diff
    b += n * 32;             // hct
    b += 9 * 256;            // each of the pieces above rounded up to 256 bytes (kem_workspace_carve)
    if (with_A) b += n * L * L * kN * 2 + 256;
    return b;
}

void kem_workspace_carve(const KemParams &P, int64_t B, uint8_t *base, KemWorkspace &W, bool with_A)
{
    const size_t L = (size_t)P.l, n = (size_t)B;
    auto take = [&](size_t bytes) {
        uint8_t *p = base;
        base += (bytes + 255) & ~(size_t)255;
        return p;
    };
    W.s = reinterpret_cast<uint16_t *>(take(n * L * kN * 2));
    W.v1 = reinterpret_cast<uint16_t *>(take(n * L * kN * 2));
    W.v2 = reinterpret_cast<uint16_t *>(take(n * L * kN * 2));
    W.bits = reinterpret_cast<uint16_t *>(take(n * kN * 2));
    W.poly = reinterpret_cast<uint16_t *>(take(n * kN * 2));
    W.buf = take(n * 64);
    W.kr = take(n * 64);
    W.diff = reinterpret_cast<uint32_t *>(take(n * 4));
    W.hct = take(n * 32);
    W.A = with_A ? reinterpret_cast<uint16_t *>(take(n * L * L * kN * 2)) : nullptr;
}

} // namespace tmvp
