// Row products of the one-launch KEM kernels, on packed operands.
//
// The block decomposition, the limbs, the LDS layouts and the matrix-core
// mapping are those of mfma_body's 16x16x64 form (tmvp_mfma_body.h); this form
// differs in where its operands come from and go to.  The public polynomials
// are read as the W-bit streams they arrive in (the raw SHAKE-128 stream of
// the matrix, b of a public key, b' of a ciphertext), the secrets as the bytes
// the sampler wrote or as the secret key's codes, the message as its 32 bytes
// in LDS, and the decrypted message goes back there.  What bounds these jobs
// inside a KEM kernel is the issue slots a sponge wave leaves and the latency
// of their loads, so nothing is decoded into memory first: a lane loads the
// eight bytes that hold its four coefficients and spreads them with seven
// instructions as it stages them.  (A separate decode pass wrote and read back
// 3.5 KB more per decapsulation, 28 us of the call at 16384 Saber instances,
// and the sponge waves spent 11 us of a call unpacking the matrix.)
#pragma once

#include "tmvp_mfma_body.h"

namespace tmvp {

// A parameter set as compile-time values, with the derived byte sizes
// (S/include/params.h:26-49, SB/include/SABLE_params.h:26-72).
template <int L_, int EQ_, int EP_, int ET_, int MU_> struct KemSet {
    static constexpr int L = L_, EQ = EQ_, EP = EP_, ET = ET_, MU = MU_;
    static constexpr bool kSable = MU == 2;
    static constexpr int kPoly = EQ * 32;      // bytes of one polynomial of the matrix stream
    static constexpr int kMatrix = L * L * kPoly;
    static constexpr int kPvc = L * EP * 32;   // compressed polynomial vector
    static constexpr int kSec = kSable ? L * 64 : L * EQ * 32; // the secret in the sk
    static constexpr int kPk = kPvc + 32, kSk = kSec + kPk + 64, kCt = kPvc + ET * 32;
};

// What the job reads as secrets and does with its sums.
enum SecretForm : int {
    kSecBytes, // [L][256] int8
    kSecKey    // the secret key's codes: EQ-bit two's complement, or Sable's 2 bits
};
enum RowOp : int {
    kRowRound,   // ((x + h1) mod q) >> (eq - ep)
    kRowSum,     // x mod 2^16 (a row's first terms: the later ones add to it)
    kRowAdd,     // the sum of the terms before added, mod 2^16
    kRowAddRound,// a row's last terms: the sum added, then as kRowRound
    kRowDecrypt  // the decryption's message bits
};

// Pointers of one job, at the workgroup's first instance; polynomials of the
// matrix and of b are found by the set's sizes.
struct RowJob {
    const uint8_t *a;   // packed rows: the matrix stream, or b' (kRowDecrypt)
    const uint8_t *b;   // kRowRound with B: packed b
    int bstride;        // bytes between instances of b
    const uint8_t *s;   // secrets
    uint16_t *out;      // [instance][L][256]
    uint16_t *out2;     // kRowRound with B: v' [instance][256]
    const uint8_t *cm;  // kRowDecrypt: packed scale polynomial (in the ct)
    uint32_t *msg;      // LDS: the message's eight dwords per instance
    int *status;
};

// Where a lane's four W-bit coefficients 4 lane .. 4 lane + 3 lie in a packed
// polynomial: in the eight bytes at off (never past the polynomial's end), sh
// bits up.
template <int W> struct PackedLane {
    uint32_t off, sh;
    __device__ __forceinline__ explicit PackedLane(int lane)
    {
        const uint32_t bit = 4 * W * lane, last = 32 * W - 8;
        off = bit / 8 < last ? bit / 8 : last;
        sh = bit - 8 * off;
    }
    // The four coefficients as two dwords of halfwords; bits above W are left
    // as they come.
    __device__ __forceinline__ u32x2 spread(u32x2 v) const
    {
        const uint32_t lo = __builtin_amdgcn_alignbit(v.y, v.x, sh), hi = v.y >> sh;
        const uint32_t t = __builtin_amdgcn_alignbit(hi, lo, (2 * W) & 31);
        // high half of the shifted word, low half of the word
        return u32x2{(uint32_t)__builtin_amdgcn_bitop3_b32(0xffff0000u, lo << (16 - W), lo, 0xca),
                     (uint32_t)__builtin_amdgcn_bitop3_b32(0xffff0000u, t << (16 - W), t, 0xca)};
    }
};

template <class T> __device__ __forceinline__ T load_bytes(const uint8_t *p)
{
    T v;
    __builtin_memcpy(&v, p, sizeof(T)); // any alignment
    return v;
}

// LDS of one wave: two slices of NR rows.
template <int NR> constexpr int kRowSlice = NR * 2 * kEPoly + kBandBytes;

// The products of one wave: local instances first, first + stride, ... < end,
// NT terms (from term0) of rows row0 .. row0 + NR - 1; with B the last of the
// NR rows is b . s (encryption epilogue to out2).  TR: rows are columns of A
// (key generation).  slice0: the wave's 2 * kRowSlice<NR> bytes.
template <class S, int NT, int NR, bool B, bool TR, RowOp OP, SecretForm SF>
__device__ __forceinline__ void rows_body(const RowJob &J, int row0, int term0, int first, int stride, int end,
                                          uint8_t *const slice0)
{
    constexpr int L = S::L, EQ = S::EQ, EP = S::EP, ET = S::ET;
    constexpr int W = OP == kRowDecrypt ? EP : EQ; // modulus bits of the sums
    constexpr int SLICE = kRowSlice<NR>, E_BYTES = NR * 2 * kEPoly;
    const int lane = threadIdx.x & 63;
    int inst = first;
    if (inst >= end) return; // wave-uniform: each wave owns private LDS slices, no barriers
    int buf = 0;
    constexpr uint32_t lo4 = 0x7f7f7f7fu, hi4 = (((1u << W) - 1u) >> 7) * 0x01010101u, two = 0x00010001u;
    constexpr uint32_t wm2 = ((1u << W) - 1u) * two;

    // lane roles, as in mfma_body
    const int il = lane & 15, g = lane >> 4;
    const int R = lane & 7, limb = (lane >> 3) & 1;
    const int shc = (il + 1) & 3;
    const int abase = band_copy(shc) / 4 + 8 * (g >> 1) - 4 * (g & 1) + ((il + 17 - shc) >> 2);
    const int bbase = limb * kEPoly + 16 * (1 - (g & 1)) + (R - (g >> 1) + 8) * kEBlock;
    const PackedLane<W> pa(lane);
    const PackedLane<EP> pb(lane);
    const PackedLane<EQ> ps(lane);
    // decryption: positions of the lane's two pairs of scale coefficients
    const int lpos = 32 * R + 4 * g + 2 * limb;

    // one instance's inputs
    u32x2 va[NT][NR];
    constexpr bool SKEY = SF == kSecKey, S2 = SKEY && S::kSable, SW = SKEY && !S::kSable;
    u32x2 vs[NT]; // kSecBytes and the 2-bit codes use .x only
    constexpr bool ADD = OP == kRowAdd || OP == kRowAddRound;
    constexpr int SR = ADD ? NR : 1;
    uint32_t vc[SR][2] = {}, vc_next[SR][2] = {}; // per half h: the scale words (decryption) or the rows' sums so far
    auto fetch_side = [&](int i, uint32_t (&c)[SR][2]) {
        if constexpr (OP == kRowDecrypt) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const uint32_t bit = ET * (lpos + 16 * h), last = 32 * ET - 4;
                const uint32_t off = bit / 8 < last ? bit / 8 : last;
                c[0][h] = load_bytes<uint32_t>(J.cm + i * S::kCt + off) >> (bit - 8 * off);
            }
        } else if constexpr (ADD) {
#pragma unroll
            for (int r = 0; r < NR; r++)
#pragma unroll
                for (int h = 0; h < 2; h++)
                    c[r][h] = *reinterpret_cast<const uint32_t *>(J.out + (i * L + row0 + r) * kN + lpos + 16 * h);
        }
    };
    // Loads of term j of instance i (an instance past the end reloads the
    // current one, so every path issues the same loads).
    auto fetch_term = [&](int i, int j) {
        const int ie = i < end ? i : inst;
        const int tj = term0 + j;
#pragma unroll
        for (int r = 0; r < NR; r++) {
            if constexpr (OP == kRowDecrypt) {
                va[j][r] = load_bytes<u32x2>(J.a + ie * S::kCt + tj * (EP * 32) + pa.off);
            } else if (B && r == NR - 1) {
                va[j][r] = load_bytes<u32x2>(J.b + ie * J.bstride + tj * (EP * 32) + pb.off);
            } else {
                const int poly = TR ? tj * L + row0 + r : (row0 + r) * L + tj;
                va[j][r] = load_bytes<u32x2>(J.a + ie * S::kMatrix + poly * S::kPoly + pa.off);
            }
        }
        if constexpr (S2) vs[j].x = J.s[ie * S::kSk + tj * 64 + lane];
        else if constexpr (SW) vs[j] = load_bytes<u32x2>(J.s + ie * S::kSk + tj * S::kPoly + ps.off);
        else vs[j].x = *reinterpret_cast<const uint32_t *>(J.s + (ie * L + tj) * kN + 4 * lane);
    };
#pragma unroll
    for (int j = 0; j < NT; j++) fetch_term(inst, j);
    fetch_side(inst, vc);

    uint32_t bad = 0;
    auto stage = [&](int j, int into) {
        uint8_t *const E = slice0 + into * SLICE;
        uint8_t *const X = E + E_BYTES;
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const u32x2 v = (B && r == NR - 1) ? pb.spread(va[j][r]) : pa.spread(va[j][r]);
            const uint32_t s0 = shr16x2(v.x, 7), s1 = shr16x2(v.y, 7);
            const uint32_t plo = perm(v.y, v.x, 0x00020406u) & lo4;
            const uint32_t phi = perm(s1, s0, 0x00020406u) & hi4;
            uint8_t *slot = E + r * 2 * kEPoly + 28 - 4 * (lane & 7);
            const int b4 = lane >> 3;
            *(uint32_t *)(slot + (b4 + 8) * kEBlock) = plo;
            *(uint32_t *)(slot + kEPoly + (b4 + 8) * kEBlock) = phi;
            *(uint32_t *)(slot + b4 * kEBlock) = neg_small(plo);
            *(uint32_t *)(slot + kEPoly + b4 * kEBlock) = neg_small(phi);
        }
        // the secret as four int8, coefficient u in byte u
        uint32_t pos;
        if constexpr (S2) { // ((x ^ 2) - 2) of each 2-bit code (SB/src/pack.cu:366-377)
            uint32_t y = vs[j].x ^ 0xaau;
            y = (y | (y << 12)) & 0x000f000fu;
            y = (y | (y << 6)) & 0x03030303u;
            pos = ((y | 0x80808080u) - 0x02020202u) ^ 0x80808080u;
        } else if constexpr (SW) {
            const u32x2 sv = ps.spread(vs[j]);
            pos = perm(sv.y, sv.x, 0x06040200u);
            // range check, as in mfma_body: the key is the caller's
            bad |= (add16x2(add16x2(sv.x, 0x007f007fu) & wm2, 0x00010001u) |
                    add16x2(add16x2(sv.y, 0x007f007fu) & wm2, 0x00010001u));
        } else {
            pos = vs[j].x;
        }
        const uint32_t neg = neg_bytes(pos);
        const uint32_t p1 = from_next_lane(pos);
        const uint32_t n1 =
            (uint32_t)__builtin_amdgcn_update_dpp((int)__builtin_amdgcn_readlane(pos, 0), (int)neg, 0x130, 0xf, 0xf, false);
        uint8_t *band = X + 32 + 4 * lane;
        *(uint32_t *)band = pos;
#pragma unroll
        for (int c = 1; c < 4; c++) *(uint32_t *)(band + band_copy(c)) = __builtin_amdgcn_alignbyte(p1, pos, c);
        if (lane >= 56) {
            uint8_t *nb = X + 4 * lane - 224;
#pragma unroll
            for (int c = 0; c < 4; c++) *(uint32_t *)(nb + band_copy(c)) = c ? __builtin_amdgcn_alignbyte(n1, neg, c) : neg;
        }
    };
    // Ordering of the slices and of the input registers as in mfma_body.
    auto wave_fence = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    auto pin_after_stage = [&] { asm volatile("" : "+v"(bad) : : "memory"); };

    stage(0, 0);
    pin_after_stage();
    fetch_term(inst + stride, 0);
    wave_fence();
    // the rounding constant enters through the lo-limb accumulators
    constexpr int h1 = 1 << (EQ - EP - 1), h2 = (1 << (EP - 2)) - (1 << (EP - ET - 1)) + h1;
    const int hinit = limb ? 0 : OP == kRowSum || OP == kRowAdd ? 0 : OP == kRowDecrypt ? h2 : h1;
    const v4i init = {hinit, hinit, hinit, hinit};
    const uint32_t lshift = limb ? 0x00070007u : 0u;
    for (;;) {
        const int next = inst + stride;
        v4i acc[NR][2];
#pragma unroll
        for (int j = 0; j < NT; j++) {
            const uint8_t *const E = slice0 + buf * SLICE;
            int aoff = buf * SLICE + E_BYTES + 4 * abase;
            asm volatile("" : "+v"(aoff));
            const uint32_t *aw = reinterpret_cast<const uint32_t *>(slice0 + aoff);
            auto read_a = [&](int p, v4i (&f)[2]) {
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const uint32_t *w = aw + 16 * p + 4 * h;
                    f[h] = v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
                }
            };
            v4i acur[2];
            read_a(0, acur);
            v4i bcur[NR];
#pragma unroll
            for (int r = 0; r < NR; r++) bcur[r] = *(const v4i *)(E + r * 2 * kEPoly + bbase);

            if (j + 1 < NT) {
                stage(j + 1, buf ^ 1);
                pin_after_stage();
                fetch_term(next, j + 1);
                if (j + 2 == NT) fetch_side(next < end ? next : inst, vc_next);
            } else if (next < end) {
                stage(0, buf ^ 1);
                pin_after_stage();
                fetch_term(next + stride, 0);
                if (NT == 1) fetch_side(next, vc_next);
            }
#pragma unroll
            for (int p = 0; p < 4; p++) {
                v4i bnxt[NR], anxt[2];
                if (p < 3) {
                    read_a(p + 1, anxt);
#pragma unroll
                    for (int r = 0; r < NR; r++) bnxt[r] = *(const v4i *)(E + r * 2 * kEPoly + bbase - 64 * (p + 1));
                }
#pragma unroll
                for (int r = 0; r < NR; r++) {
                    const bool start = (j == 0 && p == 0);
                    acc[r][0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(acur[0], bcur[r], start ? init : acc[r][0], 0, 0, 0);
                    acc[r][1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(acur[1], bcur[r], start ? init : acc[r][1], 0, 0, 0);
                }
                if (p < 3) {
                    acur[0] = anxt[0];
                    acur[1] = anxt[1];
#pragma unroll
                    for (int r = 0; r < NR; r++) bcur[r] = bnxt[r];
                }
            }
            // Schedule: chunk 0's fragment reads first, then per chunk the next
            // chunk's reads and one MFMA per three staging VALU instructions.
            __builtin_amdgcn_sched_group_barrier(0x100, 4 + NR, 0);
#pragma unroll
            for (int p = 0; p < 4; p++) {
                if (p < 3) __builtin_amdgcn_sched_group_barrier(0x100, 4 + NR, 0);
#pragma unroll
                for (int k = 0; k < 2 * NR; k++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
                }
            }
            buf ^= 1;
            wave_fence();
        }

        // Epilogue, as in mfma_body: lo-limb lanes finish rows v = 0, 1 of
        // their group, hi-limb lanes v = 2, 3.
        uint32_t mbits = 0;
        const uint32_t mword = B ? J.msg[inst * 8 + R] >> (4 * g + 2 * limb) : 0u; // bits of positions lpos + ...
#pragma unroll
        for (int r = 0; r < NR; r++) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const uint32_t p01 = shl16x2(perm((uint32_t)acc[r][h][1], (uint32_t)acc[r][h][0], 0x05040100u), lshift);
                const uint32_t p23 = shl16x2(perm((uint32_t)acc[r][h][3], (uint32_t)acc[r][h][2], 0x05040100u), lshift);
                const uint32_t keep = limb ? p23 : p01;
                const uint32_t send = limb ? p01 : p23;
                const uint32_t y = add16x2(keep, (uint32_t)__builtin_amdgcn_mov_dpp((int)send, 0x128, 0xf, 0xf, false));
                if (B && r == NR - 1) {
                    const uint32_t x = mword >> (16 * h);
                    const uint32_t m = ((x & 1u) | ((x & 2u) << 15)) << (EP - 1);
                    *(uint32_t *)(J.out2 + inst * kN + lpos + 16 * h) =
                        shr16x2(sub16x2(y, m), EP - ET) & (((1u << ET) - 1u) * two);
                } else if constexpr (OP == kRowDecrypt) {
                    const uint32_t v = vc[0][h], c = (v & ((1u << ET) - 1u)) | (((v >> ET) & ((1u << ET) - 1u)) << 16);
                    const uint32_t d = shr16x2(sub16x2(y, c << (EP - ET)), EP - 1) & two;
                    mbits |= ((d | (d >> 15)) & 3u) << (16 * h);
                } else {
                    uint16_t *o = J.out + (inst * L + row0 + r) * kN + lpos + 16 * h;
                    const uint32_t x = ADD ? add16x2(y, vc[r < SR ? r : 0][h]) : y;
                    *(uint32_t *)o = OP == kRowSum || OP == kRowAdd ? x : shr16x2(x, EQ - EP) & (((1u << EP) - 1u) * two);
                }
            }
        }
        if constexpr (OP == kRowDecrypt)
            __hip_atomic_fetch_or(J.msg + inst * 8 + R, mbits << (4 * g + 2 * limb), __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_WORKGROUP);
#pragma unroll
        for (int r = 0; r < SR; r++)
#pragma unroll
            for (int h = 0; h < 2; h++) vc[r][h] = vc_next[r][h];
        inst = next;
        if (inst >= end) break;
    }
    if (SW && (bad & 0xff00ff00u)) *J.status = 1;
}

} // namespace tmvp
