// The form of a one-launch KEM kernel by batch size.  Plain C++, so that the
// rule can be checked on the host for every size.
#pragma once

#include <stdint.h>

namespace tmvp {

constexpr int64_t kCus = 256;
constexpr int kSmallInst = 8;  // instances of a workgroup of the row form; a CU holds two such workgroups
constexpr int kGroupInst = 32; // instances of a group on lane pairs; a CU holds one workgroup of two or four groups

struct KemForm {
    int groups;     // 0: a state on a row of lanes; 2 or 4: on lane pairs
    int per;        // instances of a workgroup (the last may hold fewer)
    int64_t blocks; // workgroups
};

// Lane pairs.  Two groups (one sponge wave per SIMD) give the shortest call,
// four (two waves per SIMD) the most instances at a time: 16384 Saber
// encapsulations take 187 us with two and 264 us with four, 32768 take 391
// (two rounds of workgroups) and 300 us.  So two groups where one round holds
// the batch, and beyond that four, the batch spread evenly over the rounds.
//
// The calls of other streams run beside a call, so it takes no more CUs than
// full workgroups of 64 need, as all calls did before there were several forms,
// or an eighth of the chip: fewer instances in a workgroup make its products
// shorter, and the calls of eight streams still fit side by side.  At least a
// quarter of the chip, and all of it from half a round on, make a call alone
// shorter (Saber encapsulation, 2048 instances 181 -> 169 us, 8193 184 -> 171), but
// send streams into rounds.  Eight hardware queues: eight calls of 2048 at once
// 342 us, with the eighth 215, before 244; lists of calls of 512 to 16384
// instances on four and on eight streams up to 1.12 and 1.16 times as long as
// before, with the eighth 0.79 to 0.90.  Four queues: up to 1.06, 0.78 to 0.90.
//
// A state on a row of lanes takes 0.6 of the time and four times the CUs:
// Saber key generation, encapsulation and decapsulation of 768 instances take
// 106, 108 and 91 us, on lane pairs 162, 170 and 136.  The line lies where eight
// streams of it still take no longer than before there was this form: eight
// times 768 encapsulations 218 us (before 242; FireSaber 319 and 346, Sable type 1
// 118 and 148), eight times 1024 284 us (before 244), on lane pairs 200.
constexpr int64_t kSmallBatch = kCus * 3;

constexpr KemForm kem_form(int64_t B)
{
    constexpr int64_t two = 2 * kGroupInst, four = 4 * kGroupInst;
    const auto up = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
    if (B <= kSmallBatch) return {0, kSmallInst, up(B, kSmallInst)};
    if (B > kCus * two) {
        const int64_t per = up(B, kCus * up(B, kCus * four));
        return {4, (int)per, up(B, per)};
    }
    const int64_t spread = up(B, kCus / 8), per = spread < two ? spread : two;
    return {2, (int)per, up(B, per)};
}

} // namespace tmvp
