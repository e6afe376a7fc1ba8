// The reference's host entry points, same names and signatures, over the
// batched GPU KEM.  The reference (S/include/cuda_kernel.cuh:6-7,
// SB/include/SABLE_indcpa.cuh:8-10) takes its batch size and parameter set
// from compile-time macros (BATCH = 1 for Saber, 512 for Sable type 2) and
// its randomness from a test vector; here they come from
// tmvp_host_configure() / tmvp_host_set_randomness(), with the reference's
// values as defaults and fresh OS randomness per call.  The functions are
// void, as in the reference; tmvp_host_status() returns the status of the
// last call.  Host buffers are [batch][size] arrays in the reference layouts.
#include <hip/hip_runtime.h>
#include <string.h>
#include <sys/random.h>

#include <chrono>
#include <mutex>

#include "../../include/tmvp.h"
#include "tmvp_internal.h"

namespace {

struct DevBuf {
    void *p = nullptr;
    size_t n = 0;
    int reserve(size_t bytes)
    {
        if (n >= bytes) return TMVP_OK;
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
        if (hipMalloc(&p, bytes) != hipSuccess) return TMVP_ENOMEM;
        n = bytes;
        return TMVP_OK;
    }
    void release()
    {
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
    uint8_t *u8() const { return static_cast<uint8_t *>(p); }
};

// Page-locked host memory that the device reads and writes directly.
struct PinnedBuf {
    void *p = nullptr, *dev = nullptr;
    size_t n = 0;
    bool reserve(size_t bytes)
    {
        if (n >= bytes) return true;
        release();
        // coherent: the host reads words that a running kernel has written
        if (hipHostMalloc(&p, bytes, hipHostMallocCoherent) != hipSuccess) {
            (void)hipGetLastError();
            p = nullptr;
            return false;
        }
        if (hipHostGetDevicePointer(&dev, p, 0) != hipSuccess) {
            (void)hipGetLastError();
            n = bytes;
            release();
            return false;
        }
        n = bytes;
        return true;
    }
    void release()
    {
        if (p) (void)hipHostFree(p);
        p = dev = nullptr;
        n = 0;
    }
    uint8_t *u8() const { return static_cast<uint8_t *>(p); }
};

// Up to kStageBytes each way go through page-locked buffers and copy kernels on
// the call's own queue (page-locked buffers of the caller go directly, see route).
// The runtime's copy of pageable memory costs a synchronisation each (four and
// one for the status word: 15 to 32 us apiece, 110 us around a Sable type 2
// encapsulation of 512 instances that runs for 95), the memcpy of half a megabyte 4
// to 12 us and its copy kernel 10.  Encapsulation and decapsulation, runtime's
// copies -> these: Saber 32 instances 267 -> 129 and 226 -> 114 us, 512: 325 -> 171 and
// 302 -> 164, 2048: 485 -> 362 and 442 -> 354; 8192 and 14000 encapsulations 1036 -> 752
// and 1631 -> 1190.
//
// The buffers are rings of kSlots pieces each way, so that the bus moves one
// piece while the host copies the next and little memory is held: locking costs
// about 0.5 us a KB once (buffers as large as a call's operands made the first
// call of 8192 encapsulations take 9.3 ms, with the rings 2.7, with the
// runtime's copies 2.1).  Pieces of 256 KB, 512 KB and 1 MB: 321, 296 and 316 us for 2048
// decapsulations.  Past kStageBytes the runtime's engine outruns the copy kernel on
// page-locked inputs (8192 Saber decapsulations, 27 MB in: 687 against 736 us).
constexpr size_t kStageBytes = 16u << 20;
constexpr size_t kChunk = 512u << 10;
constexpr int kSlots = 4;
constexpr size_t kRing = kSlots * kChunk;
constexpr size_t kWipeAfter = 16u << 10; // see copy_in
constexpr size_t kWordBytes = 4096; // a page before a ring: a word per slot, then the status word

// Words that a move leaves in page-locked memory.
struct Words {
    int *status_to;    // the context's status word goes here
    const int *status;
    int *done;         // 1 once all of src has been read (to the device) or all of dst written (from it)
    int *blocks;       // counts the workgroups that have; 0 between launches
};

// n16 16-byte units from src to dst, one of them in page-locked host memory, and
// W's words (null: none).  Four loads in flight per thread.
constexpr int kMoveThreads = 256;
template <bool OUT>
__global__ __launch_bounds__(kMoveThreads) void move_kernel(uint4 *dst, const uint4 *src, size_t n16, Words W)
{
    const size_t stride = (size_t)gridDim.x * kMoveThreads;
    size_t i = (size_t)blockIdx.x * kMoveThreads + threadIdx.x;
    for (; i + 3 * stride < n16; i += 4 * stride) {
        const uint4 a = src[i], b = src[i + stride], c = src[i + 2 * stride], d = src[i + 3 * stride];
        dst[i] = a;
        dst[i + stride] = b;
        dst[i + 2 * stride] = c;
        dst[i + 3 * stride] = d;
    }
    for (; i < n16; i += stride) dst[i] = src[i];
    if (W.status_to && blockIdx.x == 0 && threadIdx.x == 0) *W.status_to = *W.status;
    if (W.done) {
        // To the device, the loads have returned when their stores are on their way;
        // from it, the stores have to arrive.
        if (OUT) __threadfence_system();
        __syncthreads();
        if (threadIdx.x == 0 && atomicAdd(W.blocks, 1) == (int)gridDim.x - 1) {
            *W.blocks = 0;
            __hip_atomic_store(W.done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

template <bool OUT> int move_bytes(void *dst, const void *src, size_t bytes, const Words &W, hipStream_t st)
{
    size_t blocks = (bytes + 64 * kMoveThreads - 1) / (64 * kMoveThreads);
    if (blocks > 256) blocks = 256;
    if (blocks == 0) blocks = 1; // the status word alone
    hipLaunchKernelGGL(move_kernel<OUT>, dim3((unsigned)blocks), dim3(kMoveThreads), 0, st, static_cast<uint4 *>(dst),
                       static_cast<const uint4 *>(src), bytes / 16, W);
    return hipGetLastError() == hipSuccess ? TMVP_OK : TMVP_EHIP;
}

// How one of a call's operands crosses the bus.
enum Route {
    kStaged, // pageable memory: copied by the host to or from page-locked buffers
    kDirect, // the caller's page-locked memory: by the copy kernel, in place
    kRuntime // by the runtime's copies: larger than kStageBytes, or neither of the above
};

// One of a call's two operands in each direction: n bytes (a multiple of 16) at h.
struct Part {
    void *h;
    size_t n;
    Route route;
    void *dev; // kDirect: the device's address
};

// Page-locked memory of the caller goes direct when all of it is one mapping
// at 16-byte alignment and no smaller than this, below which the launch of its own
// costs more than the host's pass (32 Saber encapsulations 128 us staged, 135
// direct).  Through the staging, Saber encapsulations of 512 and 4096 instances
// from page-locked buffers took 170 and 551 us, decapsulations of 4096 520; direct
// 154, 391 and 469; with the runtime's copies 290, 445 and 496.
constexpr size_t kDirectBytes = 128u << 10;

Part route(const void *h, size_t n)
{
    Part part{const_cast<void *>(h), n, kStaged, nullptr};
    if (n == 0) return part;
    hipPointerAttribute_t a, z;
    auto known = [](hipPointerAttribute_t &x, const void *p) {
        const hipError_t e = hipPointerGetAttributes(&x, p);
        (void)hipGetLastError(); // pageable memory may report an error: clear it
        return e == hipSuccess && x.type != hipMemoryTypeUnregistered;
    };
    if (!known(a, h)) return part;
    if (a.type != hipMemoryTypeHost) {
        part.route = kRuntime;
    } else if (n >= kDirectBytes && a.devicePointer && ((uintptr_t)a.devicePointer & 15) == 0 &&
               known(z, static_cast<const uint8_t *>(h) + n - 1) && z.type == hipMemoryTypeHost &&
               static_cast<uint8_t *>(z.devicePointer) - static_cast<uint8_t *>(a.devicePointer) == (ptrdiff_t)(n - 1)) {
        part.route = kDirect;
        part.dev = a.devicePointer;
    }
    return part;
}

// The secret bytes of an operand in rows of `stride`: the first `head` and the
// last `tail` of each.
struct Secret {
    size_t stride, head, tail;
};

// The staged bytes of two operands, which are neighbours on the device: from
// the first staged one on.
struct Staging {
    Part a, b; // n = 0 where not staged
    size_t skip;
    size_t n() const { return a.n + b.n; }
};

struct HostState {
    std::mutex mu;
    int device = 0;
    int64_t saber_batch = 1, sable_batch = 512;
    int saber_set = TMVP_SABER, sable_set = TMVP_SABLE2;
    tmvp_ctx *ctx = nullptr;
    hipStream_t stream = nullptr;
    DevBuf in, out;         // a call's inputs and outputs on the device, one behind the other
    PinnedBuf h_in, h_out;  // kWordBytes of words, then a ring of pieces on their way
    DevBuf blocks;          // Words::blocks
    // of the bytes that this call sent through h_in's ring, those from wipe_from
    // on hold `secret` and are still there; wipe_slot's word (if not negative) says
    // that they have been read
    size_t wipe_from = 0, wipe_to = 0;
    Secret secret{};
    int wipe_slot = -1;
    uint8_t *rnd = nullptr; // caller randomness for the next encapsulation
    size_t rnd_bytes = 0;
    int status = TMVP_OK;
};

HostState &state()
{
    static HostState s;
    return s;
}

int ensure_ctx(HostState &S)
{
    if (S.ctx) return hipSetDevice(S.device) == hipSuccess ? TMVP_OK : TMVP_EHIP;
    int rc = tmvp_init(&S.ctx, S.device);
    if (rc) {
        S.ctx = nullptr;
        return rc;
    }
    if (hipStreamCreateWithFlags(&S.stream, hipStreamNonBlocking) != hipSuccess) {
        tmvp_destroy(S.ctx);
        S.ctx = nullptr;
        return TMVP_EHIP;
    }
    rc = S.blocks.reserve(sizeof(int));
    if (!rc && hipMemset(S.blocks.p, 0, sizeof(int)) != hipSuccess) rc = TMVP_EHIP;
    if (rc) {
        S.blocks.release();
        (void)hipStreamDestroy(S.stream);
        S.stream = nullptr;
        tmvp_destroy(S.ctx);
        S.ctx = nullptr;
    }
    return rc;
}

int backend_of(int mode)
{
    switch (mode) {
    case 0: return TMVP_BACKEND_MFMA;
    case 1: return TMVP_BACKEND_VALU;
    case 2: return TMVP_BACKEND_SCHOOLBOOK;
    default: return -1;
    }
}

int fill_random(uint8_t *dst, size_t n)
{
    size_t got = 0;
    while (got < n) {
        ssize_t k = getrandom(dst + got, n - got, 0);
        if (k <= 0) return TMVP_EARG;
        got += (size_t)k;
    }
    return TMVP_OK;
}

// Which of a call's operands are staged in buf.
Staging staging(PinnedBuf &buf, Part &a, Part &b)
{
    if (a.n + b.n > kStageBytes) a.route = b.route = kRuntime;
    Staging g{a, b, a.route == kStaged ? 0 : a.n};
    if (a.route != kStaged) g.a.n = 0;
    if (b.route != kStaged) g.b.n = 0;
    if (!buf.reserve(kWordBytes + (g.n() < kRing ? g.n() : kRing))) {
        if (g.a.n) a.route = kRuntime;
        if (g.b.n) b.route = kRuntime;
        g.a.n = g.b.n = 0;
    }
    return g;
}

// The host's and the device's addresses in buf's ring and among its words.
uint8_t *ring(const PinnedBuf &buf, size_t at) { return buf.u8() + kWordBytes + at; }
uint8_t *ring_dev(const PinnedBuf &buf, size_t at) { return static_cast<uint8_t *>(buf.dev) + kWordBytes + at; }
int *word(const PinnedBuf &buf, int i) { return reinterpret_cast<int *>(buf.u8()) + i; }
int *word_dev(const PinnedBuf &buf, int i) { return static_cast<int *>(buf.dev) + i; }

// Waits until a launched move has set its word, after 5 ms for the stream; false
// on an error.
bool wait_word(HostState &S, const int *w)
{
    const auto end = std::chrono::steady_clock::now() + std::chrono::milliseconds(5);
    do {
        for (int spin = 0; spin < 1000; spin++)
            if (__atomic_load_n(w, __ATOMIC_ACQUIRE)) return true;
    } while (std::chrono::steady_clock::now() < end);
    return hipStreamSynchronize(S.stream) == hipSuccess;
}

// The part of [at, end) of two operands laid end to end that lies in each: f(host
// address, offset from at, bytes).
template <class F> void pieces(const Staging &g, size_t at, size_t end, F f)
{
    if (at < g.a.n) f(static_cast<uint8_t *>(g.a.h) + at, (size_t)0, (end < g.a.n ? end : g.a.n) - at);
    if (end > g.a.n) {
        const size_t from = at > g.a.n ? at : g.a.n;
        f(static_cast<uint8_t *>(g.b.h) + (from - g.a.n), from - at, end - from);
    }
}

// The two inputs to S.in; the secrets in the second one do not stay in the ring
// (wipe_inputs).
int copy_in(HostState &S, Part a, Part b, const Secret &secret)
{
    const Staging g = staging(S.h_in, a, b);
    const Part *const parts[2] = {&a, &b};
    uint8_t *const at_dev[2] = {S.in.u8(), S.in.u8() + a.n};
    const size_t n = g.n();
    S.wipe_from = S.wipe_to = 0;
    if (g.b.n) {
        S.wipe_from = g.a.n;
        S.wipe_to = n;
        S.secret = secret;
    }
    S.wipe_slot = -1;
    // few secrets are cleared after the wait, in less time than a word costs its move (2 us)
    const bool wipe_early = g.b.n / secret.stride * (secret.head + secret.tail) > kWipeAfter;
    auto fail = [&](int rc) { // some pieces are on their way: the whole ring is cleared after the wait
        const size_t used = n < kRing ? n : kRing;
        S.wipe_from = 0;
        S.wipe_to = used;
        S.secret = {used, used, 0};
        return rc;
    };
    for (int i = 0; i < 2; i++) // the bus beside the host's copies below
        if (parts[i]->route == kDirect) {
            const int rc = move_bytes<false>(at_dev[i], parts[i]->dev, parts[i]->n, {}, S.stream);
            if (rc) return rc;
        }
    for (size_t at = 0; at < n; at += kChunk) { // and beside the next piece's memcpy
        const size_t end = at + kChunk < n ? at + kChunk : n, off = at % kRing;
        const int slot = (int)(off / kChunk);
        if (at >= kRing && !wait_word(S, word(S.h_in, slot))) return fail(TMVP_EHIP);
        pieces(g, at, end, [&](const uint8_t *h, size_t o, size_t bytes) { memcpy(ring(S.h_in, off + o), h, bytes); });
        Words W{};
        const bool last = end == n && wipe_early;
        if (at + kRing < n || last) { // waited for: the slot is used again, or cleared
            *word(S.h_in, slot) = 0;
            W.done = word_dev(S.h_in, slot);
            W.blocks = static_cast<int *>(S.blocks.p);
        }
        if (last) S.wipe_slot = slot;
        const int rc = move_bytes<false>(S.in.u8() + g.skip + at, ring_dev(S.h_in, off), end - at, W, S.stream);
        if (rc) return fail(rc);
    }
    for (int i = 0; i < 2; i++)
        if (parts[i]->route == kRuntime && parts[i]->n &&
            hipMemcpyAsync(at_dev[i], parts[i]->h, parts[i]->n, hipMemcpyHostToDevice, S.stream) != hipSuccess)
            return TMVP_EHIP;
    return TMVP_OK;
}

// Clears the call's secrets in the ring, where the last kRing bytes sent are.
// Called when everything has been launched, so it works while the kernels run (512
// Saber decapsulations 163 -> 164 us, 2048 350 -> 354; the copy kernels clearing over
// the bus: 182 and 412).  `done`: after the wait for the stream.
void wipe_inputs(HostState &S, bool done)
{
    if (S.wipe_from == S.wipe_to) return;
    // pieces before the last were read before it
    if (!done && (S.wipe_slot < 0 || !wait_word(S, word(S.h_in, S.wipe_slot)))) return;
    const size_t left = S.wipe_to > kRing ? S.wipe_to - kRing : 0; // the first byte not overwritten
    auto clear = [&](size_t from, size_t to) {
        if (from < left) from = left;
        if (from >= to) return;
        const size_t at = from % kRing, first = to - from < kRing - at ? to - from : kRing - at;
        explicit_bzero(ring(S.h_in, at), first);
        explicit_bzero(ring(S.h_in, 0), to - from - first);
    };
    const Secret &x = S.secret;
    size_t row = S.wipe_from;
    if (row < left) row += (left - row) / x.stride * x.stride;
    for (; row < S.wipe_to; row += x.stride) {
        clear(row, row + x.head);
        clear(row + x.stride - x.tail, row + x.stride);
    }
    S.wipe_from = S.wipe_to;
}

// The wait for the call's work; the status word is read on the way out.
int finish(HostState &S)
{
    const hipError_t e = hipStreamSynchronize(S.stream);
    wipe_inputs(S, true);
    if (e != hipSuccess) return TMVP_EHIP;
    return tmvp_ctx_status(S.ctx, S.stream);
}

// The outputs from S.out, and the call's end.  The second one is secret and does
// not stay in the ring.
int copy_out(HostState &S, Part a, Part b)
{
    const Staging g = staging(S.h_out, a, b);
    const Part *const parts[2] = {&a, &b};
    uint8_t *const at_dev[2] = {S.out.u8(), S.out.u8() + a.n};
    int rc = TMVP_OK;
    for (int i = 0; i < 2 && !rc; i++) {
        if (parts[i]->route == kDirect)
            rc = move_bytes<true>(parts[i]->dev, at_dev[i], parts[i]->n, {}, S.stream);
        else if (parts[i]->route == kRuntime && parts[i]->n &&
                 hipMemcpyAsync(parts[i]->h, at_dev[i], parts[i]->n, hipMemcpyDeviceToHost, S.stream) != hipSuccess)
            rc = TMVP_EHIP;
    }
    if (rc || !S.h_out.p) {
        const int rc2 = finish(S);
        return rc ? rc : rc2;
    }
    // One piece up to the ring's size; more go as the host empties the slots.
    const size_t n = g.n(), piece = n <= kRing ? kRing : kChunk;
    const int count = n ? (int)((n + piece - 1) / piece) : 1; // without staged outputs, the status word alone
    int *const flag = word(S.h_out, kSlots);
    *flag = 1; // until the kernel has written it
    auto launch = [&](int k) {
        const size_t at = k * piece, end = at + piece < n ? at + piece : n;
        const int slot = k % kSlots;
        Words W{};
        if (k == 0) {
            W.status_to = word_dev(S.h_out, kSlots);
            W.status = tmvp::ctx_status_word(S.ctx);
        }
        if (k >= kSlots) { // the first ones are waited for with the stream
            *word(S.h_out, slot) = 0;
            W.done = word_dev(S.h_out, slot);
            W.blocks = static_cast<int *>(S.blocks.p);
        }
        return move_bytes<true>(ring_dev(S.h_out, at % kRing), S.out.u8() + g.skip + at, end - at, W, S.stream);
    };
    for (int k = 0; k < count && k < kSlots && !rc; k++) rc = launch(k);
    wipe_inputs(S, false);
    if (hipStreamSynchronize(S.stream) != hipSuccess) rc = TMVP_EHIP;
    wipe_inputs(S, true);
    for (int k = 0; k < count && !rc; k++) {
        if (k >= kSlots && !wait_word(S, word(S.h_out, k % kSlots))) rc = TMVP_EHIP;
        const size_t at = k * piece, end = at + piece < n ? at + piece : n;
        if (rc) break;
        pieces(g, at, end, [&](uint8_t *h, size_t o, size_t bytes) {
            memcpy(h, ring(S.h_out, at % kRing + o), bytes);
            if (at + o >= g.a.n) explicit_bzero(ring(S.h_out, at % kRing + o), bytes);
        });
        if (k + kSlots < count) rc = launch(k + kSlots);
    }
    if (rc) {
        (void)hipStreamSynchronize(S.stream); // nothing moves into the ring any more
        explicit_bzero(ring(S.h_out, 0), n < kRing ? n : kRing);
        return rc;
    }
    return *flag ? tmvp_ctx_status(S.ctx, S.stream) : TMVP_OK;
}

// Encapsulation of `batch` instances: h_pk in, h_c and h_k out.
int host_enc(HostState &S, int ps, int64_t batch, int mode, uint8_t *h_k, const uint8_t *h_pk, uint8_t *h_c)
{
    const int backend = backend_of(mode);
    if (backend < 0 || !h_k || !h_pk || !h_c) return TMVP_EARG;
    int rc = ensure_ctx(S);
    if (rc) return rc;
    tmvp_params P;
    tmvp_get_params(ps, &P);
    const size_t B = (size_t)batch;
    const size_t npk = B * P.pk_bytes, nct = B * P.ct_bytes;
    if ((rc = S.in.reserve(npk + B * 32)) || (rc = S.out.reserve(nct + B * 32))) return rc;
    uint8_t *rnd = S.rnd;
    uint8_t *fresh = nullptr;
    if (rnd && S.rnd_bytes != B * 32) {
        // randomness set for another batch size: an error, not a silent
        // switch to fresh randomness (the caller expects its own coins)
        delete[] S.rnd;
        S.rnd = nullptr;
        S.rnd_bytes = 0;
        return TMVP_EARG;
    }
    if (!rnd) {
        fresh = new uint8_t[B * 32];
        if ((rc = fill_random(fresh, B * 32))) {
            delete[] fresh;
            return rc;
        }
        rnd = fresh;
    }
    rc = copy_in(S, route(h_pk, npk), {rnd, B * 32, kStaged, nullptr}, {B * 32, B * 32, 0});
    if (!rc)
        rc = tmvp_kem_encaps(S.ctx, ps, backend, S.out.u8(), S.out.u8() + nct, S.in.u8(), S.in.u8() + npk, batch,
                             S.stream);
    const int rc2 = rc ? finish(S) : copy_out(S, route(h_c, nct), route(h_k, B * 32)); // either waits for the copy of `rnd`
    delete[] fresh;
    delete[] S.rnd; // randomness is used once
    S.rnd = nullptr;
    S.rnd_bytes = 0;
    return rc ? rc : rc2;
}

// Decapsulation of `batch` instances: h_c and h_sk in, h_k out.  The public
// key is read from the sk, which holds a copy (S/include/params.h:45-46).
int host_dec(HostState &S, int ps, int64_t batch, int mode, const uint8_t *h_c, const uint8_t *h_sk, uint8_t *h_k)
{
    const int backend = backend_of(mode);
    if (backend < 0 || !h_c || !h_sk || !h_k) return TMVP_EARG;
    int rc = ensure_ctx(S);
    if (rc) return rc;
    tmvp_params P;
    tmvp_get_params(ps, &P);
    const size_t B = (size_t)batch;
    const size_t nsk = B * P.sk_bytes, nct = B * P.ct_bytes;
    if ((rc = S.in.reserve(nct + nsk)) || (rc = S.out.reserve(B * 32))) return rc;
    rc = copy_in(S, route(h_c, nct), route(h_sk, nsk),
                 {(size_t)P.sk_bytes, (size_t)(P.sable ? P.l * 64 : P.l * P.eq * 32), 32}); // s and z
    if (!rc)
        rc = tmvp_kem_decaps(S.ctx, ps, backend, S.out.u8(), S.in.u8(), S.in.u8() + nct, nullptr, batch, S.stream);
    const int rc2 = rc ? finish(S) : copy_out(S, route(nullptr, 0), route(h_k, B * 32));
    return rc ? rc : rc2;
}

bool is_saber(int ps) { return ps == TMVP_LIGHTSABER || ps == TMVP_SABER || ps == TMVP_FIRESABER; }
bool is_sable(int ps) { return ps == TMVP_SABLE1 || ps == TMVP_SABLE2 || ps == TMVP_SABLE3; }

} // namespace

extern "C" {

int tmvp_host_configure(int device, int64_t saber_batch, int saber_set, int64_t sable_batch, int sable_set)
{
    if (device < 0 || saber_batch <= 0 || sable_batch <= 0 || !is_saber(saber_set) || !is_sable(sable_set))
        return TMVP_EARG;
    HostState &S = state();
    std::lock_guard<std::mutex> g(S.mu);
    if (S.ctx && device != S.device) return TMVP_EARG; // release first to move to another device
    S.device = device;
    S.saber_batch = saber_batch;
    S.saber_set = saber_set;
    S.sable_batch = sable_batch;
    S.sable_set = sable_set;
    return TMVP_OK;
}

int tmvp_host_set_randomness(const uint8_t *h_rnd, int64_t batch)
{
    HostState &S = state();
    std::lock_guard<std::mutex> g(S.mu);
    delete[] S.rnd;
    S.rnd = nullptr;
    S.rnd_bytes = 0;
    if (!h_rnd) return TMVP_OK;
    if (batch <= 0) return TMVP_EARG;
    S.rnd_bytes = (size_t)batch * 32;
    S.rnd = new uint8_t[S.rnd_bytes];
    memcpy(S.rnd, h_rnd, S.rnd_bytes);
    return TMVP_OK;
}

int tmvp_host_status(void)
{
    HostState &S = state();
    std::lock_guard<std::mutex> g(S.mu);
    return S.status;
}

int tmvp_host_release(void)
{
    HostState &S = state();
    std::lock_guard<std::mutex> g(S.mu);
    int rc = TMVP_OK;
    if (S.ctx) {
        if (S.stream && hipStreamSynchronize(S.stream) != hipSuccess) rc = TMVP_EHIP;
        S.in.release();
        S.out.release();
        S.h_in.release();
        S.h_out.release();
        S.blocks.release();
        if (S.stream) (void)hipStreamDestroy(S.stream);
        S.stream = nullptr;
        const int rc2 = tmvp_destroy(S.ctx);
        S.ctx = nullptr;
        if (!rc) rc = rc2;
    }
    delete[] S.rnd;
    S.rnd = nullptr;
    S.rnd_bytes = 0;
    return rc;
}

void saber_enc(uint8_t mode, uint8_t *h_k, uint8_t *h_pk, uint8_t *h_c)
{
    HostState &S = state();
    std::lock_guard<std::mutex> g(S.mu);
    S.status = host_enc(S, S.saber_set, S.saber_batch, mode, h_k, h_pk, h_c);
}

void saber_dec(uint8_t mode, uint8_t *h_c, uint8_t *h_pk, uint8_t *h_sk, uint8_t *h_k)
{
    (void)h_pk;
    HostState &S = state();
    std::lock_guard<std::mutex> g(S.mu);
    S.status = host_dec(S, S.saber_set, S.saber_batch, mode, h_c, h_sk, h_k);
}

void SABLE_enc(uint8_t *h_k, uint8_t *h_pk, uint8_t *h_c, int mode)
{
    HostState &S = state();
    std::lock_guard<std::mutex> g(S.mu);
    S.status = host_enc(S, S.sable_set, S.sable_batch, mode, h_k, h_pk, h_c);
}

void SABLE_dec(uint8_t *h_c, uint8_t *h_pk, uint8_t *h_sk, uint8_t *h_k, int mode)
{
    (void)h_pk;
    HostState &S = state();
    std::lock_guard<std::mutex> g(S.mu);
    S.status = host_dec(S, S.sable_set, S.sable_batch, mode, h_c, h_sk, h_k);
}

} // extern "C"
