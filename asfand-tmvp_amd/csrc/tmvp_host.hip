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
        if (hipHostMalloc(&p, bytes, hipHostMallocDefault) != hipSuccess) {
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

// Up to this many bytes each way go through page-locked buffers and copy
// kernels on the call's own queue (page-locked buffers of the caller go directly,
// see route), the inputs in pieces, so that the bus moves one while the next is
// copied on the host.  The runtime's copy of pageable memory costs a
// synchronisation each (four and one for the status word: 15 to 32 us apiece, 110
// us around a Sable type 2 encapsulation of 512 instances that runs for 95), the
// memcpy of half a megabyte 4 to 12 us and its copy kernel 10.  Encapsulation and
// decapsulation, runtime's copies -> these: Saber 32 instances 267 -> 128 and 226 ->
// 113 us, 512: 325 -> 171 and 302 -> 163, 2048: 485 -> 378 and 442 -> 351, 8192 (8 MB
// in; the decapsulations' 27 MB are past the limit): 1036 -> 890 us.
// Pieces of 256 KB and 1 MB: 321 and 316 us for 2048 decapsulations that took 296.
// The limit bounds the page-locked memory held; the outputs' copy is not in pieces,
// so the gain ends there anyway (16384 encapsulations: 1821 -> 1785).
constexpr size_t kStageBytes = 16u << 20;
constexpr size_t kChunk = 512u << 10;

// Words that a move leaves in page-locked memory.
struct Words {
    int *status_to;    // the context's status word goes here
    const int *status;
    int *read;         // 1 once every byte of src has been read; `blocks` counts the workgroups that have
    int *blocks;       // (0 between launches)
};

// n16 16-byte units from src to dst, one of them in page-locked host memory, and
// W's words (null: none).  Four loads in flight per thread.
constexpr int kMoveThreads = 256;
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
    if (W.read) {
        __syncthreads(); // every load of the workgroup has returned: its stores are on their way
        if (threadIdx.x == 0 && atomicAdd(W.blocks, 1) == (int)gridDim.x - 1) {
            *W.blocks = 0;
            __hip_atomic_store(W.read, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

int move_bytes(void *dst, const void *src, size_t bytes, const Words &W, hipStream_t st)
{
    size_t blocks = (bytes + 64 * kMoveThreads - 1) / (64 * kMoveThreads);
    if (blocks > 256) blocks = 256;
    if (blocks == 0) blocks = 1; // the status word alone
    hipLaunchKernelGGL(move_kernel, dim3((unsigned)blocks), dim3(kMoveThreads), 0, st, static_cast<uint4 *>(dst),
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
    const hipError_t e = hipPointerGetAttributes(&a, h);
    const hipError_t f = hipPointerGetAttributes(&z, static_cast<const uint8_t *>(h) + n - 1);
    (void)hipGetLastError(); // pageable memory may report an error: clear it
    if (e != hipSuccess || a.type == hipMemoryTypeUnregistered) return part;
    if (a.type != hipMemoryTypeHost) {
        part.route = kRuntime;
    } else if (f == hipSuccess && z.type == hipMemoryTypeHost && a.devicePointer &&
               static_cast<uint8_t *>(z.devicePointer) - static_cast<uint8_t *>(a.devicePointer) == (ptrdiff_t)(n - 1) &&
               ((uintptr_t)a.devicePointer & 15) == 0 && n >= kDirectBytes) {
        part.route = kDirect;
        part.dev = a.devicePointer;
    }
    return part;
}

// The secret bytes of an operand of n rows: of each row's `stride`, the first
// `head` and the last `tail`.
struct Secret {
    size_t n, stride, head, tail;
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
    PinnedBuf h_in, h_out;  // the same in page-locked memory; a word follows each: inputs read, status
    DevBuf blocks;          // Words::blocks
    uint8_t *wipe = nullptr; // staged inputs of this call that hold `secret`, not yet cleared
    Secret secret{};
    int *inputs_read = nullptr;
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

// Which of a call's operands are staged in buf (with `extra` bytes behind them).
// Beyond kStageBytes everything is left to the runtime, whose engine outruns the
// copy kernel on page-locked inputs there (8192 Saber decapsulations, 27 MB in: 687
// against 736 us).
Staging staging(PinnedBuf &buf, Part &a, Part &b, size_t extra)
{
    if (a.n + b.n > kStageBytes) a.route = b.route = kRuntime;
    Staging g{a, b, a.route == kStaged ? 0 : a.n};
    if (a.route != kStaged) g.a.n = 0;
    if (b.route != kStaged) g.b.n = 0;
    if (!buf.reserve(g.n() + extra)) {
        if (g.a.n) a.route = kRuntime;
        if (g.b.n) b.route = kRuntime;
        g.a.n = g.b.n = 0;
    }
    return g;
}

// The two inputs to S.in; the second one's secret bytes do not stay in the
// staging (wipe_inputs).
int copy_in(HostState &S, Part a, Part b, const Secret &secret)
{
    const Staging g = staging(S.h_in, a, b, 16);
    S.wipe = nullptr;
    if (g.b.n) {
        S.wipe = S.h_in.u8() + g.a.n;
        S.secret = secret;
        S.inputs_read = reinterpret_cast<int *>(S.h_in.u8() + g.n());
        *S.inputs_read = 0;
    }
    const Part *const parts[2] = {&a, &b};
    uint8_t *const at_dev[2] = {S.in.u8(), S.in.u8() + a.n};
    for (int i = 0; i < 2; i++) // the bus beside the host's copies below
        if (parts[i]->route == kDirect) {
            const int rc = move_bytes(at_dev[i], parts[i]->dev, parts[i]->n, {}, S.stream);
            if (rc) return rc;
        }
    for (size_t at = 0, n = g.n(); at < n; at += kChunk) { // and beside the next piece's memcpy
        const size_t end = at + kChunk < n ? at + kChunk : n;
        if (at < g.a.n)
            memcpy(S.h_in.u8() + at, static_cast<uint8_t *>(g.a.h) + at, (end < g.a.n ? end : g.a.n) - at);
        if (end > g.a.n) {
            const size_t from = at > g.a.n ? at : g.a.n;
            memcpy(S.h_in.u8() + from, static_cast<uint8_t *>(g.b.h) + (from - g.a.n), end - from);
        }
        Words W{};
        if (end == n && g.b.n) { // the pieces before it have been read when this one starts
            W.read = reinterpret_cast<int *>(static_cast<uint8_t *>(S.h_in.dev) + n);
            W.blocks = static_cast<int *>(S.blocks.p);
        }
        const int rc = move_bytes(S.in.u8() + g.skip + at, static_cast<uint8_t *>(S.h_in.dev) + at, end - at, W, S.stream);
        if (rc) return rc;
    }
    for (int i = 0; i < 2; i++)
        if (parts[i]->route == kRuntime && parts[i]->n &&
            hipMemcpyAsync(at_dev[i], parts[i]->h, parts[i]->n, hipMemcpyHostToDevice, S.stream) != hipSuccess)
            return TMVP_EHIP;
    return TMVP_OK;
}

// Clears the call's secrets in the staged inputs.  Called when everything has
// been launched, so it works while the kernels run and costs the call nothing until
// clearing takes longer than they do: Saber decapsulations, 1.3 KB of secrets each,
// 512 instances 163 -> 164 us, 2048 352 -> 379, 4096 530 -> 585 (the copy kernels
// clearing over the bus: 182, 412 and 650).  If the inputs' word does not come in
// time, it is left to the call after the wait (`done`).
void wipe_inputs(HostState &S, bool done)
{
    if (!S.wipe) return;
    for (int spin = 0; !done && spin < 100000; spin++)
        done = __atomic_load_n(S.inputs_read, __ATOMIC_ACQUIRE) != 0;
    if (!done) return;
    uint8_t *row = S.wipe;
    S.wipe = nullptr;
    for (size_t i = 0; i < S.secret.n; i++, row += S.secret.stride) {
        explicit_bzero(row, S.secret.head);
        if (S.secret.tail) explicit_bzero(row + S.secret.stride - S.secret.tail, S.secret.tail);
    }
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
// not stay in the staging.
int copy_out(HostState &S, Part a, Part b)
{
    const Staging g = staging(S.h_out, a, b, 16);
    const Part *const parts[2] = {&a, &b};
    uint8_t *const at_dev[2] = {S.out.u8(), S.out.u8() + a.n};
    int rc = TMVP_OK;
    for (int i = 0; i < 2 && !rc; i++) {
        if (parts[i]->route == kDirect)
            rc = move_bytes(parts[i]->dev, at_dev[i], parts[i]->n, {}, S.stream);
        else if (parts[i]->route == kRuntime && parts[i]->n &&
                 hipMemcpyAsync(parts[i]->h, at_dev[i], parts[i]->n, hipMemcpyDeviceToHost, S.stream) != hipSuccess)
            rc = TMVP_EHIP;
    }
    if (rc || S.h_out.n < g.n() + 16) {
        const int rc2 = finish(S);
        return rc ? rc : rc2;
    }
    const size_t n = g.n(); // a multiple of 16; the status word behind it
    int *const flag = reinterpret_cast<int *>(S.h_out.u8() + n);
    *flag = 1; // until the kernel has written it
    Words W{};
    W.status_to = reinterpret_cast<int *>(static_cast<uint8_t *>(S.h_out.dev) + n);
    W.status = tmvp::ctx_status_word(S.ctx);
    rc = move_bytes(S.h_out.dev, S.out.u8() + g.skip, n, W, S.stream);
    wipe_inputs(S, false);
    if (hipStreamSynchronize(S.stream) != hipSuccess) rc = TMVP_EHIP;
    wipe_inputs(S, true);
    if (!rc && g.a.n) memcpy(g.a.h, S.h_out.u8(), g.a.n);
    if (!rc && g.b.n) memcpy(g.b.h, S.h_out.u8() + g.a.n, g.b.n);
    explicit_bzero(S.h_out.u8() + g.a.n, g.b.n);
    if (rc) return rc;
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
    rc = copy_in(S, route(h_pk, npk), route(rnd, B * 32), {1, B * 32, B * 32, 0});
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
                 {B, (size_t)P.sk_bytes, (size_t)(P.sable ? P.l * 64 : P.l * P.eq * 32), 32}); // s and z
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
