// quantize.hip — the requantizer's block quantization on the GPU
// (ehip_quantize_rows), which replaces the per-row quantizer loops of
// quantize_tensor (src/quant.c:26-57) called by ember_quantize_file.
//
// fp32 rows stream from the caller's (mapped) host memory through pinned slots
// (QuantCall: one for a call of up to 24 MiB, one of 1 MiB per host thread for
// longer ones); the encoded blocks come back the same way.  Each GPU thread
// encodes one 32-weight block with the reference's arithmetic
// (src/kernels.c:73-115), so the blocks equal the host quantizers' byte for
// byte:
//   Q8_0: amax over |x| (first maximum), d = amax/127, inverse from the
//         unrounded d (0 when d is 0), codes round half away from zero,
//         clamped to +-127, d stored as fp16 (RNE).
//   Q4_0: v = the element of largest magnitude (first one), d = v/-8,
//         inverse 1/d (0 when d is 0), codes (int)(x*inv + 8.5) truncated
//         and clamped to 0..15, element i in the low and element i+16 in the
//         high nibble of byte i.
// When a block's largest magnitude is below about 3.7e-37 (Q8_0) or 2.4e-38
// (Q4_0), 1/d overflows to infinity and x*inv is infinite or NaN; a block
// holding an infinity has d infinite and inverse 0, so its infinite (and NaN)
// elements give NaN products.  The reference converts with (int)lroundf(p)
// (Q8_0) and (int)(p + 8.5f) (Q4_0); on x86-64 those give LONG_MIN and
// INT_MIN for such products, whose int values clamp to code 0 in both
// encodings whatever the sign.  The device's conversions would saturate
// instead, so such products take the host's result explicitly.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdio>
#include <cstring>
#include <exception>
#include <thread>
#include <vector>

#include "../../../include/ehip.h"
#include "kernels.h"
#include "staging.h"

namespace {

using namespace ehip;

// float -> fp16 bits, round to nearest even, with the host conversion's
// handling of every input: magnitudes that round past 65504, infinities and
// NaNs give a signed infinity; below 2^-14 the result is a multiple of 2^-24.
__device__ __forceinline__ uint16_t half_bits(float f) {
    uint32_t u = __float_as_uint(f);
    const uint32_t sign = (u >> 16) & 0x8000u;
    uint32_t a = u & 0x7fffffffu;
    if (a >= 0x477ff000u) return (uint16_t)(sign | 0x7c00u);
    if (a < 0x38800000u) return (uint16_t)(sign | (uint32_t)rintf(__uint_as_float(a) * 16777216.0f));
    a += 0xfffu + ((a >> 13) & 1u);
    return (uint16_t)(sign | ((a - 0x38000000u) >> 13));
}

// One thread per block: x holds nblk * 32 floats (16-byte aligned), out
// receives nblk encoded blocks of 34 (Q8_0) or 18 (Q4_0) bytes.
template <int DT>
__global__ __launch_bounds__(256) void k_quant_blocks(const float *__restrict__ x, size_t nblk,
                                                      uint16_t *__restrict__ out) {
    constexpr int HALVES = DT == DT_Q8 ? 17 : 9;   // block size in 16-bit words
    for (size_t b = blockIdx.x * (size_t)blockDim.x + threadIdx.x; b < nblk; b += (size_t)gridDim.x * blockDim.x) {
        float v[32];
        const float4 *src = reinterpret_cast<const float4 *>(x + b * 32);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float4 t = src[i];
            v[4 * i] = t.x; v[4 * i + 1] = t.y; v[4 * i + 2] = t.z; v[4 * i + 3] = t.w;
        }
        uint16_t *o = out + b * HALVES;
        if (DT == DT_Q8) {
            float amax = 0.0f;
#pragma unroll
            for (int i = 0; i < 32; i++) amax = fabsf(v[i]) > amax ? fabsf(v[i]) : amax;
            const float d = amax / 127.0f;
            const float inv = d > 0.0f ? 1.0f / d : 0.0f;
            o[0] = half_bits(d);
            auto code = [inv](float x) {
                // (int)lroundf(p): the rounded value (half away from zero)
                // reduced to its low 32 bits, and 0 (the low bits of
                // LONG_MIN) for NaN, infinities and |p| >= 2^63
                const float r = roundf(__fmul_rn(x, inv));
                int q = fabsf(r) < 0x1p63f ? (int)(long long)r : 0;
                q = q > 127 ? 127 : q < -127 ? -127 : q;
                return (uint32_t)q & 0xffu;
            };
#pragma unroll
            for (int i = 0; i < 16; i++) o[1 + i] = (uint16_t)(code(v[2 * i]) | (code(v[2 * i + 1]) << 8));
        } else {
            float amax = 0.0f, vmax = 0.0f;
#pragma unroll
            for (int i = 0; i < 32; i++)
                if (fabsf(v[i]) > amax) { amax = fabsf(v[i]); vmax = v[i]; }
            const float d = vmax / -8.0f;
            const float inv = d != 0.0f ? 1.0f / d : 0.0f;
            o[0] = half_bits(d);
            uint32_t byte[16];
            auto code = [inv](float x) {
                const float t = __fadd_rn(__fmul_rn(x, inv), 8.5f);
                const int q = fabsf(t) < 0x1p31f ? (int)t : 0;
                return (uint32_t)(q < 0 ? 0 : q > 15 ? 15 : q);
            };
#pragma unroll
            for (int i = 0; i < 16; i++) byte[i] = code(v[i]) | (code(v[i + 16]) << 4);
#pragma unroll
            for (int i = 0; i < 8; i++) o[1 + i] = (uint16_t)(byte[2 * i] | (byte[2 * i + 1] << 8));
        }
    }
}

// A piece: blocks of the jobs of one encoding, in the jobs' order (a job's rows
// are contiguous in both buffers, and a block never spans two), so one launch
// and one DMA each way serve many small matrices: 100 of 32 x 64 2.5 ms with a
// piece each, 0.2 together.
struct Segment { int job; size_t b0, n; };
struct Piece { size_t seg, nseg, blocks; int dtype; };
constexpr int64_t ROW_MAX = (int64_t)32 << 20;         // bytes of a row at most
constexpr int QUANT_STREAMS = 4;
// Calls of up to ALONE_BLOCKS (24 MiB of fp32) are a piece per encoding, which
// the calling thread copies itself; longer ones go in pieces of
// PIECE_BLOCKS (1 MiB) over several threads, whose start, streams and smaller
// copies cost about 1 ms a call.  One matrix, one piece against pieces over
// threads: 4 MiB 0.4 ms against 1.6, 12 MiB 0.75 against 1.5, 24 MiB 1.4
// against 1.9, 32 MiB 2.2 against 2.2; from 40 MiB on one piece falls to 20 ms.
constexpr size_t ALONE_BLOCKS = 196608, PIECE_BLOCKS = 8192;

// The call's pieces and staging: each worker thread has a pinned and a device
// slot of one piece each way, and takes the next piece when its last is done:
// copy in, DMA, one launch, DMA back, copy out.  The workers' host copies, the
// DMAs and the kernels overlap, and a long call's slots are not sized by its
// matrices: pinning dominates a call on a few of them (the feed-forward
// matrices of a 0.6B layer, 37.7 MB: three pinned slots of 32 MB 6.9 ms a call).
struct QuantCall {
    const EhipQuantJob *jobs;
    std::vector<Segment> segs;
    std::vector<Piece> pieces;
    size_t in_bytes = 0, out_bytes = 0;   // of a slot
    int workers = 0;
    uint8_t *pin = nullptr, *dev = nullptr;
    hipStream_t st[QUANT_STREAMS] = {};
    std::vector<hipEvent_t> ev;
    std::atomic<size_t> next{0};
    std::atomic<const char *> failure{nullptr};

    bool open(const EhipQuantJob *j, int n_jobs, size_t total) {
        jobs = j;
        const bool alone = total <= ALONE_BLOCKS;
        const size_t piece = alone ? ALONE_BLOCKS : PIECE_BLOCKS;
        size_t most = 0;
        for (int dtype : { DT_Q8, DT_Q4 })
            for (int i = 0; i < n_jobs; i++) {
                const size_t nblk = jobs[i].dtype == dtype ? (size_t)jobs[i].rows * (jobs[i].cols / 32) : 0;
                for (size_t b = 0; b < nblk;) {
                    if (pieces.empty() || pieces.back().blocks == piece || pieces.back().dtype != dtype)
                        pieces.push_back({ segs.size(), 0, 0, dtype });
                    Piece &p = pieces.back();
                    const size_t n = std::min(piece - p.blocks, nblk - b);
                    segs.push_back({ i, b, n });
                    p.nseg++;
                    p.blocks += n;
                    b += n;
                    most = std::max(most, p.blocks);
                }
            }
        in_bytes = most * 128;
        out_bytes = (most * 34 + 127) & ~(size_t)127;
        workers = alone ? 1 : (int)std::min<size_t>(staging_threads(), pieces.size());
        const size_t bytes = (in_bytes + out_bytes) * workers;
        if (hipHostMalloc(reinterpret_cast<void **>(&pin), bytes, hipHostMallocDefault) != hipSuccess) { pin = nullptr; return false; }
        if (hipMalloc(reinterpret_cast<void **>(&dev), bytes) != hipSuccess) { dev = nullptr; return false; }
        for (int i = 0; i < std::min(workers, QUANT_STREAMS); i++)
            if (hipStreamCreateWithFlags(&st[i], hipStreamNonBlocking) != hipSuccess) { st[i] = nullptr; return false; }
        for (int i = 0; i < workers; i++) {
            hipEvent_t e;
            if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return false;
            ev.push_back(e);
        }
        return true;
    }
    ~QuantCall() {
        for (hipStream_t s : st)
            if (s) (void)hipStreamSynchronize(s);
        for (hipEvent_t e : ev) (void)hipEventDestroy(e);
        if (dev) (void)hipFree(dev);
        if (pin) (void)hipHostFree(pin);
        for (hipStream_t s : st)
            if (s) (void)hipStreamDestroy(s);
    }

    // piece p through worker w's slot; what failed, or null
    const char *piece(int w, const Piece &p) {
        const size_t ob = p.dtype == DT_Q8 ? 34 : 18, slot = (in_bytes + out_bytes) * w;
        uint8_t *pin_in = pin + slot, *pin_out = pin_in + in_bytes, *dev_in = dev + slot, *dev_out = dev_in + in_bytes;
        const hipStream_t s = st[w % QUANT_STREAMS];
        const Segment *g0 = &segs[p.seg], *g1 = g0 + p.nseg;
        uint8_t *in = pin_in;
        for (const Segment *g = g0; g < g1; in += g->n * 128, g++)
            memcpy(in, reinterpret_cast<const uint8_t *>(jobs[g->job].src) + g->b0 * 128, g->n * 128);
        bool ok = hipMemcpyAsync(dev_in, pin_in, p.blocks * 128, hipMemcpyHostToDevice, s) == hipSuccess;
        const int grid = (int)((p.blocks + 255) / 256);
        const float *x = reinterpret_cast<const float *>(dev_in);
        uint16_t *o = reinterpret_cast<uint16_t *>(dev_out);
        if (p.dtype == DT_Q8) k_quant_blocks<DT_Q8><<<grid, 256, 0, s>>>(x, p.blocks, o);
        else k_quant_blocks<DT_Q4><<<grid, 256, 0, s>>>(x, p.blocks, o);
        ok = hipGetLastError() == hipSuccess && ok;
        ok = ok && hipMemcpyAsync(pin_out, dev_out, p.blocks * ob, hipMemcpyDeviceToHost, s) == hipSuccess &&
             hipEventRecord(ev[w], s) == hipSuccess;
        if (!ok) return "requantizer: queueing a slot's copies or kernels failed";
        if (hipEventSynchronize(ev[w]) != hipSuccess) return "requantizer: waiting for a slot failed";
        const uint8_t *out = pin_out;
        for (const Segment *g = g0; g < g1; out += g->n * ob, g++)
            memcpy(static_cast<uint8_t *>(jobs[g->job].dst) + g->b0 * ob, out, g->n * ob);
        return nullptr;
    }
    // what fails first ends every worker at its next piece; the destructor
    // waits for what is on its way
    void work(int w) {
        if (hipSetDevice(0) != hipSuccess) failure = "hipSetDevice(0) failed: no usable GPU";
        for (size_t i; !failure && (i = next.fetch_add(1)) < pieces.size();)
            if (const char *e = piece(w, pieces[i])) failure = e;
    }
    bool run() {
        std::vector<std::thread> ts;
        try {
            for (int w = 1; w < workers; w++) ts.emplace_back(&QuantCall::work, this, w);
        } catch (const std::exception &) {   // no further thread: those that run share the pieces
        }
        work(0);
        for (std::thread &t : ts) t.join();
        return !failure;
    }
};

}  // namespace

extern "C" int ehip_quantize_rows(const EhipQuantJob *jobs, int n_jobs) {
    if (n_jobs < 0 || (n_jobs > 0 && !jobs)) { set_error_text("ehip_quantize_rows: no jobs"); return -1; }
    size_t total = 0;
    for (int i = 0; i < n_jobs; i++) {
        const EhipQuantJob &j = jobs[i];
        char msg[160];
        if (j.dtype != DT_Q8 && j.dtype != DT_Q4) {
            snprintf(msg, sizeof msg, "ehip_quantize_rows: job %d: target dtype %d is not Q8_0 or Q4_0", i, j.dtype);
            set_error_text(msg);
            return -1;
        }
        if (j.cols <= 0 || j.cols % 32 || (int64_t)j.cols * 4 > ROW_MAX || j.rows < 0 ||
            (j.rows > 0 && (!j.src || !j.dst))) {
            snprintf(msg, sizeof msg, "ehip_quantize_rows: job %d: %lld rows of %d values cannot be quantized", i,
                     (long long)j.rows, j.cols);
            set_error_text(msg);
            return -1;
        }
        total += (size_t)j.rows * j.cols * 4;
    }
    if (total == 0) return 0;
    if (hipSetDevice(0) != hipSuccess) { set_error_text("hipSetDevice(0) failed: no usable GPU"); return -1; }
    try {
        QuantCall q;
        if (!q.open(jobs, n_jobs, total / 128)) { set_error_text("requantizer: allocating the staging buffers failed"); return -1; }
        if (q.run()) return 0;
        set_error_text(q.failure.load());
    } catch (const std::exception &) {
        set_error_text("requantizer: out of host memory");
    }
    return -1;
}
