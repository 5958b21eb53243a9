/* The reusable streaming-decode context: LZ4 blocks from host memory,
 * decoded on the device through cudec_lz4_decompress_batch.
 *
 * Contract: include/cudec.h:140-218 (iderex/cudec's src/stream.cpp:
 * ValidateStreamArgs 196-216, StampNotDecoded 218-230, DecodeStreamCtx
 * 238-488, the entry points 492-593, CopyWaveToHost 163-184).
 *
 * This implementation's shape: the call is split into waves, of a staging
 * budget charged to its largest chunk (so a hostile size mix cannot inflate
 * staging) and, in large calls, of an eighth of its chunks. Up to four waves
 * are in hand, each with a stream and staging of its own (pinned and device
 * source, and for host output device and pinned destination): while the
 * device takes one in, decodes another and gives a third back, host threads
 * pack the next and unpack an earlier one. Host output comes back as one
 * asynchronous copy per wave into pinned memory, then exactly bytes_written
 * bytes per chunk go to the caller. Everything but the threads grows on
 * demand and is kept for the next call.
 *
 * What bounds it is the copies between the caller's memory and pinned memory
 * (277 MB for 2048 chunks of 16 to 256 KiB, 95 in and 182 out), which one
 * thread and one wave did in a row with the transfers: 18.3 ms, 5.5 so. */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <new>
#include <vector>

#include "cudec.h"
#include "hip_owner.h"
#include "host_copy.h"

namespace cudec_amd {

/* One chunk per wave and at most INT32_MAX waves (src/batch_limits.h:28 for
 * wave64); the batch entry applies the same bound. */
constexpr size_t kStreamMaxChunks = static_cast<size_t>(INT32_MAX) * 64;
/* Staging charged per wave (pinned + device source, device + pinned
 * destination on the host-output path), against the largest chunk. */
constexpr size_t kWaveBudget = size_t{1} << 30;
constexpr size_t kWaveChunksMax = 16384;
/* Waves of a large call: enough to overlap, and none so small that its
 * launch and its largest chunk take longer than its transfers. */
constexpr size_t kWavesWanted = 8;
constexpr size_t kWaveBytesMin = size_t{24} << 20;
constexpr int kSlots = 4;

struct Slot {
    Stream stream;
    PinnedRegion p_src;
    DeviceRegion d_src;
    PinnedRegion p_meta;
    DeviceRegion d_meta;
    DeviceRegion d_dst;
    PinnedRegion p_dst;
    Event landed;  /* this slot's results and output are in pinned memory */
    bool landed_pending = false;
    size_t begin = 0, count = 0, meta_stride = 0;
};

}  // namespace cudec_amd

struct cudec_stream_ctx {
    cudec_amd::Slot slot[cudec_amd::kSlots];
    int device = 0;    /* the streams' */
    bool once = false; /* the context of a single call */
    cudec_amd::DeviceRegion d_results;
    cudec_amd::PinnedRegion p_results;
    bool poisoned = false;
};

namespace cudec_amd {
namespace {

cudec_status validate_stream_args(const void* const* h_src_ptrs, const size_t* h_src_sizes,
                                  void* const* dst_ptrs, const size_t* dst_caps,
                                  size_t chunk_count, cudec_mem_space dst_space,
                                  const cudec_chunk_result* h_results) {
    if (h_src_ptrs == nullptr || h_src_sizes == nullptr || dst_ptrs == nullptr ||
        dst_caps == nullptr || h_results == nullptr || chunk_count == 0 ||
        chunk_count > kStreamMaxChunks ||
        (dst_space != CUDEC_MEM_HOST && dst_space != CUDEC_MEM_DEVICE)) {
        return CUDEC_ERR_INVALID_ARGUMENT;
    }
    for (size_t i = 0; i < chunk_count; i++) {
        if ((h_src_ptrs[i] == nullptr && h_src_sizes[i] != 0) ||
            (dst_ptrs[i] == nullptr && dst_caps[i] != 0)) {
            return CUDEC_ERR_INVALID_ARGUMENT;
        }
    }
    return CUDEC_OK;
}

void stamp(cudec_chunk_result* r, size_t n, cudec_status st) {
    for (size_t i = 0; i < n; i++) {
        r[i].status = static_cast<int32_t>(st);
        r[i].reserved = 0;
        r[i].bytes_written = 0;
    }
}

/* Whether a host destination of the call lies over the source of a later
 * chunk or over another destination: programs decode within one arena, or
 * many chunks into one buffer of which they want the last, or none. (Over its
 * own source or an earlier one is no matter: those are read by then.) 3 ns a
 * chunk where buffers ascend, up to 140 where they lie in any order. */
bool buffers_meet(const void* const* src, const size_t* src_sizes, void* const* dst,
                  const size_t* caps, size_t n) {
    struct Range {
        uintptr_t begin, end;
        size_t chunk;
    };
    const auto range = [](const void* p, size_t len, size_t i) {
        const uintptr_t b = reinterpret_cast<uintptr_t>(p);
        return Range{b, UINTPTR_MAX - b < len ? UINTPTR_MAX : b + len, i};
    };
    size_t total = 0;
    for (size_t i = 0; i < n && total < CopyCrew::kBytesPerHelper; i++) {
        total += src_sizes[i] < CopyCrew::kBytesPerHelper ? src_sizes[i]
                                                          : CopyCrew::kBytesPerHelper;
        total += caps[i] < CopyCrew::kBytesPerHelper ? caps[i] : CopyCrew::kBytesPerHelper;
    }
    if (total < CopyCrew::kBytesPerHelper) {
        return false; /* one wave and one thread in any case */
    }
    std::vector<Range> out;
    out.reserve(n);
    for (size_t i = 0; i < n; i++) {
        if (caps[i] != 0) {
            out.push_back(range(dst[i], caps[i], i));
        }
    }
    if (out.empty()) {
        return false;
    }
    const auto before = [](const Range& x, const Range& y) { return x.begin < y.begin; };
    if (!std::is_sorted(out.begin(), out.end(), before)) {
        std::sort(out.begin(), out.end(), before);
    }
    for (size_t k = 1; k < out.size(); k++) {
        if (out[k].begin < out[k - 1].end) {
            return true;
        }
    }
    /* from the last one that ends at or before the source, which is near the
     * one of the source before where buffers ascend */
    size_t steps = 4 * n; /* sources that cover ever so many destinations: true */
    size_t k = 0;
    for (size_t i = 0; i < n; i++) {
        const Range s = range(src[i], src_sizes[i], i);
        if (s.begin == s.end || s.begin >= out.back().end || s.end <= out.front().begin) {
            continue;
        }
        if (out[k].begin > s.begin || (k + 4 < out.size() && out[k + 4].begin <= s.begin)) {
            const auto o = std::upper_bound(out.begin(), out.end(), s, before);
            k = o == out.begin() ? 0 : static_cast<size_t>(o - out.begin()) - 1;
        }
        while (k < out.size() - 1 && out[k].end <= s.begin) {
            k++;
        }
        for (size_t j = k; j < out.size() && out[j].begin < s.end; j++) {
            if (out[j].end > s.begin && (out[j].chunk < i || steps-- == 0)) {
                return true;
            }
        }
    }
    return false;
}

size_t choose_wave(const size_t* src_sizes, const size_t* caps, size_t n, bool host_out,
                   bool in_order) {
    size_t biggest = 1, total = 0;
    for (size_t i = 0; i < n; i++) {
        size_t b = src_sizes[i];
        if (host_out) {
            b = SIZE_MAX - b < caps[i] ? SIZE_MAX : b + caps[i];
        }
        if (b > biggest) {
            biggest = b;
        }
        total = SIZE_MAX - total < b ? SIZE_MAX : total + b;
    }
    size_t wave = kWaveBudget / biggest;
    if (wave == 0) {
        wave = 1;
    }
    if (wave > kWaveChunksMax) {
        wave = kWaveChunksMax;
    }
    size_t parts = in_order ? 1 : total / kWaveBytesMin;
    parts = parts < 1 ? 1 : parts > kWavesWanted ? kWavesWanted : parts;
    const size_t part = (n + parts - 1) / parts;
    return wave > part ? part : wave;
}

/* Unpacks one landed host-output wave: exactly bytes_written bytes per chunk
 * into the caller's buffer. A device-reported length beyond the chunk's
 * capacity is a device fault, never a copy length (src/stream.cpp:163-184). */
cudec_status unpack_wave(const Slot& s, cudec_chunk_result* pres, void* const* dst_ptrs,
                         const size_t* caps, CopyCrew& crew) {
    const unsigned char* base = static_cast<const unsigned char*>(s.p_dst.data());
    const unsigned char* dd = static_cast<const unsigned char*>(s.d_dst.data());
    const void* const* m_dst = reinterpret_cast<const void* const*>(
        static_cast<const unsigned char*>(s.p_meta.data()) + 2 * s.meta_stride);
    size_t good = 0;
    while (good < s.count && pres[s.begin + good].bytes_written <= caps[s.begin + good]) {
        good++;
    }
    crew.each(good, [&](size_t j) {
        const cudec_chunk_result& r = pres[s.begin + j];
        if (r.status == CUDEC_OK && r.bytes_written != 0) {
            std::memcpy(dst_ptrs[s.begin + j],
                        base + (static_cast<const unsigned char*>(m_dst[j]) - dd),
                        static_cast<size_t>(r.bytes_written));
        }
    });
    if (good != s.count) {
        cudec_chunk_result& r = pres[s.begin + good];
        r.status = static_cast<int32_t>(CUDEC_ERR_CUDA);
        r.reserved = 0;
        r.bytes_written = 0;
        return CUDEC_ERR_CUDA;
    }
    return CUDEC_OK;
}

/* Bytes (of the device's, and as many pinned) that the slots hold once the
 * first `used` hold waves of src and dst bytes. */
size_t staging(const cudec_stream_ctx& ctx, size_t used, size_t src, size_t dst) {
    size_t sum = 0;
    for (size_t k = 0; k < kSlots; k++) {
        const size_t hs = ctx.slot[k].d_src.capacity(), hd = ctx.slot[k].d_dst.capacity();
        const size_t s = k < used && src > hs ? src : hs, d = k < used && dst > hd ? dst : hd;
        const size_t both = SIZE_MAX - s < d ? SIZE_MAX : s + d;
        sum = SIZE_MAX - sum < both ? SIZE_MAX : sum + both;
    }
    return sum;
}

/* Gives the first `used` slots their streams and events, on the context's
 * device.
 *
 * A context that is kept gets all four where it is made: the runtime puts a
 * new stream on the hardware queue with the fewest, so that four in a row lie
 * on its four queues, and streams that share one do not overlap (three
 * contexts for 2048 chunks of 16 to 256 KiB each, which made the first stream
 * with the context and the others in the first call: 5.8 ms a call, 5.4 so).
 * That is 134 us instead of 34, so the context of a single call gets no more
 * than the call uses. */
hipError_t open_slots(cudec_stream_ctx& ctx, size_t used) {
    int now = 0;
    hipError_t e = hipGetDevice(&now);
    if (e == hipSuccess && now != ctx.device) {
        e = hipSetDevice(ctx.device);
    }
    for (size_t k = 0; k < used && e == hipSuccess; k++) {
        Slot& s = ctx.slot[k];
        if (!s.stream) {
            e = make_stream(s.stream);
        }
        if (e == hipSuccess && !s.landed) {
            e = make_sync_event(s.landed);
        }
    }
    if (now != ctx.device) {
        const hipError_t back = hipSetDevice(now);
        e = e == hipSuccess ? back : e;
    }
    return e;
}

/* Waits, at the latest where the call ends, whichever way it does, for
 * everything its slots' streams hold: nothing of a call outlives it. */
class Drain {
public:
    Drain(cudec_stream_ctx& ctx, size_t used) : ctx_(ctx), used_(used) {}
    ~Drain() { (void)now(); }
    Drain(const Drain&) = delete;
    Drain& operator=(const Drain&) = delete;

    hipError_t now() {
        hipError_t first = hipSuccess;
        for (; used_ != 0; used_--) {
            const hipError_t e = hipStreamSynchronize(ctx_.slot[used_ - 1].stream.get());
            first = first == hipSuccess ? e : first;
        }
        return first;
    }

private:
    cudec_stream_ctx& ctx_;
    size_t used_;
};

cudec_status decode_stream(cudec_stream_ctx& ctx, const void* const* h_src_ptrs,
                           const size_t* h_src_sizes, void* const* dst_ptrs,
                           const size_t* dst_caps, size_t n, cudec_mem_space space,
                           cudec_chunk_result* h_results) {
    const bool host_out = space == CUDEC_MEM_HOST;
    stamp(h_results, n, CUDEC_ERR_CUDA);
    /* buffers that meet keep the order that a call has with one thread and two
     * slots: a wave is as large as the budget lets it be, it is read whole
     * before its first byte is written, and chunks are written one after the
     * other */
    const bool in_order =
        host_out && buffers_meet(h_src_ptrs, h_src_sizes, dst_ptrs, dst_caps, n);
    const size_t wave = choose_wave(h_src_sizes, dst_caps, n, host_out, in_order);
    const size_t waves = (n + wave - 1) / wave;
    size_t max_src = 1, max_dst = 1, total = 0;
    for (size_t w = 0; w < waves; w++) {
        const size_t b = w * wave, e = b + wave < n ? b + wave : n;
        size_t ws = 0, wd = 0;
        for (size_t i = b; i < e; i++) {
            if (SIZE_MAX - ws < h_src_sizes[i]) {
                return CUDEC_ERR_CORRUPT_INPUT;
            }
            ws += h_src_sizes[i];
            if (host_out) {
                if (SIZE_MAX - wd < dst_caps[i]) {
                    return CUDEC_ERR_CORRUPT_INPUT;
                }
                wd += dst_caps[i];
            }
        }
        max_src = ws > max_src ? ws : max_src;
        max_dst = wd > max_dst ? wd : max_dst;
        total = SIZE_MAX - total < ws ? SIZE_MAX : total + ws;
        total = SIZE_MAX - total < wd ? SIZE_MAX : total + wd;
    }
    /* two slots where four would stage more than two full budgets, with what
     * the slots keep of earlier calls; that much is what a context keeps,
     * unless a chunk of this call is larger than a budget. Two as well where
     * the staging serves this call alone: making it and giving it back takes
     * longer than four waves in hand save (2048 chunks of 16 to 256 KiB: 20.9
     * ms with four, 11.8 with two; 100 000 of 0.1 to 2 KiB: 17.9 and 11.9) */
    size_t slots = in_order || ctx.once ? 2 : kSlots;
    size_t used = waves < slots ? waves : slots;
    const size_t wave_dst = host_out ? max_dst : 0;
    if (staging(ctx, used, max_src, wave_dst) > 2 * kWaveBudget) {
        slots = 2;
        used = waves < slots ? waves : slots;
        if (staging(ctx, used, max_src, wave_dst) > 2 * kWaveBudget) {
            for (size_t k = slots; k < kSlots; k++) {
                ctx.slot[k].p_src.release();
                ctx.slot[k].d_src.release();
                ctx.slot[k].p_dst.release();
                ctx.slot[k].d_dst.release();
            }
        }
    }
    if (n > SIZE_MAX / sizeof(cudec_chunk_result)) {
        return CUDEC_ERR_CORRUPT_INPUT;
    }
    const size_t meta_stride = wave * sizeof(void*);
    const size_t meta_bytes = 4 * meta_stride;
    const size_t res_bytes = n * sizeof(cudec_chunk_result);
    bool ok = open_slots(ctx, used) == hipSuccess;
    for (size_t k = 0; k < used && ok; k++) {
        Slot& s = ctx.slot[k];
        ok = s.p_src.reserve(max_src) == hipSuccess && s.d_src.reserve(max_src) == hipSuccess &&
             s.p_meta.reserve(meta_bytes) == hipSuccess &&
             s.d_meta.reserve(meta_bytes) == hipSuccess &&
             (!host_out || (s.d_dst.reserve(max_dst) == hipSuccess &&
                            s.p_dst.reserve(max_dst) == hipSuccess));
        s.landed_pending = false;
    }
    ok = ok && ctx.d_results.reserve(res_bytes) == hipSuccess &&
         ctx.p_results.reserve(res_bytes) == hipSuccess;
    if (!ok) {
        ctx.poisoned = true;
        return CUDEC_ERR_CUDA;
    }
    cudec_chunk_result* pres = static_cast<cudec_chunk_result*>(ctx.p_results.data());
    stamp(pres, n, CUDEC_ERR_CUDA);
    cudec_status failure = CUDEC_OK;
    Drain drain(ctx, used);
    CopyCrew crew(in_order ? 0 : total, n);

    for (size_t w = 0; w < waves && failure == CUDEC_OK; w++) {
        Slot& s = ctx.slot[w % slots];
        hipStream_t st = s.stream.get();
        /* the slot's previous wave must have landed, and on the host-output
         * path its output be unpacked, before reuse */
        if (s.landed_pending) {
            if (hipEventSynchronize(s.landed.get()) != hipSuccess) {
                failure = CUDEC_ERR_CUDA;
                break;
            }
            s.landed_pending = false;
            if (host_out) {
                failure = unpack_wave(s, pres, dst_ptrs, dst_caps, crew);
                if (failure != CUDEC_OK) {
                    break;
                }
            }
        }
        s.begin = w * wave;
        s.count = (s.begin + wave < n ? s.begin + wave : n) - s.begin;
        s.meta_stride = meta_stride;
        unsigned char* ps = static_cast<unsigned char*>(s.p_src.data());
        unsigned char* ds = static_cast<unsigned char*>(s.d_src.data());
        unsigned char* dd = static_cast<unsigned char*>(s.d_dst.data());
        unsigned char* pm = static_cast<unsigned char*>(s.p_meta.data());
        const void** m_src = reinterpret_cast<const void**>(pm);
        size_t* m_size = reinterpret_cast<size_t*>(pm + meta_stride);
        void** m_dst = reinterpret_cast<void**>(pm + 2 * meta_stride);
        size_t* m_cap = reinterpret_cast<size_t*>(pm + 3 * meta_stride);
        size_t so = 0, dof = 0;
        for (size_t j = 0; j < s.count; j++) {
            const size_t i = s.begin + j;
            m_src[j] = ds + so;
            m_size[j] = h_src_sizes[i];
            m_cap[j] = dst_caps[i];
            if (host_out) {
                m_dst[j] = dd + dof;
                dof += dst_caps[i];
            } else {
                m_dst[j] = dst_ptrs[i];
            }
            so += h_src_sizes[i];
        }
        crew.each(s.count, [&](size_t j) {
            if (m_size[j] != 0) {
                std::memcpy(ps + (static_cast<const unsigned char*>(m_src[j]) - ds),
                            h_src_ptrs[s.begin + j], m_size[j]);
            }
        });
        unsigned char* dm = static_cast<unsigned char*>(s.d_meta.data());
        cudec_chunk_result* dres = static_cast<cudec_chunk_result*>(ctx.d_results.data()) + s.begin;
        if ((so != 0 && hipMemcpyAsync(ds, ps, so, hipMemcpyHostToDevice, st) != hipSuccess) ||
            hipMemcpyAsync(dm, pm, meta_bytes, hipMemcpyHostToDevice, st) != hipSuccess) {
            failure = CUDEC_ERR_CUDA;
            break;
        }
        const cudec_status launched = cudec_lz4_decompress_batch(
            reinterpret_cast<const void* const*>(dm),
            reinterpret_cast<const size_t*>(dm + meta_stride),
            reinterpret_cast<void* const*>(dm + 2 * meta_stride),
            reinterpret_cast<const size_t*>(dm + 3 * meta_stride), s.count, dres,
            reinterpret_cast<cudec_stream_t>(st));
        if (launched != CUDEC_OK) {
            failure = launched;
            break;
        }
        if (hipMemcpyAsync(pres + s.begin, dres, s.count * sizeof(cudec_chunk_result),
                           hipMemcpyDeviceToHost, st) != hipSuccess ||
            (host_out && dof != 0 &&
             hipMemcpyAsync(s.p_dst.data(), dd, dof, hipMemcpyDeviceToHost, st) != hipSuccess) ||
            hipEventRecord(s.landed.get(), st) != hipSuccess) {
            failure = CUDEC_ERR_CUDA;
            break;
        }
        s.landed_pending = true;
    }
    /* unpack the waves still in flight, in order */
    for (size_t w = (waves > slots ? waves - slots : 0); w < waves && failure == CUDEC_OK; w++) {
        Slot& s = ctx.slot[w % slots];
        if (s.landed_pending && s.begin == w * wave) {
            s.landed_pending = false;
            if (hipEventSynchronize(s.landed.get()) != hipSuccess) {
                failure = CUDEC_ERR_CUDA;
            } else if (host_out) {
                failure = unpack_wave(s, pres, dst_ptrs, dst_caps, crew);
            }
        }
    }
    if (drain.now() != hipSuccess && failure == CUDEC_OK) {
        failure = CUDEC_ERR_CUDA;
    }
    for (size_t k = 0; k < used; k++) {
        ctx.slot[k].landed_pending = false;
    }
    if (hipGetLastError() != hipSuccess && failure == CUDEC_OK) {
        failure = CUDEC_ERR_CUDA;
    }
    std::memcpy(h_results, pres, res_bytes);
    if (failure == CUDEC_ERR_CUDA) {
        ctx.poisoned = true;
        return failure;
    }
    if (failure != CUDEC_OK) {
        return failure;
    }
    for (size_t i = 0; i < n; i++) {
        if (h_results[i].status != CUDEC_OK) {
            return static_cast<cudec_status>(h_results[i].status);
        }
    }
    return CUDEC_OK;
}

/* A context, or null: with all its streams, or, for a single call, without. */
cudec_stream_ctx* make_context(bool once) {
    const LastError taken;
    cudec_stream_ctx* ctx = new (std::nothrow) cudec_stream_ctx();
    if (ctx != nullptr &&
        (hipGetDevice(&ctx->device) != hipSuccess ||
         open_slots(*ctx, once ? 0 : kSlots) != hipSuccess)) {
        delete ctx;
        return nullptr;
    }
    if (ctx != nullptr) {
        ctx->once = once;
    }
    return ctx;
}

}  // namespace
}  // namespace cudec_amd

using namespace cudec_amd;

extern "C" {

cudec_status cudec_stream_ctx_create(cudec_stream_ctx** out_ctx) {
    if (out_ctx == nullptr) {
        return CUDEC_ERR_INVALID_ARGUMENT;
    }
    *out_ctx = make_context(false);
    return *out_ctx != nullptr ? CUDEC_OK : CUDEC_ERR_CUDA;
}

cudec_status cudec_lz4_decompress_stream_ctx(cudec_stream_ctx* ctx,
                                             const void* const* h_src_ptrs,
                                             const size_t* h_src_sizes, void* const* dst_ptrs,
                                             const size_t* dst_caps, size_t chunk_count,
                                             cudec_mem_space dst_space,
                                             cudec_chunk_result* h_results) {
    if (ctx == nullptr) {
        return CUDEC_ERR_INVALID_ARGUMENT;
    }
    const cudec_status args = validate_stream_args(h_src_ptrs, h_src_sizes, dst_ptrs, dst_caps,
                                                   chunk_count, dst_space, h_results);
    if (args != CUDEC_OK) {
        return args;
    }
    if (ctx->poisoned) {
        stamp(h_results, chunk_count, CUDEC_ERR_CUDA);
        return CUDEC_ERR_CUDA;
    }
    const LastError taken;
    try {
        return decode_stream(*ctx, h_src_ptrs, h_src_sizes, dst_ptrs, dst_caps, chunk_count,
                             dst_space, h_results);
    } catch (...) {
        ctx->poisoned = true;
        return CUDEC_ERR_CUDA;
    }
}

void cudec_stream_ctx_destroy(cudec_stream_ctx* ctx) {
    if (ctx == nullptr) {
        return;
    }
    for (Slot& s : ctx->slot) {
        if (s.stream) {
            (void)hipStreamSynchronize(s.stream.get());
        }
    }
    delete ctx;
}

cudec_status cudec_lz4_decompress_stream(const void* const* h_src_ptrs,
                                         const size_t* h_src_sizes, void* const* dst_ptrs,
                                         const size_t* dst_caps, size_t chunk_count,
                                         cudec_mem_space dst_space,
                                         cudec_chunk_result* h_results) {
    const cudec_status args = validate_stream_args(h_src_ptrs, h_src_sizes, dst_ptrs, dst_caps,
                                                   chunk_count, dst_space, h_results);
    if (args != CUDEC_OK) {
        return args;
    }
    cudec_stream_ctx* ctx = make_context(true);
    if (ctx == nullptr) {
        return CUDEC_ERR_CUDA;
    }
    const cudec_status st = cudec_lz4_decompress_stream_ctx(
        ctx, h_src_ptrs, h_src_sizes, dst_ptrs, dst_caps, chunk_count, dst_space, h_results);
    cudec_stream_ctx_destroy(ctx);
    return st;
}

}  // extern "C"
