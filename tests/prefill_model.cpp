// The host side of the library (kv_api.cpp) over a model of the device: allocations are address ranges of a bounded
// memory, and each launch checks what its kernel would read and write -- every address inside a live allocation, every
// tile holding the rows that the attention expects of it, every output row written once.  Compiled by test_host_prefill.py.
#define HIP_INCLUDE_HIP_HIP_EXT_H
#include <hip/hip_runtime.h>
#undef __align__
#define __align__(n) __attribute__((aligned(n)))
#undef HIP_SYMBOL
#define HIP_SYMBOL(x) ((const void *) (x))
#include KV_API

#include <cstdio>
#include <map>

namespace {
size_t limit_ = 0, used_ = 0, next_ = 1 << 20; // bytes of the device, allocated, next address
int error_ = 0;                                // hipMalloc returns this, if set
bool capturing_ = false;                       // a stream is being captured: hipMalloc only in the relaxed mode
hipStreamCaptureMode mode_ = hipStreamCaptureModeGlobal;
std::map<size_t, size_t> live_;                // address -> bytes
std::string bad_;
int unread_ = 0; // tiles that no attention has read
int appends_ = 0, launches_ = 0, most_pieces_ = 0, most_layers_ = 0, least_heads_ = 4;

void fail(const char * what, long long a = 0, long long b = 0) {
    char t[200];
    snprintf(t, sizeof t, "%s %lld %lld; ", what, a, b);
    if (bad_.size() < 1000) bad_ += t;
}
// bytes [p, p + n) inside one live allocation
void inside(const void * p, size_t n, const char * what) {
    if (!n) return;
    auto it = live_.upper_bound((size_t) p);
    if (it == live_.begin()) return fail(what, (long long) (size_t) p, (long long) n);
    --it;
    if ((size_t) p + n > it->first + it->second) fail(what, (long long) ((size_t) p - it->first + n), (long long) it->second);
}
struct Tile {
    int layer, g, t, rows; // rows: positions 32 t .. 32 t + rows - 1 of the layer's head
    bool read = false;
};
std::map<size_t, Tile> tiles_;
std::map<std::pair<int, int>, int> ring_; // (layer, ring row) -> position
std::map<int, int> stored_;               // layer -> rows stored
std::map<long long, int> done_;           // output rows written
const float * out0_ = nullptr;
} // namespace

namespace qkv {
hipError_t launch_append(const StoreLayout & S, int, int layer0, int nl, int pos, int T, const void *, const void *, int, hipStream_t, hipEvent_t,
                         hipEvent_t, const float *, const float2 *) {
    appends_++;
    for (int l = layer0; l < layer0 + nl; l++) {
        if (pos > stored_[l]) fail("append leaves a gap", l, pos);
        stored_[l] = std::max(stored_[l], pos + T);
        for (int p = std::max(pos, pos + T - S.kvrc); S.kvrc && p < pos + T; p++) ring_[{l, p % S.kvrc}] = p;
    }
    return hipSuccess;
}
hipError_t launch_prefill_kv(const PrefillArgs & a, int kb, int vb, hipStream_t) {
    launches_++;
    for (int u = 0; u < a.nl * a.ng; u++) {
        const int l = a.layer + u / a.ng, g = a.g0 + u % a.ng;
        if (a.S.side[l][0].bits != kb || a.S.side[l][1].bits != vb) fail("formats of layer", l);
        for (int w = 0; w < 2; w++)
            for (int t = w ? a.q0 : a.p0; t < (w ? a.q1 : a.p1); t++) {
                const uint8_t * at = w ? a.kq16 + ((size_t) u * a.q_tiles + t % a.q_tiles) * KV16_TILE : a.kv16 + ((size_t) u * a.kv_tiles + t) * KV16_TILE;
                inside(at, KV16_TILE, "tile");
                const int rows = std::min(ATP, a.L - ATP * t);
                if (rows < 1 || ATP * t + rows > stored_[l]) fail("tile of rows that are not stored", t, stored_[l]);
                for (int p = ATP * t; w && p < ATP * t + rows; p++)
                    if (ring_[{l, p % a.S.kvrc}] != p) fail("window row replaced in the ring", l, p);
                Tile & x = tiles_[(size_t) at];
                if (x.rows && !x.read) unread_++;
                x = Tile{l, g, w ? -1 - t : t, rows};
            }
    }
    inside(a.q16, (size_t) a.nl * a.ng * a.q_blocks * Q16_BLOCK, "query operands");
    return hipSuccess;
}
hipError_t launch_prefill(PrefillArgs & a, hipStream_t) {
    launches_++;
    most_pieces_ = std::max(most_pieces_, a.np);
    most_layers_ = std::max(most_layers_, a.nl);
    least_heads_ = std::min(least_heads_, a.ng);
    size_t part = 0;
    for (int i = 0; i < a.np; i++) {
        const PrefillPiece & P = a.pc[i];
        for (int u = 0; u < a.nl * a.ng; u++) {
            const int l = a.layer + u / a.ng, g = a.g0 + u % a.ng, pmax = P.n0 + P.R / GQA - 1;
            for (int t = 0; ATP * t <= pmax; t++) {
                const bool w = ATP * t >= P.ws;
                const uint8_t * at = w ? a.kq16 + ((size_t) u * a.q_tiles + t % a.q_tiles) * KV16_TILE : a.kv16 + ((size_t) u * a.kv_tiles + t) * KV16_TILE;
                const auto x = tiles_.find((size_t) at);
                if (x != tiles_.end()) x->second.read = true;
                if (x == tiles_.end() || x->second.layer != l || x->second.g != g || x->second.t != (w ? -1 - t : t) ||
                    x->second.rows < std::min(ATP, pmax + 1 - ATP * t))
                    fail("tile read before it is written", l, t);
                if (t % 2 == 0) inside(at, 2 * KV16_TILE, "pair of tiles");
            }
            for (int tok = 0; tok < P.R / GQA; tok++) {
                const long long row = (a.out - out0_) / (NH * HD) + (long long) (u / a.ng) * a.T + P.t0 + tok;
                done_[row * NKV + g]++;
            }
        }
        if (P.nseg > 1) part += (size_t) P.R * a.nl * a.ng * P.nseg;
    }
    inside(a.part, part * HD * 4, "partials");
    inside(a.ml, part * sizeof(float2), "partial sums");
    const uint8_t * const q0 = a.q16, * const q1 = q0 + (size_t) a.nl * a.ng * a.q_blocks * Q16_BLOCK;
    if (q0 != q1 && part && q0 < (const uint8_t *) (a.part + part * HD) && q1 > (const uint8_t *) a.part) fail("query operands inside the partials");
    for (const auto & x : tiles_)
        if (q0 != q1 && (size_t) q1 > x.first && (size_t) q0 < x.first + KV16_TILE) fail("query operands inside the tiles");
    return hipSuccess;
}
hipError_t launch_ring_refill(const StoreLayout & S, int, int nl, int p0, int p1, hipStream_t) {
    for (int l = 0; l < nl; l++)
        for (int p = p0; p < p1; p++) ring_[{l, p % S.kvrc}] = p;
    return hipSuccess;
}
hipError_t launch_attn(const AttnArgs &, int, int, int, int, hipStream_t, hipEvent_t, hipEvent_t) { return hipSuccess; }
hipError_t launch_combine(const AttnArgs &, hipStream_t, hipEvent_t, hipEvent_t) { return hipSuccess; }
hipError_t launch_prefetch(const AttnArgs &, int, int, int, hipStream_t) { return hipSuccess; }
} // namespace qkv

extern "C" {
hipError_t hipMalloc(void ** p, size_t n) {
    if (error_) return (hipError_t) error_;
    if (capturing_ && mode_ != hipStreamCaptureModeRelaxed) return hipErrorStreamCaptureUnsupported;
    if (limit_ && used_ + n > limit_) return hipErrorOutOfMemory;
    used_ += n;
    live_[next_] = n;
    *p = (void *) next_;
    next_ += (n + 4095) / 4096 * 4096 + (1 << 20); // (a gap: overruns do not land in the next one)
    return hipSuccess;
}
hipError_t hipFree(void * p) {
    used_ -= live_[(size_t) p];
    live_.erase((size_t) p);
    return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode * m) { return std::swap(mode_, *m), hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *, unsigned) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *, hipEvent_t, hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipGetDevice(int * d) { return *d = 0, hipSuccess; }
const char * hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : e == hipErrorIllegalState ? "illegal state" : "error"; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void ** p, const void *) { return *p = nullptr, hipErrorInvalidValue; }
hipError_t hipMemcpy(void *, const void *, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipMemset(void *, int, size_t) { return hipSuccess; }

// room: bytes that may still be allocated (0: no bound); error: what hipMalloc returns instead (0: nothing)
void model_room(size_t room, int error) {
    limit_ = room ? used_ + room : 0;
    error_ = error;
}
// -> 1 if the thread's capture mode is the program's again
int model_capture(int on) {
    capturing_ = on;
    return mode_ == hipStreamCaptureModeGlobal;
}
size_t model_used(void) { return used_; }
int model_allocations(void) { return (int) live_.size(); }
void model_begin(const float * out) {
    out0_ = out;
    done_.clear();
    bad_.clear();
    tiles_.clear(); // (a call reads nothing that an earlier one unpacked)
    unread_ = 0;
    appends_ = launches_ = most_pieces_ = most_layers_ = 0;
    least_heads_ = 4;
}
// the faults of the call since model_begin, and that each of `rows` (layer, token, kv head) was attended once
const char * model_faults(long long rows) {
    if ((long long) done_.size() != rows) fail("rows attended", (long long) done_.size(), rows);
    for (const auto & x : done_)
        if (x.second != 1) fail("row attended more than once", x.first, x.second);
    return bad_.c_str();
}
// appends, launches, most pieces and layers and fewest kv heads of a launch
void model_counts(int * c) {
    const int v[5] = {appends_, launches_, most_pieces_, most_layers_, least_heads_};
    for (int i = 0; i < 5; i++) c[i] = v[i];
}
// tiles unpacked for nothing
int model_unread(void) {
    int n = unread_;
    for (const auto & x : tiles_) n += !x.second.read;
    return n;
}
int model_stored(void * h, int seq) { return static_cast<Store *>(h)->n[seq]; }
}
