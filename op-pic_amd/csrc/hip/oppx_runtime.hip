// Device runtime of the oppx C-ABI: initialisation, errors, memory, AoS<->SoA transposes.
// Replaces opp_lib/src/hip/opp_hip.cpp:221-271 (device init) and the host-side layout
// conversions of opp_lib/src/hip/opp_hip_utils.cpp:35-153, which here run on the device.

#include <cstring>
#include <type_traits>

#include "oppx_internal.h"

namespace oppx {

static thread_local std::string g_last_error;

oppx_tuning g_tuning = {256, 16, 0, 0, 16, 64, 256, 1};

unsigned resident_blocks(const void* kernel, int block) {
    static int cus = 0;
    static const void* kern_cache[128] = {nullptr};
    static int block_cache[128] = {0}, per_cu_cache[128] = {0};
    if (cus == 0) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
            cus = 256;
    }
    int per_cu = 0;
    for (int i = 0; i < 128; i++) {
        if (kern_cache[i] == kernel && block_cache[i] == block) { per_cu = per_cu_cache[i]; break; }
        if (kern_cache[i] == nullptr) {
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, block, 0) != hipSuccess || per_cu <= 0)
                per_cu = 1;
            kern_cache[i] = kernel;
            block_cache[i] = block;
            per_cu_cache[i] = per_cu;
            break;
        }
    }
    return (unsigned)cus * (unsigned)(per_cu > 0 ? per_cu : 1);
}

void set_error(const std::string& msg) { g_last_error = msg; }

namespace {

// One thread per (element, component); reads/writes coalesced on the SoA side and
// contiguous on the AoS side.
template <typename T>
__global__ void aos_to_soa_kernel(const T* __restrict__ aos, T* __restrict__ soa, int64_t n, int dim,
                                  int64_t stride) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n * dim) return;
    const int64_t i = t / dim, d = t % dim;
    soa[d * stride + i] = aos[t];
}

template <typename T>
__global__ void soa_to_aos_kernel(const T* __restrict__ soa, T* __restrict__ aos, int64_t n, int dim,
                                  int64_t stride) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n * dim) return;
    const int64_t i = t / dim, d = t % dim;
    aos[t] = soa[d * stride + i];
}

struct Pattern {
    unsigned char b[256];
};

// element i, component d = pattern[d]; AoS when stride == 0, else SoA with the given stride
template <typename T>
__global__ void fill_pattern_kernel(T* __restrict__ dst, int64_t n, int dim, int64_t stride, Pattern pat) {
    // one record per thread and step, its components in an inner loop: no 64-bit division per element
    const T* pv = reinterpret_cast<const T*>(pat.b);
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        if (stride == 0) {
            for (int d = 0; d < dim; d++) dst[i * dim + d] = pv[d];  // AoS: record i is dim consecutive values
        } else {
            for (int d = 0; d < dim; d++) dst[d * stride + i] = pv[d];  // SoA: component d at d * stride + i
        }
    }
}

// entries [first, first + count) of every `rec`-int record: v -> v + offset unless v < 0 or v == MAX
__global__ void offset_indices_kernel(int32_t* __restrict__ base, int64_t n, int rec, int first, int count,
                                      int32_t offset) {
    // one record per thread and step (no 64-bit division per entry)
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        int32_t* p = base + i * rec + first;
        for (int k = 0; k < count; k++) {
            const int32_t v = p[k];
            if (v >= 0 && v != kMaxCell) p[k] = v + offset;
        }
    }
}

// ---- many copies and fills in one launch ----
// Small copies are bound by their launches (2 us each on the device, 8 to 10 us apart from a Python caller), large ones
// by HBM. Admitting a request took 21 copies, fills and rebasing passes, handing it back 11, a clone 9; each is one
// launch now: five requests admitted 560 -> 200 us and handed back 900 -> 660 us (of which 20 MB over the host link at
// 54 GB/s take 350), a clone of 3,000 particles 89 -> 39 us, one of 24 M 807 -> 746. 1.92 GB in 10 rows: 671 us with
// 2 units in flight a thread, 697 with 4, 722 with 8 (the runtime's own copy 775).
constexpr int kSegs = 32;      // row segments a launch takes (their table is a kernel argument)
constexpr int kSegBlock = 256;
constexpr int kSegUnits = 2;   // units a thread has in flight
constexpr int64_t kMaxChunks = 1 << 30;  // of a launch (a 32-bit index)
constexpr int64_t kMaxGrid = 1 << 22;    // its workgroups, which stride over the chunks: a grid of 2^32 threads is refused

// One contiguous piece of memory: `units` units of 1 << shift bytes and the words behind them.
struct CopySeg {
    unsigned char* dst;
    const unsigned char* src;  // nullptr: the two words of `fill` over and over
    int64_t units;
    uint32_t fill[2];
    uint32_t chunk0;           // its first chunk
    int32_t add;
    uint8_t shift, tail, mask, first, count;
};

struct CopyTable {
    CopySeg s[kSegs];
    int n;
};

template <int W>
struct Words {
    uint32_t w[W];
};

// The words of one unit that hold indices, moved by S.add; w0 is the unit's first word in the segment.
template <int W>
__device__ __forceinline__ void rebase(Words<W>& v, int64_t w0, const CopySeg& S) {
#pragma unroll
    for (int k = 0; k < W; k++) {
        const unsigned m = (unsigned)(w0 + k) & S.mask;
        const int x = (int)v.w[k];
        if (m - S.first < S.count && x >= 0 && x != kMaxCell) v.w[k] = (uint32_t)(x + S.add);
    }
}

template <int W>
__device__ __forceinline__ void copy_units(const CopySeg& S, int64_t first_unit) {
    using V = std::conditional_t<W == 4, uint4, std::conditional_t<W == 2, uint2, uint32_t>>;
    int64_t u[kSegUnits];
    Words<W> v[kSegUnits];
#pragma unroll
    for (int j = 0; j < kSegUnits; j++) {
        u[j] = first_unit + j * kSegBlock + threadIdx.x;
        if (u[j] < S.units && S.src) v[j] = __builtin_bit_cast(Words<W>, reinterpret_cast<const V*>(S.src)[u[j]]);
    }
#pragma unroll
    for (int j = 0; j < kSegUnits; j++) {
        if (u[j] >= S.units) continue;
        if (!S.src) {
#pragma unroll
            for (int k = 0; k < W; k++) v[j].w[k] = S.fill[(W == 1 ? u[j] : k) & 1];
        } else if (S.add) {
            rebase<W>(v[j], u[j] * W, S);
        }
        reinterpret_cast<V*>(S.dst)[u[j]] = __builtin_bit_cast(V, v[j]);
    }
}

// Each block takes kSegBlock * kSegUnits consecutive units of one segment at a time.
__global__ void __launch_bounds__(kSegBlock) copy_segs_kernel(CopyTable T, uint32_t chunks) {
    for (uint32_t b = blockIdx.x; b < chunks; b += gridDim.x) {
        int at = 0;
        for (int step = kSegs / 2; step; step >>= 1)
            if (at + step < T.n && T.s[at + step].chunk0 <= b) at += step;
        const CopySeg& S = T.s[at];
        const int64_t first_unit = (int64_t)(b - S.chunk0) * (kSegBlock * kSegUnits);
        if (S.shift == 4) copy_units<4>(S, first_unit);
        else if (S.shift == 3) copy_units<2>(S, first_unit);
        else copy_units<1>(S, first_unit);
        if (first_unit == 0 && threadIdx.x < S.tail) {  // the words that fill no unit
            const int64_t w = (S.units << (S.shift - 2)) + threadIdx.x;
            Words<1> v{{S.fill[w & 1]}};
            if (S.src) {
                v.w[0] = reinterpret_cast<const uint32_t*>(S.src)[w];
                if (S.add) rebase<1>(v, w, S);
            }
            reinterpret_cast<uint32_t*>(S.dst)[w] = v.w[0];
        }
    }
}

}  // namespace
}  // namespace oppx

using namespace oppx;

extern "C" {

const char* oppx_last_error(void) { return g_last_error.c_str(); }

int oppx_init(int device) {
    int count = 0;
    OPPX_HIP_TRY(hipGetDeviceCount(&count));
    OPPX_ARG_CHECK(count > 0, "oppx_init: no HIP device visible");
    OPPX_ARG_CHECK(device >= 0 && device < count, "oppx_init: device index out of range");
    OPPX_HIP_TRY(hipSetDevice(device));
    return noalloc_scratch(device, nullptr);
}

int oppx_device_malloc(void** ptr, size_t bytes) {
    OPPX_ARG_CHECK(ptr != nullptr, "oppx_device_malloc: null out pointer");
    *ptr = nullptr;
    if (bytes == 0) return OPPX_OK;
    hipError_t e = hipMalloc(ptr, bytes);
    if (e != hipSuccess) {
        set_error(std::string("hipMalloc(") + std::to_string(bytes) + "): " + hipGetErrorString(e));
        *ptr = nullptr;
        return OPPX_ERR_NOMEM;
    }
    return OPPX_OK;
}

int oppx_device_free(void* ptr) {
    if (ptr) OPPX_HIP_TRY(hipFree(ptr));
    return OPPX_OK;
}

int oppx_memcpy_htod(void* dst, const void* src, size_t bytes, void* stream) {
    if (bytes == 0) return OPPX_OK;
    OPPX_ARG_CHECK(dst && src, "oppx_memcpy_htod: null pointer");
    OPPX_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, as_stream(stream)));
    OPPX_HIP_TRY(hipStreamSynchronize(as_stream(stream)));
    return OPPX_OK;
}

int oppx_memcpy_dtoh(void* dst, const void* src, size_t bytes, void* stream) {
    if (bytes == 0) return OPPX_OK;
    OPPX_ARG_CHECK(dst && src, "oppx_memcpy_dtoh: null pointer");
    OPPX_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, as_stream(stream)));
    OPPX_HIP_TRY(hipStreamSynchronize(as_stream(stream)));
    return OPPX_OK;
}

int oppx_memcpy_dtod(void* dst, const void* src, size_t bytes, void* stream) {
    if (bytes == 0) return OPPX_OK;
    OPPX_ARG_CHECK(dst && src, "oppx_memcpy_dtod: null pointer");
    OPPX_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, as_stream(stream)));
    return OPPX_OK;
}

int oppx_memset_zero(void* dst, size_t bytes, void* stream) {
    if (bytes == 0) return OPPX_OK;
    OPPX_ARG_CHECK(dst, "oppx_memset_zero: null pointer");
    OPPX_HIP_TRY(hipMemsetAsync(dst, 0, bytes, as_stream(stream)));
    return OPPX_OK;
}

int oppx_stream_sync(void* stream) {
    OPPX_HIP_TRY(hipStreamSynchronize(as_stream(stream)));
    return OPPX_OK;
}

int oppx_aos_to_soa(const void* aos, void* soa, int64_t n, int dim, int64_t stride, int elem_bytes, void* stream) {
    OPPX_ARG_CHECK(n >= 0 && dim > 0 && stride >= n, "oppx_aos_to_soa: bad sizes");
    OPPX_ARG_CHECK(elem_bytes == 4 || elem_bytes == 8, "oppx_aos_to_soa: elem_bytes must be 4 or 8");
    if (n == 0) return OPPX_OK;
    OPPX_ARG_CHECK(aos && soa, "oppx_aos_to_soa: null pointer");
    const unsigned g = grid_for(n * dim, 256);
    if (elem_bytes == 8)
        aos_to_soa_kernel<double><<<g, 256, 0, as_stream(stream)>>>((const double*)aos, (double*)soa, n, dim, stride);
    else
        aos_to_soa_kernel<int32_t><<<g, 256, 0, as_stream(stream)>>>((const int32_t*)aos, (int32_t*)soa, n, dim, stride);
    OPPX_LAUNCH_CHECK("aos_to_soa");
    return OPPX_OK;
}

int oppx_soa_to_aos(const void* soa, void* aos, int64_t n, int dim, int64_t stride, int elem_bytes, void* stream) {
    OPPX_ARG_CHECK(n >= 0 && dim > 0 && stride >= n, "oppx_soa_to_aos: bad sizes");
    OPPX_ARG_CHECK(elem_bytes == 4 || elem_bytes == 8, "oppx_soa_to_aos: elem_bytes must be 4 or 8");
    if (n == 0) return OPPX_OK;
    OPPX_ARG_CHECK(aos && soa, "oppx_soa_to_aos: null pointer");
    const unsigned g = grid_for(n * dim, 256);
    if (elem_bytes == 8)
        soa_to_aos_kernel<double><<<g, 256, 0, as_stream(stream)>>>((const double*)soa, (double*)aos, n, dim, stride);
    else
        soa_to_aos_kernel<int32_t><<<g, 256, 0, as_stream(stream)>>>((const int32_t*)soa, (int32_t*)aos, n, dim, stride);
    OPPX_LAUNCH_CHECK("soa_to_aos");
    return OPPX_OK;
}

int oppx_fill_pattern(void* dst, int64_t n, int dim, int elem_bytes, const void* pattern, int64_t stride, void* stream) {
    OPPX_ARG_CHECK(n >= 0 && dim > 0 && (elem_bytes == 4 || elem_bytes == 8), "oppx_fill_pattern: bad sizes");
    OPPX_ARG_CHECK((int64_t)dim * elem_bytes <= 256, "oppx_fill_pattern: pattern above 256 bytes");
    OPPX_ARG_CHECK(stride == 0 || stride >= n, "oppx_fill_pattern: stride below n");
    if (n == 0) return OPPX_OK;
    OPPX_ARG_CHECK(dst && pattern, "oppx_fill_pattern: null pointer");
    Pattern p{};
    memcpy(p.b, pattern, (size_t)dim * elem_bytes);
    int64_t g = grid_for(n, 256);
    if (g > 8192) g = 8192;
    if (elem_bytes == 8)
        fill_pattern_kernel<double><<<(unsigned)g, 256, 0, as_stream(stream)>>>((double*)dst, n, dim, stride, p);
    else
        fill_pattern_kernel<int32_t><<<(unsigned)g, 256, 0, as_stream(stream)>>>((int32_t*)dst, n, dim, stride, p);
    OPPX_LAUNCH_CHECK("fill_pattern");
    return OPPX_OK;
}

int oppx_offset_indices(int32_t* base, int64_t n_records, int rec_ints, int first, int count, int32_t offset,
                        void* stream) {
    OPPX_ARG_CHECK(n_records >= 0 && rec_ints > 0 && first >= 0 && count > 0 && first + count <= rec_ints,
                   "oppx_offset_indices: bad record layout");
    if (n_records == 0 || offset == 0) return OPPX_OK;
    OPPX_ARG_CHECK(base != nullptr, "oppx_offset_indices: null pointer");
    int64_t g = grid_for(n_records, 256);
    if (g > 8192) g = 8192;
    offset_indices_kernel<<<(unsigned)g, 256, 0, as_stream(stream)>>>(base, n_records, rec_ints, first, count, offset);
    OPPX_LAUNCH_CHECK("offset_indices");
    return OPPX_OK;
}

int oppx_copy_batch(int n, const oppx_copy_job* jobs, int max_blocks, void* stream) {
    OPPX_ARG_CHECK(n >= 0 && max_blocks >= 0 && (n == 0 || jobs), "oppx_copy_batch: bad job list");
    for (int j = 0; j < n; j++) {
        const oppx_copy_job& J = jobs[j];
        OPPX_ARG_CHECK(J.bytes >= 0 && J.rows >= 0, "oppx_copy_batch: negative size");
        if (J.bytes == 0 || J.rows == 0) continue;
        const uintptr_t all = (uintptr_t)J.dst | (uintptr_t)J.src | (uintptr_t)J.bytes |
                              (J.rows > 1 ? (uintptr_t)J.dst_stride | (uintptr_t)J.src_stride : 0);
        OPPX_ARG_CHECK(J.dst && all % 4 == 0, "oppx_copy_batch: null destination, or not whole 4-byte words");
        OPPX_ARG_CHECK(J.rows == 1 || (J.dst_stride >= J.bytes && (!J.src || J.src_stride >= J.bytes)),
                       "oppx_copy_batch: row stride below the row");
        OPPX_ARG_CHECK(J.add == 0 || (J.rec_ints >= 1 && J.rec_ints <= 128 && (J.rec_ints & (J.rec_ints - 1)) == 0 &&
                                      J.first >= 0 && J.count >= 1 && J.first + J.count <= J.rec_ints),
                       "oppx_copy_batch: bad record layout");
    }
    CopyTable T;
    T.n = 0;
    int64_t chunks = 0;
    const auto launch = [&]() -> int {
        if (T.n == 0) return OPPX_OK;
        int64_t g = chunks < kMaxGrid ? chunks : kMaxGrid;
        if (max_blocks && max_blocks < g) g = max_blocks;
        copy_segs_kernel<<<(unsigned)g, kSegBlock, 0, as_stream(stream)>>>(T, (uint32_t)chunks);
        OPPX_LAUNCH_CHECK("copy_batch");
        T.n = 0;
        chunks = 0;
        return OPPX_OK;
    };
    for (int j = 0; j < n; j++) {
        const oppx_copy_job& J = jobs[j];
        if (J.bytes == 0) continue;
        for (int64_t r = 0; r < J.rows; r++) {
            CopySeg S;
            S.dst = (unsigned char*)J.dst + r * J.dst_stride;
            S.src = J.src ? (const unsigned char*)J.src + r * J.src_stride : nullptr;
            // the widest unit both ends are aligned to: a wave then moves 1 KiB per instruction, not 256 B
            const uintptr_t a = (uintptr_t)S.dst | (uintptr_t)S.src;
            S.shift = a % 16 == 0 ? 4 : (a % 8 == 0 ? 3 : 2);
            S.units = J.bytes >> S.shift;
            S.tail = (uint8_t)((J.bytes - (S.units << S.shift)) / 4);
            memcpy(S.fill, &J.fill, 8);
            S.add = J.add;
            S.mask = (uint8_t)(J.add ? J.rec_ints - 1 : 0);
            S.first = (uint8_t)J.first;
            S.count = (uint8_t)J.count;
            int64_t need = (S.units + kSegBlock * kSegUnits - 1) / (kSegBlock * kSegUnits);
            if (need == 0) need = 1;
            if (T.n == kSegs || chunks + need > kMaxChunks) {
                const int rc = launch();
                if (rc != OPPX_OK) return rc;
            }
            OPPX_ARG_CHECK(need <= kMaxChunks, "oppx_copy_batch: row too long");
            S.chunk0 = (uint32_t)chunks;
            T.s[T.n++] = S;
            chunks += need;
        }
    }
    return launch();
}

}  // extern "C"
