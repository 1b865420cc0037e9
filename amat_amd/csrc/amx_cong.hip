// amx_cong.hip -- element kernels of congruent groups: K_e = s_e K_ref for
// every element (amx_op_set_element_matrices_scaled).
//
// One lane per element: rows of K_e u_e four at a time, K_ref streaming through
// the scalar cache (the same values for all 64 lanes) and every entry rebuilt
// as the stored layouts hold it -- fl(s_e K_ref[r][c]), rounded to FP32 / BF16
// for those storages -- with the products and sums of the whole layout in the
// same order, c ascending.  The element rows are therefore the stored kernels'
// bit for bit, from 8 bytes per element instead of its matrix.
//
// What bounds it: the FP64 units, three unfused operations per entry (two
// multiplications, one addition; FP32 / BF16: multiplication, conversion, FMA).
// hex20 64^3, FP64: element kernel 830 -> 108 us (26 of 39.3 Tops/s), matvec
// 881 -> 147 us; FP32 matvec 403 -> 116, BF16 326 -> 182 us; hex8 96^3 element
// kernel 59 -> 19 us, matvec FP64 77 -> 37, FP32 51 -> 29 us.  Where few waves
// run (hex20 15^3) the time is latency: FP32 element kernel 9.2 -> 5.5 us.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "amx_device.hpp"
#include "amx_internal.hpp"
#include "amx_kernels.hpp"

namespace amx {

namespace {

constexpr uint32_t kFlagBit = 0x80000000u;
constexpr uint32_t kIdxMask = 0x7fffffffu;
constexpr int kWaveN = 8;  // largest n that cong_wave takes
constexpr int kRows = 4;  // rows formed together: independent sums, one scalar load of 8 doubles per two columns

__device__ __forceinline__ double madd(double acc, double k, double u)
{
#pragma clang fp contract(off)
    const double p = k * u;
    return acc + p;
}
__device__ __forceinline__ float madd(float acc, float k, float u) { return __builtin_fmaf(k, u, acc); }

// the stored value of storage KT in the compute type (BF16: rounded by integer
// operations; the packed conversion instruction took twice their time, hex20
// 64^3 matvec 386 against 217 us)
template <typename KT, typename VT> __device__ __forceinline__ VT stored(double x)
{
    if constexpr (std::is_same<KT, double>::value) {
        return x;
    } else if constexpr (std::is_same<KT, float>::value) {
        return (VT)(float)x;
    } else {
        const uint32_t b = __float_as_uint((float)x);
        return (VT)__uint_as_float((b + (0x7fffu + ((b >> 16) & 1u))) & 0xffff0000u);
    }
}

// K_ref through the scalar unit: uniform loads from the constant address
// space, 16 values (4 columns of 4 rows) at a time
typedef double f64x8 __attribute__((ext_vector_type(8)));
typedef const f64x8 __attribute__((address_space(4))) * KrefPtr;
struct Chunk {
    f64x8 a, b;
    __device__ __forceinline__ void load(KrefPtr p)
    {
        a = p[0];
        b = p[1];
    }
    __device__ __forceinline__ double get(int i) const { return i < 8 ? a[i & 7] : b[i & 7]; }
};

// four columns of four rows
template <typename KT, typename VT>
__device__ __forceinline__ void use_chunk(const Chunk& k, double s, const VT (&u)[4], VT (&acc)[kRows])
{
#pragma unroll
    for (int c = 0; c < 4; c++) {
        VT kv[kRows];
#pragma unroll
        for (int i = 0; i < kRows; i++) kv[i] = stored<KT, VT>(s * k.get(c * kRows + i));
#pragma unroll
        for (int i = 0; i < kRows; i++) acc[i] = madd(acc[i], kv[i], u[c]);
    }
}

// the next chunk is asked for once the current one is there: scalar loads
// return in any order, so a wait is for all of them
__device__ __forceinline__ void next_chunk(const Chunk& cur, Chunk& next, KrefPtr p)
{
    asm volatile("" : : "s"(cur.a), "s"(cur.b));
    __builtin_amdgcn_sched_barrier(0);
    next.load(p);
    __builtin_amdgcn_sched_barrier(0);
}

// rows 4 rb0 .. 4 rb1 - 1 (this wave's) of the 64 elements from slot0 on, whose
// u_e the block holds in LDS, [column][lane].  The column loop is rolled: the
// straight-line form of it (u_e in 120 registers, 6 KB of code per row block)
// left 2-3 waves per SIMD and, where a wave forms one row block only, waited
// for its instructions (hex20 15^3, 4 rows per wave: 7.7 us).
template <int N, typename KT, typename VT, bool ATOMIC>
__device__ __forceinline__ void cong_rows(const CongArgs& a, uint32_t slot0, uint32_t rb0, uint32_t rb1,
                                          const VT* __restrict__ ush)
{
    constexpr int NCH = N / 4;  // chunks of a row block
    constexpr bool BF = std::is_same<KT, uint16_t>::value;
    if (rb0 >= rb1) return;
    const uint32_t end = a.slot_begin + a.n_slots, lane = threadIdx.x & 63u;
    const bool real = slot0 + lane < end;
    const uint32_t slot = real ? slot0 + lane : end - 1u;
    const uint64_t stride = a.stride;
    VT* __restrict__ out = static_cast<VT*>(a.out);
    const double s = a.scale[slot];
    KrefPtr kp = (KrefPtr)(uintptr_t)a.kref + (uint64_t)rb0 * (N / 2);
    const VT* ul = ush + lane;
    Chunk k0, k1;
    k0.load(kp);
    for (uint32_t rb = rb0; rb < rb1; rb++) {
        VT acc[kRows] = {VT(0), VT(0), VT(0), VT(0)};
        VT kd[kRows];
        if constexpr (BF) {
#pragma unroll
            for (int i = 0; i < kRows; i++) kd[i] = (VT)a.kdiag[(uint64_t)(rb * kRows + i) * stride + slot];
        }
        auto columns = [&](int j, VT (&u)[4]) {
#pragma unroll
            for (int c = 0; c < 4; c++) u[c] = ul[(4 * j + c) * 64];
        };
        VT u[4];
#pragma unroll 1
        for (int j = 0; j + 1 < NCH; j += 2) {
            columns(j, u);
            next_chunk(k0, k1, kp + 2);
            use_chunk<KT, VT>(k0, s, u, acc);
            columns(j + 1, u);
            next_chunk(k1, k0, kp + 4);  // the last row block's is the padding of cong_pack
            use_chunk<KT, VT>(k1, s, u, acc);
            kp += 4;
        }
        if constexpr (NCH & 1) {
            columns(NCH - 1, u);
            next_chunk(k0, k1, kp + 2);
            use_chunk<KT, VT>(k0, s, u, acc);
            k0 = k1;
            kp += 2;
        }
        // the sums are complete here (they are not to be moved, row by row,
        // into the conditional stores)
#pragma unroll
        for (int i = 0; i < kRows; i++) asm volatile("" : "+v"(acc[i]));
#pragma unroll
        for (int i = 0; i < kRows; i++) {
            const uint64_t at = (uint64_t)(rb * kRows + i) * stride + slot;
            // BF16: the FP32 diagonal last, as the stored form adds it
            if constexpr (BF) acc[i] = madd(acc[i], kd[i], ul[(rb * kRows + i) * 64]);
            if (real) {
                if constexpr (ATOMIC) unsafeAtomicAdd(&out[a.map[at] & kIdxMask], acc[i]);
                else out[a.ve_base + at] = acc[i];
            }
        }
    }
}

// small elements: a wave takes 64 elements whole, u_e in registers (staging it
// in LDS for two waves that share the rows: hex8 96^3 matvec 33.3 instead of
// 30.5 us in FP32)
template <int N, typename KT, typename VT, bool ATOMIC>
__device__ __forceinline__ void cong_wave(const CongArgs& a, uint32_t slot0)
{
    constexpr int NCH = N / 4, NRB = N / kRows;
    constexpr bool BF = std::is_same<KT, uint16_t>::value;
    const uint32_t end = a.slot_begin + a.n_slots, lane = threadIdx.x & 63u;
    if (slot0 >= end) return;
    const bool real = slot0 + lane < end;
    const uint32_t slot = real ? slot0 + lane : end - 1u;
    const uint64_t stride = a.stride;
    const VT* __restrict__ u = static_cast<const VT*>(a.u);
    VT* __restrict__ out = static_cast<VT*>(a.out);
    const uint32_t zero_on = a.masked ? kFlagBit : 0u;
    const double s = a.scale[slot];
    uint32_t m[N];
#pragma unroll
    for (int c = 0; c < N; c++) m[c] = a.map[c * stride + slot];
    VT ue[NCH][4], kd[N];
    if constexpr (BF)
#pragma unroll
        for (int c = 0; c < N; c++) kd[c] = (VT)a.kdiag[c * stride + slot];
#pragma unroll
    for (int c = 0; c < N; c++) {
        const VT x = u[m[c] & kIdxMask];
        ue[c / 4][c % 4] = (m[c] & zero_on) ? VT(0) : x;
    }
    KrefPtr kp = (KrefPtr)(uintptr_t)a.kref;
    Chunk k[2];
    k[0].load(kp);
    VT acc[NRB][kRows] = {};
#pragma unroll
    for (int j = 0; j < NRB * NCH; j++) {
        next_chunk(k[j & 1], k[(j + 1) & 1], kp + 2 * (j + 1));  // the last one is the padding of cong_pack
        use_chunk<KT, VT>(k[j & 1], s, ue[j % NCH], acc[j / NCH]);
    }
#pragma unroll
    for (int r = 0; r < N; r++) asm volatile("" : "+v"(acc[r / kRows][r % kRows]));
#pragma unroll
    for (int r = 0; r < N; r++) {
        VT v = acc[r / kRows][r % kRows];
        if constexpr (BF) v = madd(v, kd[r], ue[r / 4][r % 4]);
        if (real) {
            if constexpr (ATOMIC) unsafeAtomicAdd(&out[m[r] & kIdxMask], v);
            else out[a.ve_base + r * stride + slot] = v;
        }
    }
}

// a block's 4 waves: 64 elements, row blocks of part `part` of `parts`.  The
// waves gather a quarter of the columns each into LDS, then share the rows.
template <int N, typename KT, typename VT, bool ATOMIC>
__device__ __forceinline__ void cong_block(const CongArgs& a, uint32_t slot0, uint32_t part, uint32_t parts, VT* ush)
{
    constexpr uint32_t NRB = N / kRows, C = N / 4;
    static_assert(N % 4 == 0, "columns and rows in fours");
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    const uint32_t end = a.slot_begin + a.n_slots;
    const uint32_t slot = min(slot0 + lane, end - 1u);  // lanes past the end repeat the last slot
    const uint32_t* __restrict__ map = a.map + (uint64_t)(w * C) * a.stride;
    const VT* __restrict__ u = static_cast<const VT*>(a.u);
    const uint32_t zero_on = a.masked ? kFlagBit : 0u;
    const uint32_t b0 = NRB * part / parts, nb = NRB * (part + 1u) / parts - b0;
    const uint32_t rb0 = b0 + nb * w / 4u, rb1 = b0 + nb * (w + 1u) / 4u;
    // the first row block's K_ref is fetched into the scalar cache beside the
    // gathers; in a launch of few waves nothing else covers its latency
    typedef const uint32_t __attribute__((address_space(4))) * WordPtr;
    WordPtr line = (WordPtr)(uintptr_t)(a.kref + (uint64_t)rb0 * (N * kRows));
    uint32_t touch[N / 2];
#pragma unroll
    for (int i = 0; i < N / 2; i++) touch[i] = line[16 * i];
    uint32_t m[C];
#pragma unroll
    for (uint32_t c = 0; c < C; c++) m[c] = map[(uint64_t)c * a.stride + slot];
    VT x[C];
#pragma unroll
    for (uint32_t c = 0; c < C; c++) x[c] = u[m[c] & kIdxMask];
#pragma unroll
    for (uint32_t c = 0; c < C; c++) ush[(w * C + c) * 64u + lane] = (m[c] & zero_on) ? VT(0) : x[c];
    for (int i = 0; i < N / 2; i++) asm volatile("" : : "s"(touch[i]));
    __syncthreads();
    cong_rows<N, KT, VT, ATOMIC>(a, slot0, rb0, rb1, ush);
}

// block b of a group's launch
template <int N, typename KT, typename VT, bool ATOMIC>
__device__ __forceinline__ void cong_group(const CongArgs& a, uint32_t b, uint32_t parts)
{
    if constexpr (N <= kWaveN) {
        cong_wave<N, KT, VT, ATOMIC>(a, a.slot_begin + (b * 4u + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * 64u);
    } else {
        __shared__ VT ush[N * 64];
        const uint32_t eb = b / parts;
        cong_block<N, KT, VT, ATOMIC>(a, a.slot_begin + eb * 64u, b - eb * parts, parts, ush);
    }
}

template <int N, typename KT, typename VT, bool ATOMIC>
__global__ __launch_bounds__(256) void cong_kernel(CongArgs a, uint32_t parts)
{
    if (a.skip && *a.skip) return;  // converged solver: nothing to do
    const uint32_t b = __builtin_amdgcn_readfirstlane(xcd_block(blockIdx.x, gridDim.x));
    cong_group<N, KT, VT, ATOMIC>(a, b, parts);
}

// block -> block of the launch of entry job_of(prefix)
template <int N, typename KT, typename VT>
__global__ __launch_bounds__(256) void cong_batched_kernel(const CongJob* __restrict__ jobs,
                                                          const uint32_t* __restrict__ prefix, uint32_t n_jobs)
{
    const uint32_t w = __builtin_amdgcn_readfirstlane(xcd_block(blockIdx.x, gridDim.x));
    const uint32_t j = job_of(prefix, n_jobs, w);
    const CongArgs a = jobs[j].a;
    if (a.skip && *a.skip) return;
    cong_group<N, KT, VT, false>(a, w - prefix[j], jobs[j].parts);
}

template <int N, typename KT, typename VT> void launch_n(const CongArgs& a, bool atomic, hipStream_t s)
{
    const uint32_t parts = cong_parts(N, a.n_slots), nb = cong_blocks(N, a.n_slots, parts);
    if (atomic) cong_kernel<N, KT, VT, true><<<nb, 256, 0, s>>>(a, parts);
    else cong_kernel<N, KT, VT, false><<<nb, 256, 0, s>>>(a, parts);
}

template <typename KT, typename VT>
void launch_batched_k(uint32_t n, const CongJob* jobs, const uint32_t* prefix, uint32_t n_jobs, uint32_t total,
                      hipStream_t s)
{
    switch (n) {
    case 8: cong_batched_kernel<8, KT, VT><<<total, 256, 0, s>>>(jobs, prefix, n_jobs); break;
    case 20: cong_batched_kernel<20, KT, VT><<<total, 256, 0, s>>>(jobs, prefix, n_jobs); break;
    case 24: cong_batched_kernel<24, KT, VT><<<total, 256, 0, s>>>(jobs, prefix, n_jobs); break;
    case 60: cong_batched_kernel<60, KT, VT><<<total, 256, 0, s>>>(jobs, prefix, n_jobs); break;
    default: fail(AMX_INVALID_STATE, "no congruent kernel for n = " + std::to_string(n));
    }
}

template <typename KT, typename VT> void launch_k(const CongArgs& a, uint32_t n, bool atomic, hipStream_t s)
{
    switch (n) {
    case 8: return launch_n<8, KT, VT>(a, atomic, s);
    case 20: return launch_n<20, KT, VT>(a, atomic, s);
    case 24: return launch_n<24, KT, VT>(a, atomic, s);
    case 60: return launch_n<60, KT, VT>(a, atomic, s);
    default: fail(AMX_INVALID_STATE, "no congruent kernel for n = " + std::to_string(n));
    }
}

}  // namespace

bool cong_supported(uint32_t n) { return n == 8 || n == 20 || n == 24 || n == 60; }

uint32_t cong_parts(uint32_t n, uint64_t n_slots)
{
    // one block forms all rows of its 64 elements where that fills the chip (hex20
    // 64^3 FP64 element kernel: 1, 2, 4 parts 117, 119, 130 us); fewer elements
    // share the rows among blocks, each gathering u again, down to one row block
    // per wave (32^3: 29.0, 23.8, 23.8 us; 15^3: 18.0, 12.7, 9.8 us)
    if (n <= kWaveN) return 1;
    const uint32_t most = (n / kRows + 3u) / 4u;  // a row block per wave
    const uint64_t groups = std::max<uint64_t>(1, (n_slots + 63u) / 64u);
    return (uint32_t)std::min<uint64_t>(most, std::max<uint64_t>(1, 1024u / groups));
}

uint32_t cong_blocks(uint32_t n, uint32_t n_slots, uint32_t parts)
{
    return n <= kWaveN ? (n_slots + 255u) / 256u : (n_slots + 63u) / 64u * parts;
}

uint64_t cong_pack_values(uint32_t n) { return ((uint64_t)n * n + 16 + 7) / 8 * 8; }

std::vector<double> cong_pack(const std::vector<double>& kref, uint32_t n, bool zero_diag)
{
    std::vector<double> k(cong_pack_values(n), 0.0);  // the kernel loads one chunk past the end
    for (uint32_t r = 0; r < n; r++)
        for (uint32_t c = 0; c < n; c++)
            k[(size_t)(r / kRows) * n * kRows + c * kRows + r % kRows] =
                zero_diag && r == c ? 0.0 : kref[(size_t)r * n + c];
    return k;
}

void launch_cong(uint32_t n, KType kt, bool vt_double, bool atomic, const CongArgs& a, hipStream_t s)
{
    if (a.n_slots == 0) return;
    if (kt == KType::F64) {
        AMX_REQUIRE(vt_double, AMX_INVALID_ARGUMENT, "FP32 vectors need FP32 or BF16 element matrices");
        launch_k<double, double>(a, n, atomic, s);
    } else if (kt == KType::F32) {
        if (vt_double) launch_k<float, double>(a, n, atomic, s);
        else launch_k<float, float>(a, n, atomic, s);
    } else {
        if (vt_double) launch_k<uint16_t, double>(a, n, atomic, s);
        else launch_k<uint16_t, float>(a, n, atomic, s);
    }
    AMX_HIP(hipGetLastError());
}

void launch_cong_batched(uint32_t n, KType kt, bool vt_double, const CongJob* jobs, const uint32_t* prefix,
                         uint32_t n_jobs, uint32_t total_blocks, hipStream_t s)
{
    if (n_jobs == 0 || total_blocks == 0) return;
    AMX_REQUIRE(vt_double == (kt == KType::F64), AMX_INVALID_STATE, "batched jobs: FP64, or FP32 vectors");
    if (kt == KType::F64) launch_batched_k<double, double>(n, jobs, prefix, n_jobs, total_blocks, s);
    else if (kt == KType::F32) launch_batched_k<float, float>(n, jobs, prefix, n_jobs, total_blocks, s);
    else launch_batched_k<uint16_t, float>(n, jobs, prefix, n_jobs, total_blocks, s);
    AMX_HIP(hipGetLastError());
}

}  // namespace amx
