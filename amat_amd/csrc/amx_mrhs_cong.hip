// amx_mrhs_cong.hip -- multi-RHS products of congruent groups of 60 DoFs
// (K_e = s_e K_ref): V = sum_e P_e^T s_e K_ref P_e U on MFMA.
//
// A wave takes 16 columns of U through a cluster of up to 8 neighbouring
// elements.  K_ref stays in its registers, so no matrix is read (FP32: the
// factor multiplies the product; BF16: the wave forms the rounded s_e K_ref);
// the element rows are summed in the wave's LDS rows and leave once per cluster
// (0.49 of the element rows on a structured mesh).
//   FP32: v_mfma_f32_16x16x4_f32, 60 = 15 steps of 4;
//   BF16: v_mfma_f32_16x16x32_bf16, two steps, columns 60..63 zero;
//   A lane l: row 16 m + l % 16, columns 4 ks + l/16 of mrhs_order (BF16 32 ks + 8 (l/16) + v);
//   C lane l, register i: row 16 m + 4 (l/16) + i, column l % 16.
// Rows 60..63 (tile m = 3) go to a dump row.
//
// What bounds it: FP32 the matrix cores -- 219 us of MFMA at 32768 elements x
// 128 columns, at two waves per SIMD (VGPRs) that the loads, the sums in LDS and
// the rows' way out only partly hide under it; BF16 forming the matrices (three
// instructions per value and its rounding) and the rows.  Against a kernel that
// reads the stored matrices and writes every element row (both passes of the
// scatter, one hex8 mesh beside it):
//   32^3, 128 columns, FP32   790 -> 607 us (of it 538 -> 454 and 254 -> 132)
//   31^3,  24 columns, BF16   atomics 258 -> 150 us, two passes 172 -> 150 us
//   28^3, 128 columns, BF16   atomics 559 -> 372 us
//   24^3,  64 columns, FP32   atomics 208 -> 134 us
//   31^3,   1 column,  FP32   two passes 127 -> 60 us, atomics 126 -> 59 us
//   16^3,  50 columns, FP32    58 ->  57 us
//   14^3, 128 columns, FP32    73 ->  62 us
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cfloat>
#include <cmath>
#include <cstring>
#include <new>
#include <type_traits>

#include "amx_device.hpp"
#include "amx_mrhs.hpp"

namespace amx {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int N = 60, COLS = 16;

// where the wave is: item (cluster, column group), element of the order, the
// cluster's rows of ve and its final rows
struct Cursor {
    uint32_t item, e, end, col0, ve0, n_ve, dir0, n_dir;
    __device__ __forceinline__ void open(const MrhsCongArgs& a, uint32_t ngroups)
    {
        // through the scalar cache: nothing that a kernel writes
        typedef const u32x4 __attribute__((address_space(4))) C;
        const uint32_t c = __builtin_amdgcn_readfirstlane(item / ngroups);
        const u32x4 t = reinterpret_cast<C*>(reinterpret_cast<uintptr_t>(a.clusters))[c];
        const u32x4 u = reinterpret_cast<C*>(reinterpret_cast<uintptr_t>(a.clusters))[c + 1];
        col0 = (item - c * ngroups) * COLS;
        e = t[0], end = u[0];
        ve0 = t[1], n_ve = u[1] - t[1];
        dir0 = t[2], n_dir = u[2] - t[2];
    }
    // past the last item: stays on its last element
    __device__ __forceinline__ void advance(const MrhsCongArgs& a, uint32_t ngroups, uint32_t hi, uint32_t step)
    {
        if (e + 1 < end) {
            e++;
        } else if (item + step < hi) {
            item += step;
            open(a, ngroups);
        }
    }
};

// row r, column c; WIDE: 4 GB and more (byte offsets past 32 bits)
template <bool WIDE, typename T> __device__ __forceinline__ T* at(T* p, uint32_t r, uint32_t nrhs, uint32_t c)
{
    if constexpr (WIDE) return p + ((uint64_t)r * nrhs + c);
    typedef typename std::conditional<std::is_const<T>::value, const char, char>::type B;
    return reinterpret_cast<T*>(reinterpret_cast<B*>(p) + (__umul24(r, 4u * nrhs) + 4u * c));
}

template <bool BF16, bool WIDE> struct Rhs {
    static constexpr int NB = BF16 ? 16 : 15;
    float b[NB];
    __device__ __forceinline__ void load(const MrhsCongArgs& a, int i, uint32_t d, uint32_t col)
    {
        b[i] = *at<WIDE>(a.U, d, a.nrhs, col);
    }
};

__device__ __forceinline__ void load_dofs(const MrhsCongArgs& a, uint32_t e, uint32_t q, uint32_t (&d)[16])
{
    const u32x4* p = reinterpret_cast<const u32x4*>(a.dofs + (uint64_t)e * 64 + q * 16);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const u32x4 v = p[j];
#pragma unroll
        for (int i = 0; i < 4; i++) d[4 * j + i] = v[i];
    }
}

__device__ __forceinline__ void load_slots(const MrhsCongArgs& a, uint32_t e, uint32_t q, u32x4 (&s)[2])
{
    const u32x4* p = reinterpret_cast<const u32x4*>(a.slots + (uint64_t)e * 64 + q * 16);
    s[0] = p[0];
    s[1] = p[1];
}

// two values rounded to BF16 (nearest even; in integers, half the cost of the
// conversion instructions; no NaN, whose largest payloads would carry into zero)
__device__ __forceinline__ uint32_t bf16_pair(float lo, float hi)
{
    const uint32_t a = __float_as_uint(lo), b = __float_as_uint(hi);
    return __builtin_amdgcn_perm(b + 0x7fffu + ((b >> 16) & 1u), a + 0x7fffu + ((a >> 16) & 1u), 0x07060302u);
}

// K_ref is held times a power of two, 2^-k, that brings its largest entry into
// [1, 2), and the factors times 2^k (mrhs_exponent): both then fit FP32 wherever
// their products do.
template <bool BF16> struct Ref;
// FP32: K_ref to 32 bits -- 24 in FP32, the 8 below them in BF16, whose product
// with the leading bits of U takes 8 MFMAs beside 60 -- and the factor 2^k m to
// 48: U times 2^k is exact, m (high and low part) multiplies the product.  The
// operands then carry less error than a stored matrix, whose entries s_e K_ref are
// rounded to FP32.  It costs 3 to 8 % (32^3, 128 columns 558 -> 573 us); K_ref
// and factor in FP32 alone, the same error in every element, had twice the operand
// error of a stored matrix.  High parts are cut towards zero and low parts never
// zero beside them: the products of an infinite U have one sign.
template <> struct Ref<false> {
    float k[4][15];
    u32x4 low[4][2];  // lane's columns 4 (8 t + v) + l/16, v = 0..7 (the order of B.b)
    __device__ __forceinline__ void load(const void* K)
    {
        const f32x4* p = static_cast<const f32x4*>(K) + threadIdx.x;
#pragma unroll
        for (int i = 0; i < 15; i++) {
            const f32x4 v = p[64 * i];
#pragma unroll
            for (int j = 0; j < 4; j++) k[(4 * i + j) / 15][(4 * i + j) % 15] = v[j];
        }
#pragma unroll
        for (int i = 0; i < 8; i++) low[i / 2][i % 2] = __builtin_bit_cast(u32x4, p[64 * (15 + i)]);
    }
    // side(i), i < 15: what is issued in the shadow of four MFMAs.  Two sums of
    // 8 and 7 steps: one sum of 15 had more error than the stored matrices' sums.
    template <typename R, typename F> __device__ __forceinline__ void multiply(f32x2 s, R& B, f32x4 (&acc)[4], F&& side) const
    {
        const float pow2 = __uint_as_float(__float_as_uint(s[0]) & 0x7f800000u);
#pragma unroll
        for (int ks = 0; ks < 15; ks++) B.b[ks] *= pow2;
        f32x4 more[4];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            u32x4 b;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int ks = 8 * t + 2 * j;
                b[j] = __builtin_amdgcn_perm(ks + 1 < 15 ? __float_as_uint(B.b[ks + 1 < 15 ? ks + 1 : 0]) : 0u,
                                             __float_as_uint(B.b[ks]), 0x07060302u);
            }
#pragma unroll
            for (int m = 0; m < 4; m++)
                more[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, low[m][t]),
                                                                  __builtin_bit_cast(bf16x8, b),
                                                                  t ? more[m] : f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
        }
#pragma unroll
        for (int ks = 0; ks < 15; ks++) {
#pragma unroll
            for (int m = 0; m < 4; m++)
                (ks < 8 ? acc : more)[m] =
                    __builtin_amdgcn_mfma_f32_16x16x4f32(k[m][ks], B.b[ks], (ks < 8 ? acc : more)[m], 0, 0, 0);
            side(ks);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int m = 0; m < 4; m++) acc[m] += more[m];
    }
    // the element's value of a row whose product is x
    static __device__ __forceinline__ float row(f32x2 s, float x)
    {
        const float m = __uint_as_float((__float_as_uint(s[0]) & 0x807fffffu) | 0x3f800000u);
        return fmaf(x, m, x * s[1]);
    }
};
// BF16: the stored matrices are s_e K_ref rounded to FP32, then to BF16.  Factor
// and K_ref are split in two FP32 values each: h S + (h s + l S) is their product
// to 48 bits and rounds once, in three instructions (an FP64 product and its
// conversion take 59 cycles per value, 420 us at 32768 elements x 128 columns).
template <> struct Ref<true> {
    float h[4][2][8], l[4][2][8];
    __device__ __forceinline__ void load(const void* K)
    {
        const f32x4* p = static_cast<const f32x4*>(K) + threadIdx.x;
#pragma unroll
        for (int i = 0; i < 32; i++) {
            const f32x4 v = p[64 * i];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                h[i / 8][i / 4 % 2][2 * (i % 4) + j] = v[2 * j];
                l[i / 8][i / 4 % 2][2 * (i % 4) + j] = v[2 * j + 1];
            }
        }
    }
    template <typename R, typename F> __device__ __forceinline__ void multiply(f32x2 s, R& B, f32x4 (&acc)[4], F&& side) const
    {
#pragma unroll
        for (int i = 0; i < 6; i++) side(i);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            u32x4 b;
#pragma unroll
            for (int j = 0; j < 4; j++)
                b[j] = __builtin_bit_cast(uint32_t, bf16x2{(__bf16)B.b[8 * ks + 2 * j], (__bf16)B.b[8 * ks + 2 * j + 1]});
#pragma unroll
            for (int m = 0; m < 4; m++) {
                float x[8];
#pragma unroll
                for (int j = 0; j < 8; j++) x[j] = fmaf(h[m][ks][j], s[0], fmaf(h[m][ks][j], s[1], l[m][ks][j] * s[0]));
                const u32x4 w = {bf16_pair(x[0], x[1]), bf16_pair(x[2], x[3]), bf16_pair(x[4], x[5]), bf16_pair(x[6], x[7])};
                acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w),
                                                                 __builtin_bit_cast(bf16x8, b), acc[m], 0, 0, 0);
            }
        }
#pragma unroll
        for (int i = 6; i < 15; i++) side(i);
    }
    static __device__ __forceinline__ float row(f32x2, float x) { return x; }
};

// n rows of LDS from row l0 on -> rows row(i) of out, and back to zero.  VW
// columns per lane (cols, and rows aligned to them), 1 << sh lanes per row; row
// counts are multiples of 16.
template <int VW, bool ATOMIC, bool WIDE, typename F>
__device__ __forceinline__ void put_rows(float* W, uint32_t n, float* out, uint32_t ld, uint32_t cols, uint32_t col0, F&& row)
{
    typedef float V __attribute__((ext_vector_type(VW)));
    uint32_t sh = VW == 4 ? 2 : 4;
    while (sh && (1u << (sh - 1)) * VW >= cols) sh--;
    const uint32_t r = threadIdx.x >> sh, c = VW * (threadIdx.x & ((1u << sh) - 1u)), per = 64u >> sh;
    const bool in = col0 + c < cols;
    for (uint32_t b = 0; b < n; b += 4u * per) {
        V v[4];
        uint32_t to[4];
#pragma unroll
        for (uint32_t j = 0; j < 4; j++) {
            const uint32_t x = min(b + j * per + r, n - 1u);
            to[j] = row(x);
            v[j] = *reinterpret_cast<V*>(W + x * COLS + c);
        }
#pragma unroll
        for (uint32_t j = 0; j < 4; j++) *reinterpret_cast<V*>(W + min(b + j * per + r, n - 1u) * COLS + c) = V(0.0f);
#pragma unroll
        for (uint32_t j = 0; j < 4; j++) {
            if (!in || b + j * per + r >= n) continue;
            if constexpr (ATOMIC) {
                if (to[j] != kMrhsNoRow) unsafeAtomicAdd(at<WIDE>(out, to[j], ld, col0 + c), v[j][0]);
            } else {
                // (not read again before the whole of it is written)
                __builtin_nontemporal_store(v[j], reinterpret_cast<V*>(at<WIDE>(out, to[j], ld, col0 + c)));
            }
        }
    }
}

template <bool BF16, bool V4, bool ATOMIC, bool WIDE>
__global__ __launch_bounds__(64, 2) void mrhs_cong_kernel(MrhsCongArgs a)
{
    extern __shared__ __align__(16) float W[];
    const uint32_t lane = threadIdx.x, c = lane & 15u, q = lane >> 4;
    const uint32_t ngroups = (a.nrhs + COLS - 1) / COLS;
    // slice xcd of the items, its waves interleaved: the column groups of a
    // cluster run side by side on one XCD
    const uint32_t xcd = blockIdx.x % 8u, step = gridDim.x / 8u;
    const uint64_t total = (uint64_t)a.n_clusters * ngroups;
    const uint32_t hi = (uint32_t)(total * (xcd + 1) / 8u);
    Cursor cur;
    cur.item = (uint32_t)(total * xcd / 8u) + blockIdx.x / 8u;
    if (cur.item >= hi) return;
    for (uint32_t i = lane; i < a.max_rows * COLS; i += 64u) W[i] = 0.0f;
    Ref<BF16> K;
    K.load(a.kref);
    cur.open(a, ngroups);
    Cursor nx = cur;
    nx.advance(a, ngroups, hi, step);
    // an element's DoFs are loaded two elements ahead, its rows of U, factor and
    // row slots one ahead, into the buffer that the present one does not use
    uint32_t d[2][16];
    u32x4 slots[2][2];
    Rhs<BF16, WIDE> B[2];
    f32x2 s[2];
    const f32x2* scale = static_cast<const f32x2*>(a.scale);
    load_dofs(a, cur.e, q, d[0]);
    load_slots(a, cur.e, q, slots[0]);
    s[0] = scale[cur.e];
#pragma unroll
    for (int i = 0; i < B[0].NB; i++) B[0].load(a, i, d[0][i], min(cur.col0 + c, a.nrhs - 1u));
    load_dofs(a, nx.e, q, d[1]);
    lds_sync_wave();
    // the loads for the next element have arrived (said before stores join them
    // in the counter, so that the next element does not wait for those)
    auto arrived = [&](int p) {
#pragma unroll
        for (int i = 0; i < B[0].NB; i++) asm volatile("" : "+v"(B[p].b[i]));
        asm volatile("" : "+v"(slots[p][0]), "+v"(slots[p][1]), "+v"(s[p]));
#pragma unroll
        for (int i = 0; i < 16; i++) asm volatile("" : "+v"(d[1 - p][i]));
    };
    arrived(0);
    // true: the last element of the last item
    auto element = [&](int p) {
        Cursor n2 = nx;
        n2.advance(a, ngroups, hi, step);
        const uint32_t col = min(nx.col0 + c, a.nrhs - 1u);
        f32x4 acc[4];
        float* w[16];
        float o[16];
#pragma unroll
        for (int m = 0; m < 4; m++) acc[m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        __builtin_amdgcn_sched_barrier(0);
        K.multiply(s[p], B[p], acc, [&](int i) {
            if (i < 4) {
#pragma unroll
                for (int j = 4 * i; j < 4 * i + 4 && j < B[0].NB; j++) B[1 - p].load(a, j, d[1 - p][j], col);
            }
            if (i == 3) {
                load_slots(a, nx.e, q, slots[1 - p]);
                s[1 - p] = scale[nx.e];
                load_dofs(a, n2.e, q, d[p]);
            }
            // the rows of an element are distinct (or the dump row)
            if (i >= 6 && i < 14) {
#pragma unroll
                for (int j = 2 * (i - 6); j < 2 * (i - 6) + 2; j++) {
                    const uint32_t x = slots[p][j / 8][(j / 2) % 4];
                    w[j] = reinterpret_cast<float*>(reinterpret_cast<char*>(W + c) + ((j & 1) ? x >> 16 : x & 0xffffu));
                    o[j] = *w[j];
                }
            }
        });
#pragma unroll
        for (int i = 0; i < 16; i++)
            *w[i] = o[i] + Ref<BF16>::row(s[p], acc[i / 4][i % 4]);
        lds_sync_wave();
        arrived(1 - p);
        if (cur.e + 1 == cur.end) {
            if constexpr (ATOMIC)
                put_rows<1, true, WIDE>(W, cur.n_ve, a.V, a.nrhs, a.nrhs, cur.col0,
                                        [&](uint32_t x) { return a.row_dof[cur.ve0 + x]; });
            else if (a.ve_ld == 1)
                put_rows<1, false, WIDE>(W, cur.n_ve, a.ve, 1, 1, 0, [&](uint32_t x) { return cur.ve0 + x; });
            else
                put_rows<4, false, WIDE>(W, cur.n_ve, a.ve, a.ve_ld, a.ve_ld, cur.col0,
                                         [&](uint32_t x) { return cur.ve0 + x; });
            // (atomics: another operator may add into the same V)
            if (cur.n_dir)
                put_rows<V4 ? 4 : 1, ATOMIC, WIDE>(W + cur.n_ve * COLS, cur.n_dir, a.V, a.nrhs, a.nrhs, cur.col0,
                                                  [&](uint32_t x) { return a.direct[cur.dir0 + x]; });
            lds_sync_wave();
            if (cur.item + step >= hi) return true;
        }
        __builtin_amdgcn_sched_barrier(0);
        cur = nx;
        nx = n2;
        return false;
    };
    while (!element(0) && !element(1)) {
    }
}

}  // namespace

void launch_mrhs_cong(bool bf16, const MrhsCongArgs& a, int cu_count, hipStream_t s)
{
    const uint32_t ngroups = (a.nrhs + COLS - 1) / COLS;
    const uint64_t items = (uint64_t)a.n_clusters * ngroups, slice = (items + 7) / 8;
    const uint32_t lds = a.max_rows * COLS * 4u;
    // two waves per SIMD (VGPRs)
    const uint32_t nbx = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(slice, (uint64_t)cu_count));
    const bool v4 = a.ve && a.nrhs % 4 == 0 && reinterpret_cast<uintptr_t>(a.V) % 16 == 0;
    const bool wide = (uint64_t)std::max(a.n_total, a.ve_rows) * a.ve_ld >= 1ull << 30 || a.ve_ld >= 1u << 22 ||
                      a.ve_rows >= 1u << 24;
    const dim3 grid(nbx * 8u), block(64);
#define AMX_MC(B, W)                                                                     \
    (v4 ? mrhs_cong_kernel<B, true, false, W><<<grid, block, lds, s>>>(a)                \
        : a.ve ? mrhs_cong_kernel<B, false, false, W><<<grid, block, lds, s>>>(a)        \
               : mrhs_cong_kernel<B, false, true, W><<<grid, block, lds, s>>>(a))
    if (wide) bf16 ? AMX_MC(true, true) : AMX_MC(false, true);
    else bf16 ? AMX_MC(true, false) : AMX_MC(false, false);
#undef AMX_MC
    AMX_HIP(hipGetLastError());
}

// Smaller entries and factors would lose their low parts below FP32's range, or
// their products to it; a stored matrix takes those groups.
bool mrhs_exponent(const std::vector<double>& kref, const std::vector<double>& scale, int& k)
{
    constexpr double kLeast = 0x1p-100, kMost = 0x1p126;
    double most = 0.0;
    for (double x : kref) {
        if (!std::isfinite(x)) return false;
        most = std::max(most, std::fabs(x));
    }
    if (most == 0.0) return false;
    k = std::ilogb(most);
    for (double x : kref)
        if (x != 0.0 && std::fabs(std::ldexp(x, -k)) < kLeast) return false;
    for (double x : scale) {
        const double s = std::fabs(std::ldexp(x, k));
        if (!(s == 0.0 || (s >= kLeast && s <= kMost))) return false;
    }
    return true;
}

// the FP32 value at or next to x towards zero
static float cut(double x)
{
    const float f = (float)x;
    return std::fabs((double)f) > std::fabs(x) ? std::nextafterf(f, 0.0f) : f;
}

// A row of a smooth U is a small sum of large terms; what it loses is the rounding
// of the partial sums on the way.  Column by column the one that keeps the sums
// of the three translations (every third DoF 1) smallest over all rows.  hex20
// 20^3, error relative to that of stored matrices: quadratic field 0.32, sine field
// 0.39, random U 0.82 (in the order of the DoFs 1.6, 1.5 and 0.79).
std::vector<uint8_t> mrhs_order(const std::vector<double>& kref)
{
    std::vector<uint8_t> left(N), order;
    for (int c = 0; c < N; c++) left[c] = (uint8_t)c;
    std::vector<double> sum(3 * N, 0.0);
    while (!left.empty()) {
        size_t best = 0;
        double least = 0.0;
        for (size_t i = 0; i < left.size(); i++) {
            double change = 0.0;  // of the sum of squares
            for (int r = 0; r < N; r++) {
                const double k = kref[(size_t)r * N + left[i]];
                change += k * (k + 2.0 * sum[r * 3 + left[i] % 3]);
            }
            if (i == 0 || change < least) best = i, least = change;
        }
        const int c = left[best];
        for (int r = 0; r < N; r++) sum[r * 3 + c % 3] += kref[(size_t)r * N + c];
        order.push_back((uint8_t)c);
        left.erase(left.begin() + best);
    }
    return order;
}

// K_ref in the order of Ref::load, 16-byte pieces of a lane, lanes side by side.
// BF16: value i = 16 m + 8 ks + v in two FP32 parts; FP32: i = 15 m + ks, then the
// low parts [m][t][v] in BF16 (ks = 8 t + v).
std::vector<uint8_t> mrhs_kref(const std::vector<double>& kref, int k, const std::vector<uint8_t>& order, bool bf16)
{
    const uint32_t n_val = bf16 ? 64 : 60, per = bf16 ? 2 : 4, size = bf16 ? 8 : 4, n_low = bf16 ? 0 : 64;
    std::vector<uint8_t> out((size_t)(n_val * size + n_low * 2) * 64, 0);
    for (uint32_t l = 0; l < 64; l++)
        for (uint32_t i = 0; i < n_val; i++) {
            const uint32_t m = bf16 ? i / 16 : i / 15, ks = i % 15, row = std::min(16 * m + l % 16, 59u);
            const uint32_t col = bf16 ? 32 * (i / 8 % 2) + 8 * (l / 16) + i % 8 : order[4 * ks + l / 16];
            const double x = col < N ? std::ldexp(kref[(size_t)row * N + col], -k) : 0.0;
            const float f = bf16 ? (float)x : cut(x);
            uint8_t* p = out.data() + ((size_t)(i / per * 64 + l) * per + i % per) * size;
            std::memcpy(p, &f, 4);
            float low = (float)(x - (double)f);
            if (bf16) {
                std::memcpy(p + 4, &low, 4);
            } else {
                if (low == 0.0f && f != 0.0f) low = std::copysign(FLT_MIN, f);
                uint32_t b;
                std::memcpy(&b, &low, 4);
                const uint16_t h = (uint16_t)((b + 0x7fffu + ((b >> 16) & 1u)) >> 16);
                std::memcpy(out.data() + 60 * 64 * 4 + ((size_t)(2 * m + ks / 8) * 64 + l) * 16 + ks % 8 * 2, &h, 2);
            }
        }
    return out;
}

void mrhs_factor(double s, int k, bool bf16, float (&out)[2])
{
    s = std::ldexp(s, k);
    const float hi = bf16 ? (float)s : cut(s);
    double lo = s - (double)hi;
    if (!bf16 && hi != 0.0f) {
        lo = lo == 0.0 ? std::copysign(0x1p-100, hi) : std::ldexp(lo, -std::ilogb(hi));
    }
    out[0] = hi;
    out[1] = (float)lo;
}

// Clusters: each of 8 contiguous shares of the elements by itself.  From its
// lowest free element a cluster takes, of the free elements that share nodes
// with it, the one that shares most (then the one whose shared nodes lie in
// most of its elements, then the lowest), until it has n_max elements or its
// rows are full; with no neighbour left it goes on from the next free element.
// On a structured hex20 mesh these are bricks of 2 x 2 x 2: 243 rows leave
// instead of 480, 16 of them final.  n_max: 8 where that leaves 1,024 clusters
// (four per CU), fewer below -- a wave takes the elements of a cluster in turn.
MrhsClusters mrhs_clusters(const std::vector<uint32_t>& em, const std::vector<uint8_t>& order, uint32_t n_elem,
                           uint32_t n_total, bool bf16)
{
    constexpr uint32_t kShares = 8, kNodes = N / 3, kRows = kMrhsClusterRows - 1;
    const uint32_t n_max = std::min(8u, std::max(1u, n_elem / 1024u));
    struct Share {
        std::vector<uint32_t> order, count, rows;        // elements; elements and rows per cluster
        std::vector<uint32_t> row_of;                    // DoFs of the rows, cluster by cluster
        std::vector<uint16_t> slots;                     // [element][60]
        std::vector<uint32_t> table, row_dof, direct;    // as in MrhsClusters, counted from the share's start
        uint32_t max_rows = 0;
    };
    std::vector<Share> sh(kShares);
    // every third DoF stands for its node (a map of another form only makes worse clusters)
    std::vector<uint32_t> noff(n_total + 1, 0), nel((size_t)n_elem * kNodes), valence(n_total, 0);
    for (size_t i = 0; i < em.size(); i++) valence[em[i]]++;
    for (size_t i = 0; i < em.size(); i += 3) noff[em[i] + 1]++;
    for (uint32_t d = 0; d < n_total; d++) noff[d + 1] += noff[d];
    {
        std::vector<uint32_t> fill(noff.begin(), noff.end() - 1);
        for (uint32_t e = 0; e < n_elem; e++)
            for (uint32_t a = 0; a < kNodes; a++) nel[fill[em[(size_t)e * N + 3 * a]]++] = e;
    }
    std::vector<uint8_t> taken(n_elem, 0);
    std::vector<uint32_t> shared(n_elem, 0), mult(n_elem, 0);  // of the open cluster; an element belongs to one share
    MrhsClusters C;
    C.slots.assign((size_t)n_elem * 64, 0);
    C.dofs.assign((size_t)n_elem * 64, 0);
    C.order.assign(n_elem, 0);
    auto form = [&](uint32_t p) {
        Share& S = sh[p];
        const uint32_t lo = (uint32_t)((uint64_t)n_elem * p / kShares), hi = (uint32_t)((uint64_t)n_elem * (p + 1) / kShares);
        std::vector<uint32_t> seen(n_total, 0), slot_of(n_total, 0), used(n_total, 0);
        std::vector<uint32_t> cand, members;
        uint32_t row_stamp = 0, elem_stamp = 0;
        // rows of the members, in as many clusters as they need
        auto emit = [&]() {
            uint32_t n_here = 0, rows = 0;
            row_stamp++;
            auto close = [&]() {
                if (!n_here) return;
                S.count.push_back(n_here);
                S.rows.push_back(rows);
                n_here = rows = 0;
                row_stamp++;
            };
            for (uint32_t e : members) {
                const uint32_t* d = &em[(size_t)e * N];
                // (a DoF that an element names twice gets a row each time)
                uint32_t fresh = 0;
                elem_stamp++;
                for (uint32_t r = 0; r < N; r++) {
                    fresh += seen[d[r]] != row_stamp || used[d[r]] == elem_stamp;
                    used[d[r]] = elem_stamp;
                }
                if (rows + fresh > kRows) close();
                elem_stamp++;
                for (uint32_t r = 0; r < N; r++) {
                    if (seen[d[r]] != row_stamp || used[d[r]] == elem_stamp) {
                        seen[d[r]] = row_stamp;
                        slot_of[d[r]] = rows++;
                        S.row_of.push_back(d[r]);
                    }
                    used[d[r]] = elem_stamp;
                    S.slots.push_back((uint16_t)slot_of[d[r]]);
                }
                S.order.push_back(e);
                n_here++;
            }
            close();
        };
        std::vector<uint32_t> in(n_total, 0);
        uint32_t cluster = 0, next = lo;
        for (;;) {
            while (next < hi && taken[next]) next++;
            if (next >= hi) break;
            members.clear();
            cluster++;
            uint32_t nodes = 0, seed = next;
            while (members.size() < n_max) {
                uint32_t best = 0xffffffffu;
                size_t bi = 0;
                for (size_t i = 0; i < cand.size(); i++) {
                    const uint32_t e = cand[i];
                    if (best == 0xffffffffu || shared[e] > shared[best] ||
                        (shared[e] == shared[best] && (mult[e] > mult[best] || (mult[e] == mult[best] && e < best)))) {
                        best = e;
                        bi = i;
                    }
                }
                if (best == 0xffffffffu) {
                    while (seed < hi && taken[seed]) seed++;
                    if (seed >= hi) break;
                    best = seed;
                } else {
                    cand[bi] = cand.back();
                    cand.pop_back();
                }
                if (3 * (nodes + kNodes - shared[best]) > kRows) {
                    shared[best] = mult[best] = 0;
                    break;
                }
                taken[best] = 1;
                members.push_back(best);
                nodes += kNodes - shared[best];
                for (uint32_t a = 0; a < kNodes; a++) {
                    const uint32_t d = em[(size_t)best * N + 3 * a];
                    const bool fresh = in[d] != cluster;
                    in[d] = cluster;
                    for (uint32_t j = noff[d]; j < noff[d + 1]; j++) {
                        const uint32_t e = nel[j];
                        if (e < lo || e >= hi || taken[e]) continue;
                        if (!mult[e]) cand.push_back(e);
                        shared[e] += fresh;
                        mult[e]++;
                    }
                }
                shared[best] = mult[best] = 0;
            }
            for (uint32_t e : cand) shared[e] = mult[e] = 0;
            cand.clear();
            emit();
        }
        // where the rows lie, and the elements' tables
        std::vector<uint32_t> uses, place;
        size_t e = 0, r = 0;
        for (size_t i = 0; i < S.count.size(); i++) {
            const uint32_t rows = S.rows[i], n_here = S.count[i];
            S.table.insert(S.table.end(), {(uint32_t)(lo + e), (uint32_t)S.row_dof.size(), (uint32_t)S.direct.size(), 0u});
            uses.assign(rows, 0);
            place.assign(rows, 0);
            for (size_t x = e * N; x < (e + n_here) * N; x++) uses[S.slots[x]]++;
            // final rows (every element of the DoF is here) go to V, in sixteens
            // after the others, which are padded to sixteens with at least one row,
            // the dump row; what is left of a sixteen goes through ve
            uint32_t n_dir = 0, n_ve = 0, k = 0;
            for (uint32_t x = 0; x < rows; x++) n_dir += uses[x] == valence[S.row_of[r + x]];
            n_dir &= ~15u;
            const uint32_t padded = (rows - n_dir + 16) / 16 * 16;
            // rows 4 apart, which a wave's four lane groups reach together, lie in
            // different banks: 4 x 4 transposed within 16
            auto swap4 = [](uint32_t s) { return (s & ~15u) | ((s & 3u) << 2) | ((s >> 2) & 3u); };
            const uint32_t ve0 = (uint32_t)S.row_dof.size(), dir0 = (uint32_t)S.direct.size();
            S.row_dof.resize(ve0 + padded, kMrhsNoRow);
            S.direct.resize(dir0 + n_dir);
            for (uint32_t x = 0; x < rows; x++) {
                const uint32_t d = S.row_of[r + x];
                if (k < n_dir && uses[x] == valence[d]) {
                    const uint32_t at = swap4(k++);
                    S.direct[dir0 + at] = d;
                    place[x] = padded + at;
                } else {
                    place[x] = swap4(n_ve++);
                    S.row_dof[ve0 + place[x]] = d;
                }
            }
            const uint32_t dump = swap4(n_ve);
            for (uint32_t j = 0; j < n_here; j++, e++) {
                const uint32_t el = S.order[e];
                const uint64_t at = lo + e;
                const uint32_t* d = &em[(size_t)el * N];
                const uint16_t* sl = &S.slots[e * N];
                for (uint32_t x = 0; x < 64; x++) {
                    const uint32_t q = x / 16, y = x % 16;
                    const uint32_t row = 16 * (y / 4) + 4 * q + y % 4;
                    C.slots[at * 64 + x] = (uint16_t)((row < N ? place[sl[row]] : dump) * COLS * 4);
                    const uint32_t col = bf16 ? 32 * (y / 8) + 8 * q + y % 8 : 4 * y + q;
                    C.dofs[at * 64 + x] = d[col >= N ? 0 : bf16 ? col : order[col]];
                }
                C.order[at] = el;
            }
            r += rows;
            S.max_rows = std::max(S.max_rows, padded + n_dir);
        }
    };
    std::atomic<bool> failed{false};  // (no exception leaves a parallel region)
#pragma omp parallel for schedule(static, 1) num_threads(kShares) if (n_elem > 1024)
    for (uint32_t p = 0; p < kShares; p++) {
        try {
            form(p);
        } catch (...) {
            failed = true;
        }
    }
    if (failed) throw std::bad_alloc();
    for (const Share& S : sh) {
        const uint32_t ve0 = (uint32_t)C.row_dof.size(), dir0 = (uint32_t)C.direct.size();
        for (size_t i = 0; i < S.table.size(); i += 4)
            C.table.insert(C.table.end(), {S.table[i], S.table[i + 1] + ve0, S.table[i + 2] + dir0, 0u});
        C.row_dof.insert(C.row_dof.end(), S.row_dof.begin(), S.row_dof.end());
        C.direct.insert(C.direct.end(), S.direct.begin(), S.direct.end());
        C.max_rows = std::max(C.max_rows, S.max_rows);
    }
    C.table.insert(C.table.end(), {(uint32_t)C.order.size(), (uint32_t)C.row_dof.size(), (uint32_t)C.direct.size(), 0u});
    // second pass: the DoFs that are not final, with their rows of ve in
    // ascending order
    std::vector<uint32_t> cnt(n_total, 0);
    std::vector<uint8_t> final(n_total, 0);
    for (uint32_t d : C.direct) final[d] = 1;
    for (uint32_t d : C.row_dof)
        if (d != kMrhsNoRow) cnt[d]++;
    std::vector<uint32_t> at(n_total, 0);
    C.off.push_back(0);
    for (uint32_t d = 0; d < n_total; d++)
        if (!final[d]) {
            at[d] = C.off.back();
            C.ids.push_back(d);
            C.off.push_back(C.off.back() + cnt[d]);
        }
    C.pos.resize(C.off.back());
    for (size_t i = 0; i < C.row_dof.size(); i++)
        if (C.row_dof[i] != kMrhsNoRow) C.pos[at[C.row_dof[i]]++] = (uint32_t)i;
    return C;
}

}  // namespace amx
