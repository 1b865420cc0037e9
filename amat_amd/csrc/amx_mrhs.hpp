// amx_mrhs.hpp -- multi-RHS products of congruent 60-DoF groups (amx_mrhs_cong.hip)
#pragma once
#include <cstdint>
#include <vector>

#include "amx_internal.hpp"

namespace amx {

constexpr uint32_t kMrhsNoRow = 0xffffffffu;   // row_dof of a padding row
constexpr int kMrhsClusterRows = 256;          // rows of a cluster, the dump row included, before padding

// elements in clusters; a cluster's rows are summed in LDS before they leave
struct MrhsClusters {
    std::vector<uint32_t> order;          // elements, cluster by cluster
    std::vector<uint32_t> table;          // [cluster][4]: first element of order, first row of ve, of direct
                                          // (one more entry at the end)
    std::vector<uint32_t> dofs;           // [element of order][4][16]: DoFs in B fragment order
    std::vector<uint16_t> slots;          // [element of order][4][16]: LDS byte offsets of the rows in C fragment order
    std::vector<uint32_t> row_dof;        // row of ve -> DoF or kMrhsNoRow
    std::vector<uint32_t> direct;         // DoFs whose rows are final
    std::vector<uint32_t> ids, off, pos;  // the other DoFs, their rows of ve in ascending order
    uint32_t max_rows = 0;
};
// the order in which the FP32 product takes the columns of K_ref (row-major)
std::vector<uint8_t> mrhs_order(const std::vector<double>& kref);
// em: n_elem x 60 DoFs below n_total
MrhsClusters mrhs_clusters(const std::vector<uint32_t>& em, const std::vector<uint8_t>& order, uint32_t n_elem,
                           uint32_t n_total, bool bf16);
// k: the largest entry of K_ref times 2^-k is in [1, 2).  false where an entry or a
// factor (times 2^k) leaves the range that the kernel takes.
bool mrhs_exponent(const std::vector<double>& kref, const std::vector<double>& scale, int& k);
// K_ref times 2^-k in A fragment order
std::vector<uint8_t> mrhs_kref(const std::vector<double>& kref, int k, const std::vector<uint8_t>& order, bool bf16);
// a factor as the kernel takes it: 2^k s = out[0] + out[1] (FP32: out[0] cut
// towards zero, out[1] divided by the power of two of out[0])
void mrhs_factor(double s, int k, bool bf16, float (&out)[2]);

struct MrhsCongArgs {
    const void* kref;        // mrhs_kref
    const void* scale;       // [element of order][2], mrhs_factor
    const uint32_t* dofs;
    const uint16_t* slots;
    const uint32_t *clusters, *row_dof, *direct;
    const float* U;
    float* V;
    float* ve;               // rows of ve_ld values (1 or a multiple of 4), 16-byte aligned; NULL: atomics into V (zeroed before)
    uint32_t n_clusters, nrhs, ve_ld, max_rows, n_total, ve_rows;
};
void launch_mrhs_cong(bool bf16, const MrhsCongArgs& a, int cu_count, hipStream_t s);

}  // namespace amx
