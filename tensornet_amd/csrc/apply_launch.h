// The launches of the updates that come in a kernel per optimizer, row length and alignment: compiled by themselves, once per
// optimizer (apply_kind.hip).
#ifndef TN_APPLY_LAUNCH_H_
#define TN_APPLY_LAUNCH_H_

#include "table_level.h"

namespace tn {

// How the update kernels share a row out: `lanes` lanes, four elements each (0: the row is too long for that).
// any: the rows do not fill the lanes, or stand at other than 16-byte boundaries (row_part<true>).
struct RowShare {
    int lanes;
    bool any;
};
inline RowShare row_share(const Store& s, bool aligned) {
    RowShare r{1, !aligned || s.D % 4 != 0};
    while (4 * r.lanes < s.D) r.lanes *= 2;
    if (4 * r.lanes != s.D) r.any = true;
    if (r.lanes > 32) r.lanes = 0;
    return r;
}

struct SmallApplyCall {
    SmallShape b;
    SmallPlan p;
    const float* flat;
    Store s;
    OptDev o;
    const DevStatus* status;
    uint32_t* host_seq;
    uint32_t seq;
    int dim;
    RowShare share;
    bool with_big;  // the plan lists signs with many records
    hipStream_t st;
    hipEvent_t done;
};
template <int KIND>
void launch_small_apply(const SmallApplyCall& c);

struct TableApplyCall {
    TableShape b;
    Store s;
    OptDev o;
    const tn_sign_info* infos;
    const float* grads;
    int dim;
    const uint2* recs;
    const uint16_t* boff;
    DevStatus* ds;
    uint32_t* host_err;
    RowShare share;
    hipStream_t st;
    bool* lds_told;  // [4]: the kernels (rows in 16-byte pieces / any, the variants for few / many workgroups) have been told how much LDS they may have
};
template <int KIND>
void launch_table_apply(const TableApplyCall& c);

}  // namespace tn

#endif  // TN_APPLY_LAUNCH_H_
