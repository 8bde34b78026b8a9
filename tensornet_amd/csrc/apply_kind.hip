// The kernels of apply_launch.h for one optimizer, TN_KIND (the library has this file three times).
#include "apply_launch.h"

#ifndef TN_KIND
#error "compiled once per optimizer: -DTN_KIND=0, 1, 2"
#endif

namespace tn {

template <int KIND>
void launch_small_apply(const SmallApplyCall& c) {
    const Store& s = c.s;
    const SmallShape& b = c.b;
    const int gfloats = small_gbuf_floats(s.D, b.N);
    const size_t arrays = align_up((size_t)(gfloats + 3 * s.D) * sizeof(float), 8), wave_lds = arrays + BIG_CHUNK * (8 + 4);
    const bool lds_big = c.with_big && (s.D > 64 || (s.D & (s.D - 1)) != 0);  // (others keep their staging in static LDS)
    const size_t lds = small_apply_slots_lds(c.flat ? 0 : b.N) + (lds_big ? 4 * wave_lds : 0);
#define TN_LAUNCH_SMALL_BIG(LPG, ANY, BIG)                                                                               \
    TN_LAUNCH_LDS_EVENT(c.done, (k_small_apply<KIND, LPG, ANY, BIG>), dim3(b.buckets()), dim3(256), lds, c.st, b, c.p,   \
                        c.flat, s, c.o, c.status, c.host_seq, c.seq, c.dim, gfloats, (uint32_t)wave_lds, (uint32_t)arrays)
// (aligned rows that fill their lanes have 4, 8 .. 128 elements; of these the last are too long for apply_big_wave)
#define TN_LAUNCH_SMALL_ROWS(LPG)                                                 \
    do {                                                                          \
        constexpr int WAVE = LPG <= 16 ? 4 * LPG : BIG_GROUPS;                    \
        if (!c.with_big && c.share.any) TN_LAUNCH_SMALL_BIG(LPG, true, BIG_NONE); \
        else if (!c.with_big) TN_LAUNCH_SMALL_BIG(LPG, false, BIG_NONE);          \
        else if (!c.share.any) TN_LAUNCH_SMALL_BIG(LPG, false, WAVE);             \
        else if (lds_big) TN_LAUNCH_SMALL_BIG(LPG, true, BIG_GROUPS);             \
        else if (s.D == 1) TN_LAUNCH_SMALL_BIG(LPG, true, (LPG == 1 ? 1 : WAVE)); \
        else if (s.D == 2) TN_LAUNCH_SMALL_BIG(LPG, true, (LPG == 1 ? 2 : WAVE)); \
        else TN_LAUNCH_SMALL_BIG(LPG, true, WAVE);                                \
    } while (0)
    switch (c.share.lanes) {
        case 1: TN_LAUNCH_SMALL_ROWS(1); break;
        case 2: TN_LAUNCH_SMALL_ROWS(2); break;
        case 4: TN_LAUNCH_SMALL_ROWS(4); break;
        case 8: TN_LAUNCH_SMALL_ROWS(8); break;
        case 16: TN_LAUNCH_SMALL_ROWS(16); break;
        default: TN_LAUNCH_SMALL_ROWS(32); break;
    }
#undef TN_LAUNCH_SMALL_ROWS
#undef TN_LAUNCH_SMALL_BIG
}
template void launch_small_apply<TN_KIND>(const SmallApplyCall& c);

template <int KIND>
void launch_table_apply(const TableApplyCall& c) {
    const Store& s = c.s;
    const bool lds_big = s.D > 64 || (s.D & (s.D - 1)) != 0;
    const size_t wave_lds = small_apply_wave_lds(s.D), lists = table_apply_lists_lds(c.b.tiles);
    const size_t lds = lists + (lds_big ? TABLE_WAVES * wave_lds : 0);
    const bool many = c.b.nb > table_apply_held(KIND);
// (MANY in the kernel's arguments: the profiler's name of the launch tells which variant it is)
#define TN_LAUNCH_TABLE_BY(LPG, ANY, BIG, MANY)                                                                             \
    do {                                                                                                                    \
        bool& told = c.lds_told[(MANY ? 2 : 0) + ANY];                                                                      \
        if (lds_big && !told) {                                                                                             \
            told = true;                                                                                                    \
            (void)big_lds_bytes_for(reinterpret_cast<const void*>(                                                          \
                k_table_apply<KIND, LPG, ANY, BIG, table_apply_most(KIND, BIG, MANY), table_apply_waves(KIND, BIG, LPG, MANY)>)); \
        }                                                                                                                   \
        TN_LAUNCH_LDS((k_table_apply<KIND, LPG, ANY, BIG, table_apply_most(KIND, BIG, MANY), table_apply_waves(KIND, BIG, LPG, MANY)>), \
                      dim3(c.b.nb), dim3(256), lds, c.st, c.b, s, c.o, c.infos, c.grads, c.dim, c.recs, c.boff, c.ds, c.host_err, \
                      big_gbuf_floats(s.D), (uint32_t)wave_lds, (uint32_t)align_up(big_lds_bytes(s.D), 8), (uint32_t)lists); \
    } while (0)
#define TN_LAUNCH_TABLE_BIG(LPG, ANY, BIG)                             \
    do {                                                               \
        if (many) TN_LAUNCH_TABLE_BY(LPG, ANY, BIG, true);             \
        else TN_LAUNCH_TABLE_BY(LPG, ANY, BIG, false);                 \
    } while (0)
#define TN_LAUNCH_TABLE(LPG)                                                      \
    do {                                                                          \
        constexpr int WAVE = LPG <= 16 ? 4 * LPG : BIG_GROUPS;                    \
        if (!c.share.any) TN_LAUNCH_TABLE_BIG(LPG, false, WAVE);                  \
        else if (lds_big) TN_LAUNCH_TABLE_BIG(LPG, true, BIG_GROUPS);             \
        else if (s.D == 1) TN_LAUNCH_TABLE_BIG(LPG, true, (LPG == 1 ? 1 : WAVE)); \
        else if (s.D == 2) TN_LAUNCH_TABLE_BIG(LPG, true, (LPG == 1 ? 2 : WAVE)); \
        else TN_LAUNCH_TABLE_BIG(LPG, true, WAVE);                                \
    } while (0)
    switch (c.share.lanes) {
        case 1: TN_LAUNCH_TABLE(1); break;
        case 2: TN_LAUNCH_TABLE(2); break;
        case 4: TN_LAUNCH_TABLE(4); break;
        case 8: TN_LAUNCH_TABLE(8); break;
        case 16: TN_LAUNCH_TABLE(16); break;
        default: TN_LAUNCH_TABLE(32); break;
    }
#undef TN_LAUNCH_TABLE
#undef TN_LAUNCH_TABLE_BIG
#undef TN_LAUNCH_TABLE_BY
}
template void launch_table_apply<TN_KIND>(const TableApplyCall& c);

}  // namespace tn
