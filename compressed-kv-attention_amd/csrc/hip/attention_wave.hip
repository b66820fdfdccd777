// Entry points of the one-wave split kernel (attention_wave.h) and its
// merges; the split kernels themselves are instantiated per head_dim and
// score order in attention_wave_d<D>_o<O>.hip.
#include "attention_team.h"

namespace kvexp_launch {
using namespace kvexp_dev;

// The split kernel of each head_dim: the one-wave kernel (attention_wave.h) at
// 32 and 64, the team kernel (attention_team.h) at the larger ones; the AVX-512
// order needs a multiple of 32. X(head_dim): the sizes with a kernel.
#define KVEXP_WAVE_DIMS(X) X(32) X(64)
#define KVEXP_TEAM_DIMS_32(X) X(96) X(128) X(160) X(192) X(224) X(256)
#define KVEXP_TEAM_DIMS_16(X) X(80) X(112)

#define KVEXP_WAVE_DECL(D, O)                                                                                        \
    hipError_t attention_wave_d##D##_o##O(bool xkv, int G, const HeadDev *heads, const WorkItem *items,             \
                                         int n_items, int wpg, const BlockDesc *desc,                  \
                                         const uint16_t *q, float *out, float *lse, float *ws, hipStream_t s);
#define KVEXP_TEAM_DECL(D, O)                                                                                        \
    hipError_t attention_team_d##D##_o##O(bool xkv, int G, const HeadDev *heads, const WorkItem *items,             \
                                         int n_items, const BlockDesc *desc, const uint16_t *q,        \
                                         float *out, float *lse, float *ws, hipStream_t s);
#define KVEXP_WAVE_DECL_BOTH(D) KVEXP_WAVE_DECL(D, 0) KVEXP_WAVE_DECL(D, 1)
#define KVEXP_TEAM_DECL_BOTH(D) KVEXP_TEAM_DECL(D, 0) KVEXP_TEAM_DECL(D, 1)
#define KVEXP_TEAM_DECL_0(D) KVEXP_TEAM_DECL(D, 0)
KVEXP_WAVE_DIMS(KVEXP_WAVE_DECL_BOTH)
KVEXP_TEAM_DIMS_32(KVEXP_TEAM_DECL_BOTH)
KVEXP_TEAM_DIMS_16(KVEXP_TEAM_DECL_0)

#define KVEXP_DIM_CASE(D) case D:

// The head_dims of these kernels, both score orders where the order allows
// the size (the host sends other sizes to the general kernel).
bool wave_supports(int dim) {
    switch (dim) {
        KVEXP_WAVE_DIMS(KVEXP_DIM_CASE)
        KVEXP_TEAM_DIMS_32(KVEXP_DIM_CASE)
        KVEXP_TEAM_DIMS_16(KVEXP_DIM_CASE)
        return true;
    default: return false;
    }
}

// Splits of G query rows that stay resident on a CU: at head_dim 32 and 64 the
// one-wave kernel's waves (four per SIMD, and three, or two at eight rows,
// whose LDS leaves room for two workgroups), else the team kernel's teams; the
// general kernel of the other sizes counts as two four-wave workgroups of four
// splits each. `uneven` (lengths of several sizes, or query rows in launches of
// several sizes): more teams than fit above four rows, and twice those that fit
// at 160 to 224, since the short splits fill in behind the long and a launch of
// some of the rows holds less than a round. Four sequences of up to 25,003
// tokens x 8 heads, eight rows of 256: cut for 1,024 teams 90.1 us, for the 768
// that fit 93.7 (other batches 130.6 and 143.0, 122.4 and 117.8); 8 heads x
// 30,000 tokens, 20 rows of 192: for 2,048 teams 155.9, for 1,024 171.9; 16 x
// 4,000, twelve plain rows of 256: for 1,024 48.6, for 768 58.0.
int resident_splits(int dim, int G, bool uneven) {
#define KVEXP_RESIDENT_CASE(D)                                                                                       \
    case D:                                                                                                          \
        return uneven ? (D == 256 ? 4 : 8)                                                                           \
                      : (G > 4 ? team::kTeamOcc<8, D> : team::kTeamOcc<4, D>) * 4 / team::TShape<D>::W;
    switch (dim) {
    case 32: return 16;
    case 64: return G < 8 ? 12 : 8;
        KVEXP_TEAM_DIMS_32(KVEXP_RESIDENT_CASE)
        KVEXP_TEAM_DIMS_16(KVEXP_RESIDENT_CASE)
    default: return 8;
    }
#undef KVEXP_RESIDENT_CASE
}

// Work items per workgroup of the split kernel: consecutive ones share a
// workgroup of the one-wave kernel; a team is a workgroup.
int wave_waves_per_wg(int dim) { return dim <= 64 ? wave::Shape<64>::kWaves : 1; }

hipError_t wave_merge(int dim, const MergeItem *mitems, int n_mitems, const MergeItem &uni, float *out, float *lse,
                      const float *ws, hipStream_t s) {
    if (n_mitems <= 0) return hipSuccess;
    const int grid = (n_mitems + wave::kMergeWaves - 1) / wave::kMergeWaves;
#define KVEXP_MERGE_CASE(D)                                                                                          \
    case D:                                                                                                          \
        hipLaunchKernelGGL(wave::wave_merge_kernel<D>, dim3(grid, (D + 63) / 64), dim3(wave::kMergeWaves * 64), 0, s, \
                           mitems, n_mitems, uni, out, lse, ws);                                                             \
        break;
    switch (dim) {
        KVEXP_WAVE_DIMS(KVEXP_MERGE_CASE)
        KVEXP_TEAM_DIMS_32(KVEXP_MERGE_CASE)
        KVEXP_TEAM_DIMS_16(KVEXP_MERGE_CASE)
    default: return hipErrorInvalidValue;
    }
#undef KVEXP_MERGE_CASE
    return hipGetLastError();
}

hipError_t attention_wave(bool xkv, int order, int G, int dim, const HeadDev *heads, const WorkItem *items,
                          int n_items, int wpg, const BlockDesc *desc, const uint16_t *q, float *out,
                          float *lse, float *ws, hipStream_t s) {
    if (n_items <= 0) return hipSuccess;
    if (order != 0 && order != 1) return hipErrorInvalidValue;
#define KVEXP_WAVE_CASE(D)                                                                                           \
    case D:                                                                                                          \
        return order == 0 ? attention_wave_d##D##_o0(xkv, G, heads, items, n_items, wpg, desc, q, out, lse, ws, s)   \
                          : attention_wave_d##D##_o1(xkv, G, heads, items, n_items, wpg, desc, q, out, lse, ws, s);
#define KVEXP_TEAM_CASE_32(D)                                                                                        \
    case D:                                                                                                          \
        return order == 0 ? attention_team_d##D##_o0(xkv, G, heads, items, n_items, desc, q, out, lse, ws, s)        \
                          : attention_team_d##D##_o1(xkv, G, heads, items, n_items, desc, q, out, lse, ws, s);
#define KVEXP_TEAM_CASE_16(D)                                                                                        \
    case D:                                                                                                          \
        if (order != 0) break;                                                                                       \
        return attention_team_d##D##_o0(xkv, G, heads, items, n_items, desc, q, out, lse, ws, s);
    switch (dim) {
        KVEXP_WAVE_DIMS(KVEXP_WAVE_CASE)
        KVEXP_TEAM_DIMS_32(KVEXP_TEAM_CASE_32)
        KVEXP_TEAM_DIMS_16(KVEXP_TEAM_CASE_16)
    default: break;
    }
#undef KVEXP_WAVE_CASE
#undef KVEXP_TEAM_CASE_32
#undef KVEXP_TEAM_CASE_16
    return hipErrorInvalidValue;
}

} // namespace kvexp_launch

#if defined(KVEXP_PHASE_TRACE)
namespace kvexp_launch {
hipError_t attention_wave_d64_o0_trace_read(unsigned long long *host, size_t n);
hipError_t attention_team_d128_o0_trace_read(unsigned long long *host, size_t n);
hipError_t attention_team_d256_o0_trace_read(unsigned long long *host, size_t n);
} // namespace kvexp_launch
// Copies the phase trace of the last traced launch at head_dim `dim` (n
// words) to the host (trace builds only).
extern "C" int kvexp_hip_phase_trace_read(unsigned long long *host, size_t n, int dim) {
    using namespace kvexp_launch;
    if (dim == 64) return int(attention_wave_d64_o0_trace_read(host, n));
    if (dim == 128) return int(attention_team_d128_o0_trace_read(host, n));
    if (dim == 256) return int(attention_team_d256_o0_trace_read(host, n));
    return int(hipErrorInvalidValue);
}
#endif
