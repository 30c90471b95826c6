// Internal launchers of the DEC kernels (host side).
#pragma once

#include "common.hpp"

namespace sil {

int launch_coboundary(int k, bool transposed, const double* in, const sil_view& vin, double* out,
                      const sil_view& vout, hipStream_t stream);
int launch_fill_hodge(const DevGeom& g, int k, double* out, hipStream_t stream);
int launch_hodge_apply(const DevGeom& g, int k, const double* in, const sil_view& vin, double* out,
                       const sil_view& vout, hipStream_t stream);
int launch_codifferential(const DevGeom& g, int k, const double* in, const sil_view& vin, double* out,
                          const sil_view& vout, hipStream_t stream);
int launch_laplacian_generic(const DevGeom& g, int k, const double* in, const sil_view& vin, double* out,
                             const sil_view& vout, hipStream_t stream);

// The same operators with the dimension and the degree as template constants
// (dec_rect.hip): rectilinear grids of regular spacings with identity or
// diagonal metric, N ≤ 3.  `g` is null for the coboundary.
enum class RectOp { Coboundary, Hodge, Codifferential, Laplacian };
bool rect_views_ok(const sil_view& vin, const sil_view& vout);
inline bool rect_geom_ok(const DevGeom& g)
{
    return g.rectilinear && g.regular && g.metric_kind != SIL_METRIC_SYMMETRIC;
}
int launch_rect(RectOp op, int k, const DevGeom* g, const double* in, const sil_view& vin, double* out,
                const sil_view& vout, hipStream_t stream);

// Fused single-pass Laplacians on rectilinear grids with identity or diagonal
// metric, index-last dense arrays.  `spacing[a]` holds the per-node edge
// length along axis a (forward, backward at the last node).
struct FusedGeom {
    int64_t ext[3];
    const double* spacing[3];
    const double* metric; // diagonal [node][ndim] or null for the identity
};

// Planes per workgroup of a march along x over `tiles` columns: the chunk with
// the least time when a compute unit takes the workgroups it is dealt in
// rounds of `resident` and a plane's step lasts 2 + (workgroups resident): the
// chain of loads and barriers of one workgroup hides behind the others'.  A
// chunk pays two more planes to start.  Within 10% of the best chunk measured
// for Δ on grids of 65³ to 513 × 300 × 301 nodes; one chunk of 32 for all took
// 49 µs where 6 take 11 (1-form, 65³).
inline int march_chunk(int64_t tiles, int64_t planes, int resident, int64_t* blocks)
{
    int64_t least = 0;
    int chunk = 2;
    for (int c = 64; c >= 2; --c) {
        const int64_t nb = tiles * ((planes + c - 1) / c), per_cu = (nb + 255) / 256;
        const int64_t full = per_cu / resident, rest = per_cu % resident;
        const int64_t cost = (full * (2 + resident) + (rest ? 2 + rest : 0)) * (c + 2);
        if (least == 0 || cost < least) {
            least = cost;
            chunk = c;
            *blocks = nb;
        }
    }
    return chunk;
}

// FUSED_DIRECT: one thread per output node, neighbours through the caches;
// FUSED_MARCH: x-march with guarded global loads, one plane prefetched;
// FUSED_PIPE: x-march with branch-free buffer accesses, two planes in flight
// FUSED_STAGE: FUSED_PIPE with z neighbours by DPP and staged contiguous stores
enum FusedVariant { FUSED_DIRECT = 0, FUSED_MARCH = 1, FUSED_PIPE = 2, FUSED_STAGE = 3 };

struct FusedTile {
    int variant;  // FusedVariant
    int tz, ty;   // tile in (z, y)
    int xchunk;   // x planes per workgroup (march)
    int nt = 0;   // pipelined 64 × 12 tile: non-temporal output stores
};

int launch_laplacian_2d_0form(const FusedGeom& g, const double* in, double* out, int64_t ox, int64_t oy,
                              hipStream_t stream);
int launch_laplacian_3d_1form(const FusedGeom& g, const double* in, double* out, const int64_t* oext,
                              const FusedTile& tile, hipStream_t stream);
int launch_coboundary_3d_0form(const double* in, double* out, const int64_t* ext, hipStream_t stream);
int launch_stream_copy(const double* in, double* out, int64_t n, hipStream_t stream);

}  // namespace sil
