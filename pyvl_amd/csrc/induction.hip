// Line-vortex induction on gfx950: dense matrix assembly, induction tensors and
// point-velocity sums.  All kernels are compiled with -ffp-contract=off, so every FP64
// expression below rounds exactly as written (no FMA contraction), matching the
// reference's x86-64 baseline build.
#include "pvl_internal.hpp"
#include "induction_core.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>

// Calls f(std::integral_constant<int, P>{}) for the precision form P selected at run time.
template <class F> static void dispatch_precision(int precision, F &&f)
{
    if (precision == PVL_FP32)
        f(std::integral_constant<int, PVL_FP32>{});
    else if (precision == PVL_FP64_REF_FORM)
        f(std::integral_constant<int, PVL_FP64_REF_FORM>{});
    else
        f(std::integral_constant<int, PVL_FP64>{});
}

using namespace pvl;

namespace
{

constexpr int kWave = 64;
constexpr int kBlock = 256; // 4 waves
constexpr int kCptTile = 64; // control points per workgroup (one per lane)

// ---------------------------------------------------------------------------------------
// Per-line prologue (src/core/flow_solver.c:95-103): end points, |d| and d/|d| with three
// true divisions.
// A line shorter than tol is cut off for every point (K = 0 in every form); its direction
// and length are stored as 0 (instead of the 0/0 of a zero-length line), so that its angle
// and the fused accumulation (0 * direction) are 0.  With tol <= 0 nothing is cut by length
// and the reference's values, NaN included, are kept.
__device__ __forceinline__ LineGeom line_geom(const uint32_t *__restrict__ ab, const double *__restrict__ pos,
                                              double tol)
{
    const uint32_t p1 = ab[0] & kInvalidId, p2 = ab[1] & kInvalidId;
    LineGeom g;
    g.r1x = pos[3 * p1 + 0], g.r1y = pos[3 * p1 + 1], g.r1z = pos[3 * p1 + 2];
    g.r2x = pos[3 * p2 + 0], g.r2y = pos[3 * p2 + 1], g.r2z = pos[3 * p2 + 2];
    const double dx = g.r2x - g.r1x, dy = g.r2y - g.r1y, dz = g.r2z - g.r1z;
    g.len = sqrt(dx * dx + dy * dy + dz * dz);
    g.ex = dx / g.len;
    g.ey = dy / g.len;
    g.ez = dz / g.len;
    if (g.len < tol)
        g.ex = g.ey = g.ez = g.len = 0.0;
    return g;
}
__global__ void __launch_bounds__(256) line_geom_kernel(unsigned n_lines, const uint32_t *__restrict__ lines,
                                                       const double *__restrict__ pos, double tol,
                                                       LineGeom *__restrict__ out)
{
    main_stream_priority();
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n_lines)
        out[i] = line_geom(lines + 2 * i, pos, tol);
}

__device__ __forceinline__ unsigned wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x / kWave); }
__device__ __forceinline__ unsigned lane_id() { return threadIdx.x % kWave; }

// ---------------------------------------------------------------------------------------
// Surface-reduced induction tensor: one lane per control point, the wave walks a run of
// surfaces (wave-uniform, so surface/line metadata and line geometry come through scalar
// loads).  Each surface accumulates +-K in its CSR order (src/core/flow_solver.c:141-172).
// K of the lines of the previous surface is kept in registers: consecutive surfaces of
// structured meshes share a line.  Results are staged in LDS and written row-contiguous.
//   VEC:    out[n_cpts][n_surf][3]   (induction_matrix)
//   NORMAL: out[n_cpts][n_surf], dotted with the control point's normal (:202); the library
//           assembles induction_matrix3 with assembly_kernel instead.
template <bool NORMAL, int PREC, int SURF_PER_WAVE>
__global__ void __launch_bounds__(kBlock)
    surface_induction_kernel(unsigned n_cpts, unsigned n_surf, const uint32_t *__restrict__ offsets,
                             const uint32_t *__restrict__ entries, const LineGeom *__restrict__ geom,
                             const double *__restrict__ cpts, const double *__restrict__ normals,
                             double *__restrict__ out, double tol)
{
    main_stream_priority();
    constexpr int kSurfTile = 4 * SURF_PER_WAVE;
    constexpr int kComp = NORMAL ? 1 : 3;
    constexpr int kRow = kSurfTile * kComp + 1; // padded LDS row (doubles)
    __shared__ double tile[kCptTile * kRow];

    const unsigned w = wave_id(), lane = lane_id();
    const unsigned cp0 = blockIdx.y * kCptTile;
    const unsigned s_tile0 = blockIdx.x * kSurfTile;
    const unsigned cp = cp0 + lane;
    const bool live = cp < n_cpts;
    const unsigned cpc = live ? cp : n_cpts - 1;
    const double px = cpts[3 * cpc + 0], py = cpts[3 * cpc + 1], pz = cpts[3 * cpc + 2];
    double nx = 0, ny = 0, nz = 0;
    if (NORMAL)
        nx = normals[3 * cpc + 0], ny = normals[3 * cpc + 1], nz = normals[3 * cpc + 2];
    const double tol2 = tol * tol;

    // register cache of the previous surface's first four lines
    uint32_t oid0 = 0xFFFFFFFFu, oid1 = 0xFFFFFFFFu, oid2 = 0xFFFFFFFFu, oid3 = 0xFFFFFFFFu;
    double o0x = 0, o0y = 0, o0z = 0, o1x = 0, o1y = 0, o1z = 0, o2x = 0, o2y = 0, o2z = 0, o3x = 0, o3y = 0,
           o3z = 0;

    for (int j = 0; j < SURF_PER_WAVE; ++j)
    {
        const unsigned sl = w * SURF_PER_WAVE + j; // local surface
        const unsigned s = s_tile0 + sl;
        double rx = 0.0, ry = 0.0, rz = 0.0;
        uint32_t nid0 = 0xFFFFFFFFu, nid1 = 0xFFFFFFFFu, nid2 = 0xFFFFFFFFu, nid3 = 0xFFFFFFFFu;
        double c0x = 0, c0y = 0, c0z = 0, c1x = 0, c1y = 0, c1z = 0, c2x = 0, c2y = 0, c2z = 0, c3x = 0, c3y = 0,
               c3z = 0;
        if (s < n_surf)
        {
            const uint32_t k0 = offsets[s], k1 = offsets[s + 1];
            for (uint32_t k = k0; k < k1; ++k)
            {
                const uint32_t e = entries[k];
                const uint32_t l = e & kInvalidId;
                double kx, ky, kz;
                if (l == oid0)
                    kx = o0x, ky = o0y, kz = o0z;
                else if (l == oid1)
                    kx = o1x, ky = o1y, kz = o1z;
                else if (l == oid2)
                    kx = o2x, ky = o2y, kz = o2z;
                else if (l == oid3)
                    kx = o3x, ky = o3y, kz = o3z;
                else
                    line_k<PREC>(geom[l], px, py, pz, tol, tol2, kx, ky, kz);
                const uint32_t slot = k - k0;
                if (slot == 0)
                    nid0 = l, c0x = kx, c0y = ky, c0z = kz;
                else if (slot == 1)
                    nid1 = l, c1x = kx, c1y = ky, c1z = kz;
                else if (slot == 2)
                    nid2 = l, c2x = kx, c2y = ky, c2z = kz;
                else if (slot == 3)
                    nid3 = l, c3x = kx, c3y = ky, c3z = kz;
                if (e & kReversed)
                {
                    rx = rx - kx;
                    ry = ry - ky;
                    rz = rz - kz;
                }
                else
                {
                    rx = rx + kx;
                    ry = ry + ky;
                    rz = rz + kz;
                }
            }
        }
        oid0 = nid0, oid1 = nid1, oid2 = nid2, oid3 = nid3;
        o0x = c0x, o0y = c0y, o0z = c0z, o1x = c1x, o1y = c1y, o1z = c1z;
        o2x = c2x, o2y = c2y, o2z = c2z, o3x = c3x, o3y = c3y, o3z = c3z;
        if (NORMAL)
        {
            tile[lane * kRow + sl] = rx * nx + ry * ny + rz * nz;
        }
        else
        {
            tile[lane * kRow + 3 * sl + 0] = rx;
            tile[lane * kRow + 3 * sl + 1] = ry;
            tile[lane * kRow + 3 * sl + 2] = rz;
        }
    }
    __syncthreads();
    // Row-contiguous store: each wave writes 16 control-point rows.
    const unsigned s_count = (n_surf - s_tile0) < kSurfTile ? (n_surf - s_tile0) : kSurfTile;
    const unsigned row_len = s_count * kComp;
    for (unsigned r = w; r < kCptTile; r += 4)
    {
        const unsigned cpr = cp0 + r;
        if (cpr >= n_cpts)
            break;
        double *dst = out + ((size_t)cpr * n_surf + s_tile0) * kComp;
        for (unsigned c = lane; c < row_len; c += kWave)
            dst[c] = tile[r * kRow + c];
    }
}

// Normal-reduced assembly (induction_matrix3), out[n_cpts][n_surf]: one lane per control
// point, one wave per run of one to kAsmGroups groups of kAsmSurfaces consecutive surfaces,
// executing the run's program (build_assembly_program): each line of the run is evaluated
// once, as n . K, and kept in an LDS slot while a later surface of the run needs it; a
// surface's value is the sum of its lines' +-n.K in CSR order (src/core/flow_solver.c:188-202
// sums the vectors first and then dots with the normal: the same terms, another association).
// Program entries are wave-uniform (scalar loads and branches); per lane the inner step is one
// K and one LDS access at most.  Each group's results are staged in LDS and stored as rows of
// kAsmSurfaces consecutive doubles.  Bound by FP64 issue where the chip is full (~60 slots per line
// in the far form, which all but 1 % of the waves' lines take at 16,384 surfaces: 1.50 ms, 2.10 in
// the general form) and by the latency of a wave's chain of evaluations where it is not.  A pair's
// program words are loaded one pair ahead; loading its lines ahead as well (two records more in
// scalar registers, or one with everything copied to VGPRs first) spilled and was slower (2.1 ms).
// Four waves per SIMD, which the LDS allows, leave the registers for the coefficients.
template <int PREC>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4)))
    assembly_kernel(unsigned n_cpts, unsigned n_surf, unsigned n_runs, const uint32_t *__restrict__ run_off,
                    const uint32_t *__restrict__ run_grp, const uint32_t *__restrict__ prog,
                    const LineGeom *__restrict__ geom, const double *__restrict__ cpts,
                    const double *__restrict__ normals, double *__restrict__ out, double tol)
{
    main_stream_priority();
    __shared__ double slots[4][kAsmSlots][kWave];
    __shared__ double res[4][kAsmSurfaces][kWave + 1];
    const unsigned w = wave_id(), lane = lane_id();
    const unsigned cp0 = blockIdx.y * kCptTile;
    const unsigned cp = cp0 + lane;
    const unsigned cpc = cp < n_cpts ? cp : n_cpts - 1;
    const double px = cpts[3 * cpc + 0], py = cpts[3 * cpc + 1], pz = cpts[3 * cpc + 2];
    const double nx = normals[3 * cpc + 0], ny = normals[3 * cpc + 1], nz = normals[3 * cpc + 2];
    const double tol2 = tol * tol;
    const unsigned run = blockIdx.x * 4 + w;
    if (run >= n_runs)
        return;
    const uint32_t k0 = run_off[run], k1 = run_off[run + 1];
    unsigned gi = 0;
    uint32_t grp = run_grp[run * kAsmGroups];
    unsigned ns = min(kAsmSurfaces, n_surf - grp * kAsmSurfaces); // surfaces of the current group
    unsigned sl = 0;
    double acc = 0.0;
    // pairs of entries: both entries' scalar loads (program words and line geometry) are
    // issued before either is evaluated, so one wait covers two evaluations (scalar loads
    // return out of order: a wave can only wait for all of them)
    auto step = [&](uint32_t e, uint32_t op, const LineGeom &g) {
        const uint32_t kind = op & 3u, slot = (op >> 2) & 15u;
        double v;
        if (kind == kAsmLoad)
            v = slots[w][slot][lane];
        else if (kind == kAsmNone)
            v = 0.0;
        else
        {
            v = line_nk<PREC>(g, px, py, pz, nx, ny, nz, tol, tol2);
            if (kind == kAsmEvalStore)
                slots[w][slot][lane] = v;
        }
        acc = (e & kReversed) ? acc - v : acc + v;
        if (op & kAsmEnd)
        {
            res[w][sl][lane] = acc;
            acc = 0.0;
            ++sl;
        }
    };
    // groups have even entry counts (padded), so a group ends on a pair boundary
    if (k0 >= k1)
        return;
    const uint4 *words = (const uint4 *)prog;
    uint4 next = words[k0 / 2];
    for (uint32_t k = k0; k < k1; k += 2)
    {
        // a kAsmNone entry names line 0 (the geometry buffer always has one element)
        const uint32_t ea = next.x, opa = next.y, eb = next.z, opb = next.w;
        const LineGeom ga = geom[ea & kInvalidId], gb = geom[eb & kInvalidId];
        next = words[min(k + 2, k1 - 2) / 2];
        // both geometries in SGPRs here (the compiler would otherwise sink the second load
        // into the branch that uses it, after the first evaluation)
        asm volatile("" ::"s"(ga.r1x), "s"(ga.r2x), "s"(ga.ex), "s"(ga.len), "s"(gb.r1x), "s"(gb.r2x), "s"(gb.ex),
                     "s"(gb.len), "s"(next.x));
        step(ea, opa, ga);
        step(eb, opb, gb);
        if (sl == ns)
        {
            // the group's rows: lane = 8 rows x 8 surfaces per store instruction
            const unsigned s0 = grp * kAsmSurfaces, c = lane % kAsmSurfaces;
            for (unsigned r = lane / kAsmSurfaces; r < kCptTile; r += kWave / kAsmSurfaces)
            {
                const unsigned p = cp0 + r;
                if (p < n_cpts && c < ns)
                    out[(size_t)p * n_surf + s0 + c] = res[w][c][r];
            }
            sl = 0;
            if (++gi < kAsmGroups)
            {
                grp = run_grp[run * kAsmGroups + gi];
                if (grp != kAsmNoGroup)
                    ns = min(kAsmSurfaces, n_surf - grp * kAsmSurfaces);
            }
        }
    }
}

// Raw line tensor out[n_cpts][n_lines][3] (src/core/flow_solver.c:86-139 with its
// cpt-major layout :110,136).
template <int PREC, int LINES_PER_WAVE>
__global__ void __launch_bounds__(kBlock)
    line_induction_kernel(unsigned n_cpts, unsigned n_lines, const LineGeom *__restrict__ geom,
                          const double *__restrict__ cpts, double *__restrict__ out, double tol)
{
    main_stream_priority();
    constexpr int kLineTile = 4 * LINES_PER_WAVE;
    constexpr int kRow = kLineTile * 3 + 1;
    __shared__ double tile[kCptTile * kRow];
    const unsigned w = wave_id(), lane = lane_id();
    const unsigned cp0 = blockIdx.y * kCptTile;
    const unsigned l_tile0 = blockIdx.x * kLineTile;
    const unsigned cp = cp0 + lane;
    const unsigned cpc = cp < n_cpts ? cp : n_cpts - 1;
    const double px = cpts[3 * cpc + 0], py = cpts[3 * cpc + 1], pz = cpts[3 * cpc + 2];
    const double tol2 = tol * tol;
    for (int j = 0; j < LINES_PER_WAVE; ++j)
    {
        const unsigned ll = w * LINES_PER_WAVE + j;
        const unsigned l = l_tile0 + ll;
        double kx = 0, ky = 0, kz = 0;
        if (l < n_lines)
            line_k<PREC>(geom[l], px, py, pz, tol, tol2, kx, ky, kz);
        tile[lane * kRow + 3 * ll + 0] = kx;
        tile[lane * kRow + 3 * ll + 1] = ky;
        tile[lane * kRow + 3 * ll + 2] = kz;
    }
    __syncthreads();
    const unsigned l_count = (n_lines - l_tile0) < kLineTile ? (n_lines - l_tile0) : kLineTile;
    const unsigned row_len = 3 * l_count;
    for (unsigned r = w; r < kCptTile; r += 4)
    {
        const unsigned cpr = cp0 + r;
        if (cpr >= n_cpts)
            break;
        double *dst = out + ((size_t)cpr * n_lines + l_tile0) * 3;
        for (unsigned c = lane; c < row_len; c += kWave)
            dst[c] = tile[r * kRow + c];
    }
}

// ---------------------------------------------------------------------------------------
// Point-velocity sums.  Line circulation gamma_l = sum over the surfaces holding line l
// of +-Gamma_s, in increasing surface order (deterministic).
__device__ __forceinline__ double line_circulation(unsigned i, const uint32_t *__restrict__ loff,
                                                   const uint32_t *__restrict__ lsurf,
                                                   const double *__restrict__ circ)
{
    double g = 0.0;
    for (uint32_t k = loff[i]; k < loff[i + 1]; ++k)
    {
        const uint32_t e = lsurf[k];
        const double c = circ[e & kInvalidId];
        g = (e & kReversed) ? g - c : g + c;
    }
    return g;
}
__global__ void __launch_bounds__(256) line_circulation_kernel(unsigned n_lines, const uint32_t *__restrict__ loff,
                                                               const uint32_t *__restrict__ lsurf,
                                                               const double *__restrict__ circ,
                                                               double *__restrict__ gamma)
{
    main_stream_priority();
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n_lines)
        gamma[i] = line_circulation(i, loff, lsurf, circ);
}
// Both in one launch, for the point-velocity sums.
__global__ void __launch_bounds__(256) line_record_kernel(unsigned n_lines, const uint32_t *__restrict__ lines,
                                                          const double *__restrict__ pos, double tol,
                                                          const uint32_t *__restrict__ loff,
                                                          const uint32_t *__restrict__ lsurf,
                                                          const double *__restrict__ circ, LineGeom *__restrict__ geom,
                                                          double *__restrict__ gamma)
{
    main_stream_priority();
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_lines)
        return;
    geom[i] = line_geom(lines + 2 * i, pos, tol);
    gamma[i] = line_circulation(i, loff, lsurf, circ);
}

// PPL points per lane (64 PPL per wave, point j * 64 + lane of the block); the workgroup's
// four waves split a chunk of lines, partial sums are combined in LDS in wave order and
// written per chunk; a second pass adds the chunks in chunk order.  No atomics: the result
// does not depend on scheduling.  Work items are (64 PPL-point block, line chunk) pairs,
// item = chunk * pblocks + block; workgroup b takes items b, b + gridDim.x, .. (a grid
// smaller than the item count leaves CU slots to other work on the device; each item's
// arithmetic is the same either way).  Bound by FP64 issue: 46 slots per far pair (by counters
// 50 VALU instructions per pair at 81 % issue, the near ones among them).  With PPL = 2
// each lane runs two independent evaluation chains per line and every line's record, loaded once
// into scalar registers, serves twice the points: 30,000 points x 16,256 lines take 0.75 ms (1.45 ms
// in the general form with one point per lane).
// SITE only gives the free-wake self-induction launch its own symbol for profilers.
// Where items of two points per lane would leave SIMDs short of waves, each lane takes one
// (point_velocity_ppl): a wave's chain of lines takes half the time.
template <int PREC, int SITE, int PPL>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4)))
    point_velocity_kernel(unsigned n_pts, const double *__restrict__ pts, unsigned n_lines,
                          const LineGeom *__restrict__ geom, const double *__restrict__ gamma,
                          unsigned lines_per_chunk, double *__restrict__ partial, double tol, unsigned pblocks,
                          unsigned n_items)
{
    if constexpr (SITE == 0)
        main_stream_priority();
    __shared__ double red[4][3][kWave * PPL];
    const unsigned w = wave_id(), lane = lane_id();
    const double tol2 = tol * tol;
    const unsigned per_wave = (lines_per_chunk + 3) / 4;
    for (unsigned item = blockIdx.x; item < n_items; item += gridDim.x)
    {
        const unsigned chunk = item / pblocks;
        const unsigned p0 = (item - chunk * pblocks) * (kWave * PPL) + lane;
        double px[PPL], py[PPL], pz[PPL], vx[PPL], vy[PPL], vz[PPL];
#pragma unroll
        for (int j = 0; j < PPL; ++j)
        {
            const unsigned p = p0 + j * kWave;
            const unsigned pc = p < n_pts ? p : n_pts - 1;
            px[j] = pts[3 * pc + 0], py[j] = pts[3 * pc + 1], pz[j] = pts[3 * pc + 2];
            vx[j] = 0.0, vy[j] = 0.0, vz[j] = 0.0;
        }
        const unsigned l0 = chunk * lines_per_chunk;
        const unsigned l1 = (l0 + lines_per_chunk) < n_lines ? (l0 + lines_per_chunk) : n_lines;
        const unsigned a = l0 + w * per_wave;
        const unsigned b = (a + per_wave) < l1 ? (a + per_wave) : l1;
        for (unsigned l = a; l < b; ++l)
        {
            const LineGeom g = geom[l];
            line_k_acc<PREC, PPL>(g, gamma[l], px, py, pz, tol, tol2, vx, vy, vz);
        }
#pragma unroll
        for (int j = 0; j < PPL; ++j)
        {
            red[w][0][j * kWave + lane] = vx[j];
            red[w][1][j * kWave + lane] = vy[j];
            red[w][2][j * kWave + lane] = vz[j];
        }
        __syncthreads();
        if (w == 0)
        {
#pragma unroll
            for (int j = 0; j < PPL; ++j)
            {
                const unsigned p = p0 + j * kWave;
                if (p >= n_pts)
                    continue;
                const unsigned i = j * kWave + lane;
                double sx = red[0][0][i], sy = red[0][1][i], sz = red[0][2][i];
                for (int q = 1; q < 4; ++q)
                {
                    sx = sx + red[q][0][i];
                    sy = sy + red[q][1][i];
                    sz = sz + red[q][2][i];
                }
                double *dst = partial + ((size_t)chunk * n_pts + p) * 3;
                dst[0] = sx;
                dst[1] = sy;
                dst[2] = sz;
            }
        }
        __syncthreads(); // red is rewritten by the next item
    }
}

__global__ void __launch_bounds__(256) chunk_reduce_kernel(unsigned n_pts, unsigned n_chunks,
                                                           const double *__restrict__ partial,
                                                           double *__restrict__ out, int accumulate)
{
    main_stream_priority();
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 3 * n_pts)
        return;
    double s = accumulate ? out[i] : 0.0;
#pragma unroll 8
    for (unsigned c = 0; c < n_chunks; ++c)
        s = s + partial[(size_t)c * 3 * n_pts + i];
    out[i] = s;
}

// ---------------------------------------------------------------------------------------
// Surface normal and centre (src/core/mesh.c:14-68).
__global__ void __launch_bounds__(256) surface_geometry_kernel(unsigned n_surf, const uint32_t *__restrict__ offsets,
                                                               const uint32_t *__restrict__ entries,
                                                               const uint32_t *__restrict__ lines,
                                                               const double *__restrict__ pos,
                                                               double *__restrict__ normal_out,
                                                               double *__restrict__ center_out)
{
    main_stream_priority();
    const unsigned s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n_surf)
        return;
    const uint32_t k0 = offsets[s], k1 = offsets[s + 1];
    if (k1 <= k0)
    {
        // empty surface: no entries to read (the reference divides 0 by 0 here)
        const double nan = __builtin_nan("");
        for (int c = 0; c < 3; ++c)
        {
            if (center_out)
                center_out[3 * s + c] = nan;
            if (normal_out)
                normal_out[3 * s + c] = nan;
        }
        return;
    }
    if (center_out)
    {
        // sum of each line's start point in traversal direction, times 1/n
        double cx = 0.0, cy = 0.0, cz = 0.0;
        for (uint32_t k = k0; k < k1; ++k)
        {
            const uint32_t e = entries[k];
            const uint32_t l = e & kInvalidId;
            const uint32_t p = (e & kReversed) ? (lines[2 * l + 1] & kInvalidId) : (lines[2 * l] & kInvalidId);
            cx = cx + pos[3 * p + 0];
            cy = cy + pos[3 * p + 1];
            cz = cz + pos[3 * p + 2];
        }
        const double div = 1.0 / (double)(k1 - k0);
        center_out[3 * s + 0] = cx * div;
        center_out[3 * s + 1] = cy * div;
        center_out[3 * s + 2] = cz * div;
    }
    if (normal_out)
    {
        // line_direction: p1 - p2 for a forward line, p2 - p1 for a reversed one
        auto dir = [&](uint32_t e, double &x, double &y, double &z) {
            const uint32_t l = e & kInvalidId;
            const uint32_t a = lines[2 * l] & kInvalidId, b = lines[2 * l + 1] & kInvalidId;
            const uint32_t u = (e & kReversed) ? b : a, v = (e & kReversed) ? a : b;
            x = pos[3 * u + 0] - pos[3 * v + 0];
            y = pos[3 * u + 1] - pos[3 * v + 1];
            z = pos[3 * u + 2] - pos[3 * v + 2];
        };
        double d1x, d1y, d1z;
        dir(entries[k0], d1x, d1y, d1z);
        const double d0x = d1x, d0y = d1y, d0z = d1z;
        double ox = 0.0, oy = 0.0, oz = 0.0;
        for (uint32_t k = k0 + 1; k < k1; ++k)
        {
            double d2x, d2y, d2z;
            dir(entries[k], d2x, d2y, d2z);
            // cross(d2, d1)
            ox = ox + (d2y * d1z - d2z * d1y);
            oy = oy + (d2z * d1x - d2x * d1z);
            oz = oz + (d2x * d1y - d2y * d1x);
            d1x = d2x, d1y = d2y, d1z = d2z;
        }
        // closing term cross(d0, d_last), then unit: times 1/|.|
        ox = ox + (d0y * d1z - d0z * d1y);
        oy = oy + (d0z * d1x - d0x * d1z);
        oz = oz + (d0x * d1y - d0y * d1x);
        const double inv = 1.0 / sqrt(ox * ox + oy * oy + oz * oz);
        normal_out[3 * s + 0] = ox * inv;
        normal_out[3 * s + 1] = oy * inv;
        normal_out[3 * s + 2] = oz * inv;
    }
}

// ---------------------------------------------------------------------------------------
int compute_line_geom(const pvl_mesh *m, const double *pos, double tol, LineGeom **out, unsigned n_lines, int slot = 0)
{
    LineGeom *g = (LineGeom *)scratch(slot, sizeof(LineGeom) * (size_t)(n_lines ? n_lines : 1));
    if (!g)
        return PVL_ERR_NOMEM;
    if (n_lines)
    {
        line_geom_kernel<<<(n_lines + 255) / 256, 256, 0, stream()>>>(n_lines, m->d_lines, pos, tol, g);
        PVL_HIP(hipGetLastError());
    }
    *out = g;
    return PVL_OK;
}

int compute_line_geom(const pvl_mesh *m, const double *pos, double tol, LineGeom **out)
{
    return compute_line_geom(m, pos, tol, out, m->n_lines, 0);
}

int check_common(const pvl_mesh *m, double tol, int precision)
{
    if (!m)
    {
        set_error("null mesh");
        return PVL_ERR_ARG;
    }
    if (precision != PVL_FP64 && precision != PVL_FP32 && precision != PVL_FP64_REF_FORM)
    {
        set_error("unknown precision %d", precision);
        return PVL_ERR_ARG;
    }
    (void)tol;
    return ensure_init();
}

template <bool NORMAL>
int launch_surface(const pvl_mesh *m, double tol, const double *pos, unsigned n_cpts, const double *cpts,
                   const double *normals, double *out, int precision)
{
    if (n_cpts == 0 || m->n_surfaces == 0)
        return PVL_OK;
    LineGeom *g;
    if (int st = compute_line_geom(m, pos, tol, &g))
        return st;
    constexpr int spw = 8;
    const dim3 grid(NORMAL ? (m->n_asm_runs + 3) / 4 : (m->n_surfaces + 4 * spw - 1) / (4 * spw),
                    (n_cpts + kCptTile - 1) / kCptTile);
    if (grid.y > 65535u)
    {
        set_error("too many control points (%u) for one launch", n_cpts);
        return PVL_ERR_ARG;
    }
    ProfScope prof(NORMAL ? "induction_matrix3" : "induction_matrix", (double)n_cpts * (double)m->n_lines);
    dispatch_precision(precision, [&](auto P) {
        if constexpr (NORMAL)
            assembly_kernel<decltype(P)::value><<<grid, kBlock, 0, stream()>>>(
                n_cpts, m->n_surfaces, m->n_asm_runs, m->d_asm_off, m->d_asm_grp, m->d_asm, g, cpts, normals, out,
                tol);
        else
            surface_induction_kernel<NORMAL, decltype(P)::value, spw><<<grid, kBlock, 0, stream()>>>(
                n_cpts, m->n_surfaces, m->d_offsets, m->d_entries, g, cpts, normals, out, tol);
    });
    PVL_HIP(hipGetLastError());
    return PVL_OK;
}

// ---------------------------------------------------------------------------------------
// Segment chains (the wake's self-induction).  Prologue: each segment's end node, unit
// direction in the chain's direction (three true divisions, the reference's line prologue;
// direction 0 below tol as line_geom_kernel) and circulation, signed for the direction.
__global__ void __launch_bounds__(256) chain_segment_kernel(unsigned n_seg, const uint32_t *__restrict__ seg_ab,
                                                            const uint32_t *__restrict__ seg_line,
                                                            const double *__restrict__ nodes,
                                                            const double *__restrict__ gamma, unsigned n_active,
                                                            double tol, SegRec *__restrict__ out)
{
    const unsigned j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n_seg)
        return;
    const uint32_t a = seg_ab[2 * j], b = seg_ab[2 * j + 1], ln = seg_line[j];
    const double ax = nodes[3 * a + 0], ay = nodes[3 * a + 1], az = nodes[3 * a + 2];
    SegRec r;
    r.nx = nodes[3 * b + 0], r.ny = nodes[3 * b + 1], r.nz = nodes[3 * b + 2];
    const double dx = r.nx - ax, dy = r.ny - ay, dz = r.nz - az;
    r.len = sqrt(dx * dx + dy * dy + dz * dz);
    r.ex = dx / r.len;
    r.ey = dy / r.len;
    r.ez = dz / r.len;
    if (r.len < tol)
        r.ex = r.ey = r.ez = r.len = 0.0;
    const uint32_t l = ln & kInvalidId;
    double g = l < n_active ? gamma[l] : 0.0;
    g = (ln & kReversed) ? -g : g;
    r.gamma = g;
    const double l2 = r.len * r.len;
    constexpr double fa[kFarTerms] = {kFar1, kFar2, kFar3, kFar4, kFar5, kFar6, kFar7};
    double q = r.len * g;
    r.c[0] = q;
#pragma unroll
    for (int k = 0; k < kFarTerms; ++k)
    {
        q = q * l2;
        r.c[k + 1] = fa[k] * q;
    }
    out[j] = r;
}

// Segments of a piece that are active at cr filled rows.
__device__ __forceinline__ unsigned active_segments(const ChainPiece &pc, unsigned cr)
{
    if (!pc.row1)
        return pc.n_seg;
    const unsigned avail = cr - (pc.row1 - 1);
    return pc.n_seg < avail ? pc.n_seg : avail;
}

// Axis-aligned box of the wave's points (64 PPL of them), the same in every lane.
struct PointBox
{
    double lo[3], hi[3];
};
__device__ __forceinline__ double wave_uniform(double v)
{
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)u);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(u >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
template <int PPL>
__device__ __forceinline__ PointBox point_box(const double (&px)[PPL], const double (&py)[PPL], const double (&pz)[PPL])
{
    PointBox b;
    const double *c[3] = {px, py, pz};
#pragma unroll
    for (int k = 0; k < 3; ++k)
    {
        double lo = c[k][0], hi = c[k][0];
#pragma unroll
        for (int i = 1; i < PPL; ++i)
            lo = fmin(lo, c[k][i]), hi = fmax(hi, c[k][i]);
        for (int off = 32; off > 0; off >>= 1)
        {
            lo = fmin(lo, __shfl_xor(lo, off));
            hi = fmax(hi, __shfl_xor(hi, off));
        }
        b.lo[k] = wave_uniform(lo), b.hi[k] = wave_uniform(hi);
    }
    return b;
}
// True when every point of the box is at least s.reach from the lines' box: the far form then
// holds for every pair (SegBox::reach).  False for anything that is not a number.
__device__ __forceinline__ bool box_far(const PointBox &b, const SegBox &s)
{
    double d2 = 0.0;
#pragma unroll
    for (int k = 0; k < 3; ++k)
    {
        const double g = fmax(fmax(s.lo[k] - b.hi[k], b.lo[k] - s.hi[k]), 0.0);
        d2 = fma(g, g, d2);
    }
    return __builtin_amdgcn_ballot_w64(d2 >= s.reach * s.reach) != 0;
}

// v += w K of a segment in the far form (induction_core.hpp) for a lane's PPL points, a = p - r1
// before and p - r2 after; step by step over the points, whose chains of dependent operations
// then fill each other's latency.
template <int PPL>
__device__ __forceinline__ void far_add(const SegRec &r, const double (&px)[PPL], const double (&py)[PPL],
                                        const double (&pz)[PPL], double (&ax)[PPL], double (&ay)[PPL],
                                        double (&az)[PPL], double tol2, double (&vx)[PPL], double (&vy)[PPL],
                                        double (&vz)[PPL])
{
    double bx[PPL], by[PPL], bz[PPL], q[PPL], cx[PPL], cy[PPL], cz[PPL], h2[PPL], u[PPL], f[PPL];
#pragma unroll
    for (int i = 0; i < PPL; ++i)
    {
        bx[i] = px[i] - r.nx, by[i] = py[i] - r.ny, bz[i] = pz[i] - r.nz;
        q[i] = fma(ax[i], bx[i], fma(ay[i], by[i], az[i] * bz[i]));
    }
#pragma unroll
    for (int i = 0; i < PPL; ++i)
    {
        cx[i] = fma(ay[i], r.ez, -(az[i] * r.ey));
        cy[i] = fma(az[i], r.ex, -(ax[i] * r.ez));
        cz[i] = fma(ax[i], r.ey, -(ay[i] * r.ex));
        ax[i] = bx[i], ay[i] = by[i], az[i] = bz[i];
    }
#pragma unroll
    for (int i = 0; i < PPL; ++i)
    {
        q[i] = far_rcp(q[i]);
        h2[i] = fma(cx[i], cx[i], fma(cy[i], cy[i], cz[i] * cz[i]));
    }
#pragma unroll
    for (int i = 0; i < PPL; ++i)
        u[i] = q[i] * (q[i] * h2[i]), f[i] = r.c[kFarTerms];
#pragma unroll
    for (int k = kFarTerms - 1; k >= 0; --k)
#pragma unroll
        for (int i = 0; i < PPL; ++i)
            f[i] = fma(f[i], u[i], r.c[k]);
#pragma unroll
    for (int i = 0; i < PPL; ++i)
    {
        // the angle's sign: K = -(dr1 x e) angle / h
        const double wm = h2[i] < tol2 ? 0.0 : -(q[i] * f[i]);
        vx[i] = fma(wm, cx[i], vx[i]);
        vy[i] = fma(wm, cy[i], vy[i]);
        vz[i] = fma(wm, cz[i], vz[i]);
    }
}

// Head of each piece: its active segments, start and bounds; one lane per segment.
__global__ void __launch_bounds__(256) chain_head_kernel(unsigned n_pieces, const ChainPiece *__restrict__ pieces,
                                                           unsigned cr, const double *__restrict__ nodes,
                                                           const SegRec *__restrict__ segs, ChainHead *__restrict__ out,
                                                           unsigned *__restrict__ queue)
{
    if (blockIdx.x == 0 && threadIdx.x == 0)
        *queue = 0u;
    constexpr unsigned L = kChainPiece;
    static_assert((L & (L - 1)) == 0 && L <= 64, "the pieces of a wave");
    const unsigned k = blockIdx.x * (256 / L) + threadIdx.x / L, lane = threadIdx.x % L;
    if (k >= n_pieces)
        return;
    const ChainPiece pc = pieces[k];
    const unsigned n = active_segments(pc, cr);
    ChainHead hd;
    hd.first_seg = pc.first_seg, hd.n_seg = n;
    SegBox &b = hd.box;
    b.reach = 0.0;
#pragma unroll
    for (int c = 0; c < 3; ++c)
        hd.start[c] = b.lo[c] = b.hi[c] = nodes[3 * pc.start_node + c];
    if (lane < n)
    {
        const SegRec &r = segs[pc.first_seg + lane];
        const double e[3] = {r.nx, r.ny, r.nz};
#pragma unroll
        for (int c = 0; c < 3; ++c)
            b.lo[c] = fmin(b.lo[c], e[c]), b.hi[c] = fmax(b.hi[c], e[c]);
        b.reach = far_reach(r.len);
    }
    for (int off = L / 2; off > 0; off >>= 1)
    {
#pragma unroll
        for (int c = 0; c < 3; ++c)
        {
            b.lo[c] = fmin(b.lo[c], __shfl_xor(b.lo[c], off, L));
            b.hi[c] = fmax(b.hi[c], __shfl_xor(b.hi[c], off, L));
        }
        b.reach = fmax(b.reach, __shfl_xor(b.reach, off, L));
    }
    if (lane == 0)
        out[k] = hd;
}

// Waits until the far form's part of a record is in scalar registers (SegRec::len is not part
// of it), with nothing moved across.
__device__ __forceinline__ void arrived(const SegRec &r)
{
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::"s"(r.nx), "s"(r.ny), "s"(r.nz), "s"(r.ex), "s"(r.ey), "s"(r.ez), "s"(r.c[0]), "s"(r.c[1]),
                 "s"(r.c[2]), "s"(r.c[3]), "s"(r.c[4]), "s"(r.c[5]), "s"(r.c[6]), "s"(r.c[7]));
}

// A lane has PPL points, a wave 64 PPL.  FP64 and the reference form: a workgroup has four times that
// and its waves walk the same pieces, a chunk of them (every n_chunks-th piece, so that the pieces near
// the points are spread over the chunks) per item, so that a segment's record is read into the scalar
// cache once for four waves (with a piece per wave the records' latency held the kernel at twice
// its issue time); sums are written per chunk, with no exchange between waves.
// Bound by VALU issue: 37 slots per pair in the far form (induction_core.hpp), 73 in the general
// one.  A piece whose box is far enough from the box of the wave's points takes the far form for
// all its segments without any test inside the loop (93 to 95 % of the pairs of a 400-row wake);
// the end node's dr = p - r is the next segment's dr1.  Work items are (point block, piece chunk)
// pairs, taken from a grid that may be smaller than their number (side stream).
// FP32 keeps its single-precision angle at every distance (the far form is more exact, but would move
// the results by the mode's own rounding), 68 slots for every pair, which hide the records' latency:
// there the four waves share the points and take every fourth piece of the chunk, and add their sums
// in LDS (chain_split).  Waves on one record wait and issue together; a free-wake step of 1,024 /
// 2,048 / 2,048 surfaces and 25,600 / 19,200 / 32,000 wake panels took 2.43 / 1.81 / 4.18 ms with the
// pieces shared and takes 2.36 / 1.63 / 3.74 ms.
constexpr bool chain_split(int precision) { return precision == PVL_FP32; }
template <int PREC, int PPL>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(PREC == PVL_FP32 ? 8 : 4)))
    chain_velocity_kernel(unsigned n_pts, const double *__restrict__ pts, const ChainHead *__restrict__ heads,
                          unsigned n_pieces, const SegRec *__restrict__ segs,
                          unsigned n_chunks, double *__restrict__ partial, double tol, unsigned pblocks,
                          unsigned n_items, unsigned *__restrict__ queue)
{
    constexpr bool SPLIT = chain_split(PREC);
    const unsigned w = wave_id(), lane = lane_id();
    const double tol2 = tol * tol;
    __shared__ unsigned s_item;
    for (;;)
    {
        if (threadIdx.x == 0)
            s_item = atomicAdd(queue, 1u);
        __syncthreads();
        const unsigned item = __builtin_amdgcn_readfirstlane(s_item);
        __syncthreads(); // s_item is rewritten for the next item
        if (item >= n_items)
            return;
        const unsigned chunk = item / pblocks;
        const unsigned pb = item - chunk * pblocks;
        const unsigned w0 = (SPLIT ? pb : pb * 4 + w) * (kWave * PPL);
        if (w0 >= n_pts)
            continue;
        const unsigned p0 = w0 + lane;
        double px[PPL], py[PPL], pz[PPL], vx[PPL], vy[PPL], vz[PPL];
#pragma unroll
        for (int i = 0; i < PPL; ++i)
        {
            const unsigned p = p0 + i * kWave;
            const unsigned pc = p < n_pts ? p : n_pts - 1;
            px[i] = pts[3 * pc + 0], py[i] = pts[3 * pc + 1], pz[i] = pts[3 * pc + 2];
            vx[i] = 0.0, vy[i] = 0.0, vz[i] = 0.0;
        }
        PointBox box;
        if constexpr (PREC == PVL_FP64)
            box = point_box<PPL>(px, py, pz);
        for (unsigned k = SPLIT ? 4 * chunk + w : chunk; k < n_pieces; k += (SPLIT ? 4 : 1) * n_chunks)
        {
            const ChainHead &hd = heads[k];
            const unsigned n = hd.n_seg;
            const double sx = hd.start[0], sy = hd.start[1], sz = hd.start[2];
            double ax[PPL], ay[PPL], az[PPL], aq[PPL]; // aq (|p - node|^2) only for the reference form
#pragma unroll
            for (int i = 0; i < PPL; ++i)
            {
                ax[i] = px[i] - sx, ay[i] = py[i] - sy, az[i] = pz[i] - sz;
                aq[i] = PREC == PVL_FP64_REF_FORM ? ax[i] * ax[i] + ay[i] * ay[i] + az[i] * az[i] : 0.0;
            }
            const SegRec *sg = segs + hd.first_seg;
            // one segment in the general form, and on to its end node
            struct Seg
            {
                double nx, ny, nz, ex, ey, ez, len, gamma;
            };
            auto load = [&](unsigned j) {
                return Seg{sg[j].nx, sg[j].ny, sg[j].nz, sg[j].ex, sg[j].ey, sg[j].ez, sg[j].len, sg[j].gamma};
            };
            auto general = [&](const Seg &r, AtanTable table) {
                const double nx = r.nx, ny = r.ny, nz = r.nz;
                const double ex = r.ex, ey = r.ey, ez = r.ez, len = r.len, gamma = r.gamma;
#pragma unroll
                for (int i = 0; i < PPL; ++i)
                {
                    bool cut;
                    if constexpr (PREC == PVL_FP64_REF_FORM)
                    {
                        const double bx = px[i] - nx, by = py[i] - ny, bz = pz[i] - nz;
                        const double bq = bx * bx + by * by + bz * bz;
                        const double m =
                            pair_m<PREC>(ex, ey, ez, len, ax[i], ay[i], az[i], aq[i], bx, by, bz, bq, tol, tol2, cut);
                        const double kx = cut ? 0.0 : (ay[i] * ez - az[i] * ey) * m;
                        const double ky = cut ? 0.0 : (az[i] * ex - ax[i] * ez) * m;
                        const double kz = cut ? 0.0 : (ax[i] * ey - ay[i] * ex) * m;
                        vx[i] = vx[i] + gamma * kx;
                        vy[i] = vy[i] + gamma * ky;
                        vz[i] = vz[i] + gamma * kz;
                        aq[i] = bq;
                        ax[i] = bx, ay[i] = by, az[i] = bz;
                    }
                    else
                    {
                        double cx, cy, cz;
                        const double m =
                            cross_m<PREC, 2>(ex, ey, ez, len, ax[i], ay[i], az[i], tol2, cx, cy, cz, cut, table);
                        const double wm = cut ? 0.0 : gamma * m;
                        vx[i] = fma(wm, cx, vx[i]);
                        vy[i] = fma(wm, cy, vy[i]);
                        vz[i] = fma(wm, cz, vz[i]);
                        ax[i] = px[i] - nx, ay[i] = py[i] - ny, az[i] = pz[i] - nz;
                        if constexpr (PREC == PVL_FP64)
                            __builtin_amdgcn_sched_barrier(0); // one point after the other: fewer registers
                    }
                }
            };
            bool far = false;
            if constexpr (PREC == PVL_FP64)
                far = box_far(box, hd.box);
            if (far)
            {
                // the next segment's record is on its way to scalar registers while this one is
                // worked on (scalar loads return out of order, so a wait is for all of them: the
                // one for the next record stands at the end of this one's work)
                auto work = [&](const SegRec &r) { far_add<PPL>(r, px, py, pz, ax, ay, az, tol2, vx, vy, vz); };
                SegRec r = sg[0], q;
                arrived(r);
                unsigned j = 0;
                for (; j + 1 < n; j += 2)
                {
                    q = sg[j + 1];
                    __builtin_amdgcn_sched_barrier(0);
                    work(r);
                    arrived(q);
                    r = sg[j + 2 < n ? j + 2 : j];
                    __builtin_amdgcn_sched_barrier(0);
                    work(q);
                    arrived(r);
                }
                if (j < n)
                    work(r);
            }
            else if constexpr (PREC == PVL_FP32)
            {
                // every pair comes here: the next record on its way as above
                Seg r = load(0);
                for (unsigned j = 0; j < n; ++j)
                {
                    const Seg q = load(j + 1 < n ? j + 1 : j);
                    __builtin_amdgcn_sched_barrier(0);
                    general(r, nullptr);
                    __builtin_amdgcn_sched_barrier(0);
                    asm volatile("" ::"s"(q.nx), "s"(q.ny), "s"(q.nz), "s"(q.ex), "s"(q.ey), "s"(q.ez), "s"(q.len),
                                 "s"(q.gamma));
                    r = q;
                }
            }
            else
            {
                AtanTable table = PREC == PVL_FP64 ? atan_table() : nullptr;
                for (unsigned j = 0; j < n; ++j)
                    general(load(j), table);
            }
        }
        if constexpr (SPLIT)
        {
            // the waves' sums in wave order (red is next written after the next item's barriers)
            __shared__ double red[3][3][kWave * PPL];
            if (w > 0)
            {
#pragma unroll
                for (int i = 0; i < PPL; ++i)
                {
                    red[w - 1][0][i * kWave + lane] = vx[i];
                    red[w - 1][1][i * kWave + lane] = vy[i];
                    red[w - 1][2][i * kWave + lane] = vz[i];
                }
            }
            __syncthreads();
            if (w > 0)
                continue;
#pragma unroll
            for (int i = 0; i < PPL; ++i)
#pragma unroll
                for (int u = 0; u < 3; ++u)
                {
                    vx[i] = vx[i] + red[u][0][i * kWave + lane];
                    vy[i] = vy[i] + red[u][1][i * kWave + lane];
                    vz[i] = vz[i] + red[u][2][i * kWave + lane];
                }
        }
#pragma unroll
        for (int i = 0; i < PPL; ++i)
        {
            const unsigned p = p0 + i * kWave;
            if (p < n_pts)
            {
                double *dst = partial + ((size_t)chunk * n_pts + p) * 3;
                dst[0] = vx[i], dst[1] = vy[i], dst[2] = vz[i];
            }
        }
    }
}

} // namespace

namespace pvl
{

// Point-velocity sum over the first n_active lines of the mesh (all lines for the public
// entry point; the wake passes the prefix of lines its filled rows use -- the other lines
// carry zero circulation).
// Chunking: aim for 4,096 workgroups of two points per lane while keeping >= 64 lines per wave.  Half
// of that left the last round of waves half empty (30,000 points: 11 % more time); twice of
// it gains 3 % there and costs 1 % in a wake of 3,200 panels, in partial sums.  Where the partial sums and the line records of such a
// plan would not fit pvl_point_velocity_noalloc's fixed scratch, the chunk count of 2,048 workgroups
// of one point per lane, which is half as many.  One rule for both entry points: same sums.
static bool self_site(const char *prof_name) { return std::strcmp(prof_name, "wake_self_velocity") == 0; }

static void plan_chunks(unsigned n_pts, unsigned n_active, unsigned *n_chunks_out, unsigned *lpc_out)
{
    const auto plan = [&](unsigned groups, unsigned points, unsigned *lpc) {
        const unsigned pblocks = (n_pts + points - 1) / points;
        unsigned n_chunks = (groups + pblocks - 1) / pblocks;
        const unsigned max_chunks = (n_active + 255) / 256;
        if (n_chunks > max_chunks)
            n_chunks = max_chunks;
        if (n_chunks < 1)
            n_chunks = 1;
        if (n_chunks > 65535u)
            n_chunks = 65535u;
        *lpc = (n_active + n_chunks - 1) / n_chunks;
        return (n_active + *lpc - 1) / *lpc;
    };
    *n_chunks_out = plan(4096, 2 * kWave, lpc_out);
    if (point_velocity_scratch(n_pts, n_active, *n_chunks_out) > PVL_NOALLOC_SCRATCH_BYTES)
        *n_chunks_out = plan(2048, kWave, lpc_out);
}

// Points per lane: two where items of 128 points give every SIMD four waves (1,024 workgroups).  FP64 with
// one / two points per lane: 300 points and 100 lines 21 / 26 us, 2,054 and 960 33 / 44, 28,077 and 410
// 45 / 50, 1,000 and 7,300 41 / 58; 100 points and 20,100 lines 42 / 36.
static int point_velocity_ppl(unsigned n_pts, unsigned n_chunks)
{
    return (unsigned long long)((n_pts + 2 * kWave - 1) / (2 * kWave)) * n_chunks >= 1024 ? 2 : 1;
}

unsigned point_velocity_chunks(unsigned n_pts, unsigned n_active)
{
    unsigned nc, lpc;
    plan_chunks(n_pts, n_active, &nc, &lpc);
    return nc;
}

size_t line_geom_bytes(unsigned n_lines) { return sizeof(LineGeom) * (size_t)(n_lines ? n_lines : 1); }

int point_velocity_partials(const pvl_mesh *m, double tol, const double *pos, const double *circ, unsigned n_pts,
                            const double *pts, int precision, unsigned n_active, const char *prof_name,
                            hipStream_t s, void *geom, double *gamma, double *partial, unsigned max_groups)
{
    const LineGeom *g = (const LineGeom *)geom;
    line_record_kernel<<<(n_active + 255) / 256, 256, 0, s>>>(n_active, m->d_lines, pos, tol, m->d_line_offsets,
                                                              m->d_line_surfs, circ, (LineGeom *)geom, gamma);
    PVL_HIP(hipGetLastError());
    unsigned n_chunks, lpc;
    plan_chunks(n_pts, n_active, &n_chunks, &lpc);
    const unsigned points = kWave * point_velocity_ppl(n_pts, n_chunks);
    const unsigned pblocks = (n_pts + points - 1) / points;
    const unsigned n_items = pblocks * n_chunks;
    const unsigned grid = max_groups && max_groups < n_items ? max_groups : n_items;
    ProfScope prof(prof_name, (double)n_pts * (double)n_active, s);
    dispatch_precision(precision, [&](auto P) {
        const auto launch = [&](auto site, auto ppl) {
            point_velocity_kernel<decltype(P)::value, decltype(site)::value, decltype(ppl)::value>
                <<<grid, kBlock, 0, s>>>(n_pts, pts, n_active, g, gamma, lpc, partial, tol, pblocks, n_items);
        };
        const auto at = [&](auto ppl) {
            if (self_site(prof_name))
                launch(std::integral_constant<int, 1>{}, ppl);
            else
                launch(std::integral_constant<int, 0>{}, ppl);
        };
        if (points == kWave)
            at(std::integral_constant<int, 1>{});
        else
            at(std::integral_constant<int, 2>{});
    });
    PVL_HIP(hipGetLastError());
    return PVL_OK;
}

int line_circulations(const pvl_mesh *m, unsigned n_active, const double *circ, double *gamma, hipStream_t s)
{
    if (n_active == 0)
        return PVL_OK;
    line_circulation_kernel<<<(n_active + 255) / 256, 256, 0, s>>>(n_active, m->d_line_offsets, m->d_line_surfs,
                                                                     circ, gamma);
    PVL_HIP(hipGetLastError());
    return PVL_OK;
}

int chain_segments(unsigned n_seg, const uint32_t *seg_ab, const uint32_t *seg_line, const double *nodes,
                   const double *gamma, unsigned n_active_lines, double tol, SegRec *out, hipStream_t s)
{
    if (n_seg == 0)
        return PVL_OK;
    chain_segment_kernel<<<(n_seg + 255) / 256, 256, 0, s>>>(n_seg, seg_ab, seg_line, nodes, gamma, n_active_lines,
                                                             tol, out);
    PVL_HIP(hipGetLastError());
    return PVL_OK;
}

constexpr int kChainPPL = 2;
constexpr unsigned kChainItems = 4608;
// points per workgroup
constexpr unsigned chain_points(int precision) { return (chain_split(precision) ? 1 : 4) * kWave * kChainPPL; }

unsigned chain_velocity_chunks(unsigned n_pts, unsigned n_pieces, int precision)
{
    const unsigned points = chain_points(precision), pblocks = (n_pts + points - 1) / points;
    const unsigned max_chunks = std::max(1u, (n_pieces + 7) / 8);
    if (chain_split(precision)) // 2,048 and 7,680 items: up to 4 % more time in the sizes above
        return std::min(max_chunks, (3840u + pblocks - 1) / pblocks);
    // kChainItems work items (six per workgroup of the side stream: the last ones claimed are
    // the kernel's tail), a chunk of at least 8 pieces each.  More items cost more partial sums
    // (24 bytes per point and chunk, written and read once).
    return std::min(max_chunks, std::max(1u, kChainItems / pblocks));
}

int chain_velocity_partials(unsigned n_pts, const double *pts, const double *nodes, const ChainPiece *pieces,
                            unsigned n_pieces, unsigned cr, const SegRec *segs, ChainHead *heads, int precision, double tol, double work, hipStream_t s, double *partial,
                            unsigned max_groups)
{
    const unsigned n_chunks = chain_velocity_chunks(n_pts, n_pieces, precision);
    const unsigned points = chain_points(precision), pblocks = (n_pts + points - 1) / points;
    const unsigned n_items = pblocks * n_chunks;
    const unsigned grid = max_groups && max_groups < n_items ? max_groups : n_items;
    unsigned *queue = (unsigned *)(heads + n_pieces); // one spare head
    chain_head_kernel<<<(n_pieces * kChainPiece + 255) / 256, 256, 0, s>>>(n_pieces, pieces, cr, nodes, segs, heads, queue);
    PVL_HIP(hipGetLastError());
    ProfScope prof("wake_self_velocity", work, s);
    dispatch_precision(precision, [&](auto P) {
        chain_velocity_kernel<decltype(P)::value, kChainPPL><<<grid, kBlock, 0, s>>>(
            n_pts, pts, heads, n_pieces, segs, n_chunks, partial, tol, pblocks, n_items, queue);
    });
    PVL_HIP(hipGetLastError());
    return PVL_OK;
}

int point_velocity_reduce(unsigned n_pts, unsigned n_chunks, const double *partial, double *out, int accumulate,
                          hipStream_t s)
{
    chunk_reduce_kernel<<<(3 * n_pts + 255) / 256, 256, 0, s>>>(n_pts, n_chunks, partial, out, accumulate);
    PVL_HIP(hipGetLastError());
    return PVL_OK;
}

int point_velocity_impl(const pvl_mesh *m, double tol, const double *pos, const double *circ, unsigned n_pts,
                        const double *pts, double *out, int accumulate, int precision, unsigned n_active,
                        const char *prof_name)
{
    if (n_pts == 0)
        return PVL_OK;
    if (n_active > m->n_lines)
        n_active = m->n_lines;
    if (n_active == 0)
    {
        if (!accumulate)
            if (int st = device_fill32(out, 0u, sizeof(double) * 3 * n_pts))
                return st;
        return PVL_OK;
    }
    const unsigned n_chunks = point_velocity_chunks(n_pts, n_active);
    void *g = scratch(0, line_geom_bytes(n_active));
    double *gamma = (double *)scratch(1, sizeof(double) * n_active);
    double *partial = (double *)scratch(2, sizeof(double) * 3 * (size_t)n_pts * n_chunks);
    if (!g || !gamma || !partial)
        return PVL_ERR_NOMEM;
    if (int st = point_velocity_partials(m, tol, pos, circ, n_pts, pts, precision, n_active, prof_name, stream(), g,
                                         gamma, partial, 0))
        return st;
    return point_velocity_reduce(n_pts, n_chunks, partial, out, accumulate, stream());
}

} // namespace pvl

extern "C" {

int pvl_induction_matrix3(const pvl_mesh *m, double tol, const double *pos, unsigned n_cpts, const double *cpts,
                          const double *normals, double *out, int precision)
{
    PVL_API_LOCK;
    if (int st = check_common(m, tol, precision))
        return st;
    return launch_surface<true>(m, tol, pos, n_cpts, cpts, normals, out, precision);
}

int pvl_induction_matrix(const pvl_mesh *m, double tol, const double *pos, unsigned n_cpts, const double *cpts,
                         double *out, int precision)
{
    PVL_API_LOCK;
    if (int st = check_common(m, tol, precision))
        return st;
    return launch_surface<false>(m, tol, pos, n_cpts, cpts, nullptr, out, precision);
}

int pvl_line_induction_matrix(const pvl_mesh *m, double tol, const double *pos, unsigned n_cpts, const double *cpts,
                              double *out, int precision)
{
    PVL_API_LOCK;
    if (int st = check_common(m, tol, precision))
        return st;
    if (n_cpts == 0 || m->n_lines == 0)
        return PVL_OK;
    LineGeom *g;
    if (int st = compute_line_geom(m, pos, tol, &g))
        return st;
    constexpr int lpw = 8;
    const dim3 grid((m->n_lines + 4 * lpw - 1) / (4 * lpw), (n_cpts + kCptTile - 1) / kCptTile);
    if (grid.y > 65535u)
    {
        set_error("too many control points (%u) for one launch", n_cpts);
        return PVL_ERR_ARG;
    }
    ProfScope prof("line_induction_matrix", (double)n_cpts * (double)m->n_lines);
    dispatch_precision(precision, [&](auto P) {
        line_induction_kernel<decltype(P)::value, lpw>
            <<<grid, kBlock, 0, stream()>>>(n_cpts, m->n_lines, g, cpts, out, tol);
    });
    PVL_HIP(hipGetLastError());
    return PVL_OK;
}

int pvl_point_velocity(const pvl_mesh *m, double tol, const double *pos, const double *circ, unsigned n_pts,
                       const double *pts, double *out, int accumulate, int precision)
{
    PVL_API_LOCK;
    if (int st = check_common(m, tol, precision))
        return st;
    return pvl::point_velocity_impl(m, tol, pos, circ, n_pts, pts, out, accumulate, precision, m->n_lines);
}

int pvl_surface_normal(const pvl_mesh *m, const double *pos, double *out)
{
    PVL_API_LOCK;
    if (int st = check_common(m, 0.0, PVL_FP64))
        return st;
    if (m->n_surfaces == 0)
        return PVL_OK;
    surface_geometry_kernel<<<(m->n_surfaces + 255) / 256, 256, 0, stream()>>>(
        m->n_surfaces, m->d_offsets, m->d_entries, m->d_lines, pos, out, nullptr);
    PVL_HIP(hipGetLastError());
    return PVL_OK;
}

int pvl_surface_center(const pvl_mesh *m, const double *pos, double *out)
{
    PVL_API_LOCK;
    if (int st = check_common(m, 0.0, PVL_FP64))
        return st;
    if (m->n_surfaces == 0)
        return PVL_OK;
    surface_geometry_kernel<<<(m->n_surfaces + 255) / 256, 256, 0, stream()>>>(
        m->n_surfaces, m->d_offsets, m->d_entries, m->d_lines, pos, nullptr, out);
    PVL_HIP(hipGetLastError());
    return PVL_OK;
}

// Host-buffer forms: stage inputs, run, copy back, synchronise.
static int stage(const pvl_mesh *m, const double *pos, unsigned n_cpts, const double *cpts, const double *normals,
                 double **d_pos, double **d_cpts, double **d_norm)
{
    const size_t pb = sizeof(double) * 3 * (size_t)m->n_points, cb = sizeof(double) * 3 * (size_t)n_cpts;
    *d_pos = (double *)scratch(8, pb ? pb : 8);
    *d_cpts = (double *)scratch(9, cb ? cb : 8);
    *d_norm = normals ? (double *)scratch(10, cb ? cb : 8) : nullptr;
    if (!*d_pos || !*d_cpts || (normals && !*d_norm))
        return PVL_ERR_NOMEM;
    PVL_HIP(hipMemcpyAsync(*d_pos, pos, pb, hipMemcpyHostToDevice, stream()));
    PVL_HIP(hipMemcpyAsync(*d_cpts, cpts, cb, hipMemcpyHostToDevice, stream()));
    if (normals)
        PVL_HIP(hipMemcpyAsync(*d_norm, normals, cb, hipMemcpyHostToDevice, stream()));
    return PVL_OK;
}

static int unstage(double *out, const double *d_out, size_t bytes)
{
    PVL_HIP(hipMemcpyAsync(out, d_out, bytes, hipMemcpyDeviceToHost, stream()));
    PVL_HIP(hipStreamSynchronize(stream()));
    return PVL_OK;
}

int pvl_induction_matrix3_host(const pvl_mesh *m, double tol, const double *pos, unsigned n_cpts, const double *cpts,
                               const double *normals, double *out, int precision)
{
    PVL_API_LOCK;
    if (int st = check_common(m, tol, precision))
        return st;
    double *dp, *dc, *dn;
    if (int st = stage(m, pos, n_cpts, cpts, normals, &dp, &dc, &dn))
        return st;
    const size_t ob = sizeof(double) * (size_t)n_cpts * m->n_surfaces;
    double *d_out = (double *)scratch(11, ob ? ob : 8);
    if (!d_out)
        return PVL_ERR_NOMEM;
    if (int st = pvl_induction_matrix3(m, tol, dp, n_cpts, dc, dn, d_out, precision))
        return st;
    return unstage(out, d_out, ob);
}

int pvl_induction_matrix_host(const pvl_mesh *m, double tol, const double *pos, unsigned n_cpts, const double *cpts,
                              double *out, int precision)
{
    PVL_API_LOCK;
    if (int st = check_common(m, tol, precision))
        return st;
    double *dp, *dc, *dn;
    if (int st = stage(m, pos, n_cpts, cpts, nullptr, &dp, &dc, &dn))
        return st;
    const size_t ob = sizeof(double) * 3 * (size_t)n_cpts * m->n_surfaces;
    double *d_out = (double *)scratch(11, ob ? ob : 8);
    if (!d_out)
        return PVL_ERR_NOMEM;
    if (int st = pvl_induction_matrix(m, tol, dp, n_cpts, dc, d_out, precision))
        return st;
    return unstage(out, d_out, ob);
}

int pvl_line_induction_matrix_host(const pvl_mesh *m, double tol, const double *pos, unsigned n_cpts,
                                   const double *cpts, double *out, int precision)
{
    PVL_API_LOCK;
    if (int st = check_common(m, tol, precision))
        return st;
    double *dp, *dc, *dn;
    if (int st = stage(m, pos, n_cpts, cpts, nullptr, &dp, &dc, &dn))
        return st;
    const size_t ob = sizeof(double) * 3 * (size_t)n_cpts * m->n_lines;
    double *d_out = (double *)scratch(11, ob ? ob : 8);
    if (!d_out)
        return PVL_ERR_NOMEM;
    if (int st = pvl_line_induction_matrix(m, tol, dp, n_cpts, dc, d_out, precision))
        return st;
    return unstage(out, d_out, ob);
}

} // extern "C"
