// Adjoint of the raymarch pass with respect to the float density volume and
// the absorption / ADSM-thickness / Kajiya-Kay-exponent parameters.
//
// The reference's march accumulates plain sums (volume_rendering.glsl:36-37,
// approximate_deep_shadows.glsl:28-33): no transmittance product runs along a
// ray, so every sample of one ray carries the same gradient weight -- for the
// primary ray dL/d(acc) (through the coverage a = lod * alpha * acc / iso),
// for the shadow ray dL/d(strands) (through (1-alpha)^(k * sum)).  The
// isosurface and surface choices are piecewise constant and carry none; the
// clamp to [0,1] passes gradient only strictly inside.
//
// Rays are re-walked from the ray set-up (nothing per sample is stored); the
// scatter of weight * trilinear weight is bound by the line requests of
// device atomics, and there are two ways to need fewer:
//   * cells: each sample goes to a corner-packed accumulator of 8 floats per
//     cell (the cell layout of the density: cell (i,j,k) for i,j,k in
//     [-1, n-1] holds texels i..i+1 x j..j+1 x k..k+1), 8 lanes adding the 8
//     corners of one sample in one 32-byte request, and neighbouring rays of
//     a pixel row in one cell add once.  A gather pass folds the cells into
//     the texel gradient;
//   * windows, for primary rays: the 64 rays of a wave march side by side, so
//     a wave adds a chunk of up to 16 steps into an LDS window over the
//     texels they touch there (float64: LDS float32 adds run a lane at a
//     time, ~200 cycles per wave instruction against ~11) and flushes the
//     window with one atomic per texel, rows of texels together.
// Windows pay only while the rays of a wave are close in texels and not all
// in one (window_scatter): at 128^3 / 512^2 / 256 steps 0.25 ms against 0.32
// in cells, at 128^2 pixels 0.87 against 0.25.  Shadow rays and LAO taps start at
// surfaces of different depths, so their samples share little and go to the
// cells (0.45 ms with the LAO taps in windows: each of their surfaces needs a
// window of its own).  Parameter gradients are reduced per block, then one
// atomic each.
#include "march.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

namespace vkhr {
namespace {

constexpr uint32_t kNoCell = 0xffffffffu;

struct AdjointArgs {
    RaymarchArgs f;
    const MarchRecord* record;
    const float4* d_rgba;
    // The texels the windows are flushed to, texel (x, y, z) at x + y * texel_row
    // + z * texel_slice: in the scratch with the cells' pitch, since rows and
    // slices of a power of two put a column's atomics on few memory channels.
    float* texel_grad;
    size_t texel_row, texel_slice;
    float* cell_grad;           // 8 floats per cell, (nx+1)(ny+1)(nz+1) cells
    float* d_params;            // absorption, ADSM thickness, shininess
    double* param_sums;         // their sums over the workgroups, added to d_params at the end (nullable: added at once)
    const float4* target;       // with a target: dL/d(rgba) = 2 (rgba - target), L = sum of squares
    float* loss;                // L is added here (with a target; nullable)
    int n_steps;                // iterations of the shader's float loop
    double ln_transmit;         // log(1 - alpha)
    double light_texel[3];
};

__device__ __forceinline__ bool in_range(const RaymarchArgs& f, const double x[3]) {
    return x[0] >= -1.0 && x[1] >= -1.0 && x[2] >= -1.0 && x[0] < double(f.nx) && x[1] < double(f.ny) &&
           x[2] < double(f.nz);
}

// A wave's window of texel gradients.  Any box of at most kWindow texels
// will do; rays that don't share one are grouped by cubes of kWindowSide
// (measured, us of the adjoint: 512 texels 361, 768 277, 1264 280, 1728 267,
// 2500 272).
constexpr int kWindow = 1728, kWindowSide = 12;
struct WindowLds {
    double window[kWindow];
};

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Minimum / maximum over the wave's 64 lanes (every lane calls it).
template <class Op>
__device__ __forceinline__ int wave_reduce(int v, Op op) {
    v = op(v, __builtin_amdgcn_update_dpp(v, v, 0xb1, 0xf, 0xf, false));    // quad: [1, 0, 3, 2]
    v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x4e, 0xf, 0xf, false));    // quad: [2, 3, 0, 1]
    v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x141, 0xf, 0xf, false));   // half row mirrored
    v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x140, 0xf, 0xf, false));   // row mirrored
    v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x142, 0xa, 0xf, false));   // row's last lane into the next
    v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x143, 0xc, 0xf, false));   // half's last lane into the next
    return __builtin_amdgcn_readlane(v, kWave - 1);
}
__device__ __forceinline__ int wave_min(int v) {
    return wave_reduce(v, [](int a, int b) { return a < b ? a : b; });
}
__device__ __forceinline__ int wave_max(int v) {
    return wave_reduce(v, [](int a, int b) { return a > b ? a : b; });
}

// The window while it is filled: its first texel and its strides.
struct Window {
    double* w;
    int origin[3];
    int row, slice;
};

// Adds c * (trilinear weights) at texel coordinate x, inside [-1, n)^3 and
// with its in-volume texels inside the window; a corner outside the volume
// adds 0 to the texel beside it.
__device__ __forceinline__ void window_add(const Window& win, const RaymarchArgs& f, const double x[3], float c) {
    const int n[3] = {f.nx, f.ny, f.nz};
    int at[3][2];
    float w[3][2];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const double fl = floor(x[a]);
        const float frac = float(x[a] - fl);
        const int i = int(fl);
        w[a][0] = i >= 0 ? 1.0f - frac : 0.0f;
        w[a][1] = i + 1 < n[a] ? frac : 0.0f;
        at[a][0] = max(i, 0) - win.origin[a];
        at[a][1] = min(i + 1, n[a] - 1) - win.origin[a];
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const int i = at[0][q & 1] + win.row * at[1][(q >> 1) & 1] + win.slice * at[2][q >> 2];
        const float v = c * (w[0][q & 1] * w[1][(q >> 1) & 1] * w[2][q >> 2]);
        __hip_atomic_fetch_add(&win.w[i], double(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
}

// Calls add(window) for every active lane, once, with a window that holds
// the lane's texels lo .. hi (inside the volume, at most kWindowSide along
// an axis), and flushes each window into the gradient.  Every lane of the
// wave calls it.
template <class Add>
__device__ __forceinline__ void scatter_windows(const AdjointArgs& a, WindowLds& lds, bool active, const int lo[3],
                                                const int hi[3], Add add) {
    const int lane = __lane_id();
    unsigned long long rest = __ballot(active);
    while (rest != 0ull) {
        bool in = (rest >> lane) & 1ull;
        Window win;
        win.w = lds.window;
        int end[3], size[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            win.origin[c] = wave_min(in ? lo[c] : 0x7fffffff);
            end[c] = wave_max(in ? hi[c] : -1);
            size[c] = end[c] - win.origin[c] + 1;
        }
        if (size[0] > kWindow || size[1] > kWindow || size[2] > kWindow || size[0] * size[1] > kWindow ||
            size[0] * size[1] * size[2] > kWindow) {
            // the lanes within a cube about the first one's texels
            const int leader = __ffsll((long long)rest) - 1;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const int l = __builtin_amdgcn_readlane(lo[c], leader), h = __builtin_amdgcn_readlane(hi[c], leader);
                win.origin[c] = max(win.origin[c], l - (kWindowSide - (h - l + 1)) / 2);
                end[c] = min(end[c], win.origin[c] + kWindowSide - 1);
                size[c] = end[c] - win.origin[c] + 1;
                in = in && lo[c] >= win.origin[c] && hi[c] <= end[c];
            }
        }
        win.row = size[0];
        win.slice = size[0] * size[1];
        const int count = win.slice * size[2];
        for (int e = lane; e < count; e += kWave) lds.window[e] = 0.0;
        wave_lds_sync();
        if (in) add(win);
        wave_lds_sync();
        const float inv_slice = 1.0f / float(win.slice), inv_row = 1.0f / float(win.row);
        for (int e = lane; e < count; e += kWave) {
            const float v = float(lds.window[e]);
            // (exact: e < kWindow, and e + 1/2 is a half away from every multiple)
            const int z = int((float(e) + 0.5f) * inv_slice), r = e - z * win.slice;
            const int y = int((float(r) + 0.5f) * inv_row), x = r - y * win.row;
            if (v != 0.0f)
                unsafeAtomicAdd(&a.texel_grad[size_t(win.origin[0] + x) + a.texel_row * size_t(win.origin[1] + y) +
                                              a.texel_slice * size_t(win.origin[2] + z)],
                                v);
        }
        wave_lds_sync();  // the window is cleared next
        rest &= ~__ballot(in);
    }
}

// One family of rays (primary or shadow): x(t) = x0 + t * dx for the
// sample parameters t of the shader's float loop, samples [0, n) of each
// active lane's ray, weight c per sample.  The loop runs to the wave's
// longest ray so that every lane takes part in the windows.
__device__ void scatter_rays(const AdjointArgs& a, WindowLds& lds, bool active, const double x0[3], const double dx[3],
                             int n, float c) {
    const RaymarchArgs& f = a.f;
    const float step = f.step_size;
    const int dims[3] = {f.nx, f.ny, f.nz};
    const int n_lane = active ? n : 0;
    const int n_wave = wave_max(n_lane);
    // samples per chunk: at most 8 texels along any axis, so that a lane's
    // texels fit in a window's cube
    double longest = 0.0;
    if (active) longest = fmax(fmax(fabs(dx[0]), fabs(dx[1])), fabs(dx[2])) * double(step);
    const int chunk = wave_min(longest > 0.5 ? max(int(fmin(8.0 / longest, 16.0)), 1) : 16);
    float t = 0.0f;  // the march state carried across chunks
    for (int i0 = 0; i0 < n_wave; i0 += chunk) {
        float last = t;
        for (int i = 1; i < chunk; ++i) last += step;
        const int i1 = min(i0 + chunk, n_lane);
        // the texels of the chunk's samples: between those of its ends
        bool in = i0 < i1;
        int lo[3], hi[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const double p = fma(double(t), dx[k], x0[k]), q = fma(double(last), dx[k], x0[k]);
            const double l = fmin(p, q), h = fmax(p, q);
            in = in && h >= -1.0 && l < double(dims[k]);
            lo[k] = max(in ? int(floor(fmax(l, -1.0))) : 0, 0);
            hi[k] = min(in ? int(floor(fmin(h, double(dims[k])))) + 1 : 0, dims[k] - 1);
        }
        scatter_windows(a, lds, in, lo, hi, [&](const Window& win) {
            float tt = t;
            for (int i = i0; i < i1; ++i, tt += step) {
                const double x[3] = {fma(double(tt), dx[0], x0[0]), fma(double(tt), dx[1], x0[1]),
                                     fma(double(tt), dx[2], x0[2])};
                if (in_range(f, x)) window_add(win, f, x, c);
            }
        });
        t = last + step;
    }
}

// The cell of a texel coordinate inside [-1, n)^3 and its trilinear
// fractions (the weights of march_tap).
__device__ __forceinline__ uint32_t cell_of(const RaymarchArgs& f, const double x[3], float w[3]) {
    const double fx = floor(x[0]), fy = floor(x[1]), fz = floor(x[2]);
    w[0] = float(x[0] - fx);
    w[1] = float(x[1] - fy);
    w[2] = float(x[2] - fz);
    const uint32_t cx = uint32_t(f.nx) + 1u, cy = uint32_t(f.ny) + 1u;
    return uint32_t(int(fx) + 1) + cx * (uint32_t(int(fy) + 1) + cy * uint32_t(int(fz) + 1));
}

// A wave's staging area of the scatter: every lane's sample (its cell and
// the 8 corner weights times the ray's gradient weight).
struct CellLds {
    uint32_t cell[kWave];
    float w[8][kWave];
};

static_assert(sizeof(CellLds) <= sizeof(WindowLds), "the wave's LDS holds either");

// Adds c * (trilinear corner weights) of every lane's sample to the cell
// accumulator; lanes without a sample pass cell == kNoCell.  The samples
// are staged in LDS and transposed: the 8 lanes of each group of 8 (one
// row of the wave's 8x8 pixel tile) walk the group's 8 samples in order,
// lane k adding corner k, so one sample is one 32-byte line request; a run
// of samples of the same cell along the row (neighbouring rays in one cell)
// is summed first and added once.  Every lane of the wave must call it.
__device__ __forceinline__ void scatter_wave(float* __restrict__ cg, CellLds& L, uint32_t cell, float wx,
                                             float wy, float wz, float c) {
    if (!__ballot(cell != kNoCell)) return;
    const int lane = __lane_id();
    const int k = lane & 7, group = lane & 56;
    L.cell[lane] = cell;
#pragma unroll
    for (int q = 0; q < 8; ++q)
        L.w[q][lane] = c * (((q & 1) ? wx : 1.0f - wx) * ((q & 2) ? wy : 1.0f - wy) * ((q & 4) ? wz : 1.0f - wz));
    wave_lds_sync();
    uint32_t run = kNoCell;
    float acc = 0.0f;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        const uint32_t sc = L.cell[group | r];
        const float v = L.w[k][group | r];
        if (sc != run) {
            if (run != kNoCell) unsafeAtomicAdd(&cg[size_t(run) * 8u + size_t(k)], acc);
            run = sc;
            acc = 0.0f;
        }
        acc += v;  // (kNoCell runs are never added)
    }
    if (run != kNoCell) unsafeAtomicAdd(&cg[size_t(run) * 8u + size_t(k)], acc);
    wave_lds_sync();  // the area is rewritten by the next call
}

// The samples of a family of rays into the cells (as scatter_rays; the loop
// runs to the wave's longest ray so that every lane takes part).
__device__ void scatter_rays_cells(const AdjointArgs& a, CellLds& L, bool active, const double x0[3], const double dx[3],
                             int n, float c) {
    const RaymarchArgs& f = a.f;
    const float step = f.step_size;
    const int n_lane = active ? n : 0;
    const int n_wave = wave_max(n_lane);
    float t = 0.0f;
    for (int i = 0; i < n_wave; ++i, t += step) {
        const double x[3] = {fma(double(t), dx[0], x0[0]), fma(double(t), dx[1], x0[1]), fma(double(t), dx[2], x0[2])};
        float w[3] = {0.0f, 0.0f, 0.0f};
        uint32_t cell = kNoCell;
        if (i < n_lane && in_range(f, x)) cell = cell_of(f, x, w);
        scatter_wave(a.cell_grad, L, cell, w[0], w[1], w[2], c);
    }
}

// Folds the corner-packed accumulator and the windows' texels into the texel
// gradient, and the workgroups' parameter sums into the parameter gradient
// (added; the sums are float64, since float32 adds in any order left them 2e-6
// off).  A wave takes 64 columns of kFoldRows rows and walks
// kFoldLevels levels up: a lane loads whole cells, adds the corners that are
// its own texels', takes the rest from its neighbour, and keeps the sums of
// two levels, so that a cell is loaded 1.7 times instead of its corners one
// by one in eight strided loads (bound by the lines those touch: 32.5 us at
// 128^3, 69 MB; 19.5 now, 23.4 with four rows, 20.4 with four levels).
constexpr int kFoldRows = 2, kFoldLevels = 8;

// kTexels: there are windows' texels.
template <bool kTexels>
__global__ void __launch_bounds__(256)
gather_cells_kernel(const float* __restrict__ cg, const float* __restrict__ texels, float* __restrict__ grad, int nx,
                    int ny, int nz, const double* __restrict__ param_sums, float* __restrict__ d_params) {
    // (atomic: calls on other streams may add to the same parameters)
    if (blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0 && threadIdx.x < 3)
        atomicAdd(&d_params[threadIdx.x], float(param_sums[threadIdx.x]));
    const int lane = threadIdx.x % kWave;
    const int x = int(blockIdx.x) * kWave + lane;
    const int y0 = (int(blockIdx.y) * (256 / kWave) + int(threadIdx.x) / kWave) * kFoldRows;
    const int z0 = int(blockIdx.z) * kFoldLevels, z1 = min(z0 + kFoldLevels, nz);
    if (y0 >= ny) return;   // wave-uniform
    const size_t cx = size_t(nx) + 1, cy = size_t(ny) + 1;
    float below[kFoldRows], above[kFoldRows];
#pragma unroll
    for (int r = 0; r < kFoldRows; ++r) below[r] = above[r] = 0.0f;
    for (int z = z0; z <= z1; ++z) {   // cell level z: corners of texel levels z - 1 and z
        float4 lo[kFoldRows + 1], hi[kFoldRows + 1], lo_end[kFoldRows + 1], hi_end[kFoldRows + 1];
#pragma unroll
        for (int r = 0; r <= kFoldRows; ++r) {   // cell row y0 + r: texel rows y0 + r - 1 and y0 + r
            lo[r] = hi[r] = lo_end[r] = hi_end[r] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            const size_t row = cx * (size_t(y0 + r) + cy * size_t(z));
            const float4* cell = reinterpret_cast<const float4*>(cg) + 2 * (row + size_t(x));
            if (x <= nx && y0 + r <= ny) {
                lo[r] = cell[0];
                hi[r] = cell[1];
                if (lane == kWave - 1 && x < nx) {   // the neighbour of the last lane
                    lo_end[r] = cell[2];
                    hi_end[r] = cell[3];
                }
            }
        }
#pragma unroll
        for (int r = 0; r <= kFoldRows; ++r) {
            // corners (1, b, c) of the lane's cell, (0, b, c) of the next one
            const bool end = lane == kWave - 1;
            const float n0 = __shfl_down(lo[r].x, 1, kWave), n2 = __shfl_down(lo[r].z, 1, kWave);
            const float n4 = __shfl_down(hi[r].x, 1, kWave), n6 = __shfl_down(hi[r].z, 1, kWave);
            const float s00 = lo[r].y + (end ? lo_end[r].x : n0), s10 = lo[r].w + (end ? lo_end[r].z : n2);
            const float s01 = hi[r].y + (end ? hi_end[r].x : n4), s11 = hi[r].w + (end ? hi_end[r].z : n6);
            if (r > 0) {   // b = 0: the row below the cell row
                below[r - 1] += s00;
                above[r - 1] += s01;
            }
            if (r < kFoldRows) {
                below[r] += s10;
                above[r] += s11;
            }
        }
        if (z > z0) {
#pragma unroll
            for (int r = 0; r < kFoldRows; ++r) {
                if (x >= nx || y0 + r >= ny) continue;
                const size_t i = size_t(x) + size_t(nx) * (size_t(y0 + r) + size_t(ny) * size_t(z - 1));
                const size_t t = size_t(x) + cx * (size_t(y0 + r) + cy * size_t(z - 1));
                grad[i] += (kTexels ? texels[t] : 0.0f) + below[r];
            }
        }
#pragma unroll
        for (int r = 0; r < kFoldRows; ++r) {
            below[r] = above[r];
            above[r] = 0.0f;
        }
    }
}

// What adjoint_tile takes: the primary rays with the parameter gradients (and
// the loss) and nothing else, or the shadow rays, the LAO taps or both.
enum AdjointWalk { kWalkPrimary = 1, kWalkShadow = 2, kWalkOcclusion = 4 };

// The adjoint of one pixel (volume.frag:31-102 differentiated).  Called by
// all 256 threads of a block: 2x2 waves of 8x8 pixels from (x0, y0); red is
// the block's reduction buffer for the parameter gradients.  Lds: WindowLds
// when the primary rays go through windows, else CellLds.
template <class Lds>
__device__ __forceinline__ void adjoint_tile(const AdjointArgs& a, int x0, int y0, double (*red)[256 / kWave],
                                             Lds* scatter, int walks) {
    // red: 4 x (waves per block) doubles
    constexpr bool kWindows = std::is_same<Lds, WindowLds>::value;
    const RaymarchArgs& f = a.f;
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    Lds& L = scatter[wave];
    CellLds& cells = *reinterpret_cast<CellLds*>(&L);
    // the windows' walk spreads a wave over the whole tile (lanes two pixels
    // apart): rays in one cell would add to the same LDS words in turn
    const bool primary = walks == kWalkPrimary, spread = kWindows && primary;
    const int px = spread ? x0 + (wave & 1) + 2 * (lane & 7) : x0 + (wave & 1) * 8 + (lane & 7);
    const int py = spread ? y0 + (wave >> 1) + 2 * (lane >> 3) : y0 + (wave >> 1) * 8 + (lane >> 3);
    const bool inside = px < f.width && py < f.height;
    const size_t pix = inside ? size_t(py) * f.width + px : 0;

    bool frag = false;
    MarchRecord r;
    float4 g = make_float4(0, 0, 0, 0);
    float sq = 0.0f;
    if (inside) {
        r = a.record[pix];
        frag = r.state == 1;
        if (a.target) {  // L2 loss against the target image
            const float4 o = f.rgba[pix], t = a.target[pix];
            const float4 d = make_float4(o.x - t.x, o.y - t.y, o.z - t.z, o.w - t.w);
            g = make_float4(2.0f * d.x, 2.0f * d.y, 2.0f * d.z, 2.0f * d.w);
            sq = d.x * d.x + d.y * d.y + d.z * d.z + d.w * d.w;
        } else {
            g = a.d_rgba[pix];
        }
    }
    double c_primary = 0.0, c_shadow = 0.0, G = 0.0;
    double d_alpha = 0.0, d_k = 0.0, d_p = 0.0;
    const bool adsm_on = f.adsm_on == 1 && f.shading_model != 3;
    const bool lao_on = f.shading_model != 2;
    if (frag) {
        const double gv[4] = {g.x, g.y, g.z, g.w};
        const double cov = f.lod * f.alpha * double(r.acc) / f.iso;
        const bool ua = cov > 0.0 && cov < 1.0;
        double rgb[3];
        for (int c = 0; c < 3; ++c) {
            rgb[c] = double(r.shade[c]) * double(r.adsm) * double(r.lao);
            const bool uc = rgb[c] > 0.0 && rgb[c] < 1.0;
            if (uc) G += gv[c] * rgb[c];
            if (uc && f.shading_model == 0 && r.spec_base > 0.0f) {
                double spec = pow(double(r.spec_base), f.shininess);
                d_p += gv[c] * double(r.adsm) * double(r.lao) * f.intensity[c] * spec * log(double(r.spec_base));
            }
        }
        if (ua) {
            c_primary = gv[3] * f.lod * f.alpha / f.iso;
            d_alpha += gv[3] * f.lod * double(r.acc) / f.iso;
        }
        if (adsm_on) {
            c_shadow = G * a.ln_transmit * f.adsm_k;
            d_k = G * a.ln_transmit * double(r.shadow_sum);
            d_alpha += G * (f.adsm_k * double(r.shadow_sum)) * (-1.0 / (1.0 - f.alpha));
        }
    }
    if (primary) {  // workgroup-uniform
        // parameter gradients (and the loss): wave, then block, then one atomic each
        const double pv[4] = {d_alpha, d_k, d_p, double(sq)};
        for (int k = 0; k < 4; ++k) {
            double v = pv[k];
            for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
            if (lane == 0) red[k][wave] = v;
        }
        __syncthreads();
        if (threadIdx.x < 4) {
            double v = 0.0;
            for (int w = 0; w < int(blockDim.x / kWave); ++w) v += red[threadIdx.x][w];
            float* dst = threadIdx.x < 3 ? &a.d_params[threadIdx.x] : a.loss;
            if (v != 0.0 && threadIdx.x < 3 && a.param_sums)
                unsafeAtomicAdd(&a.param_sums[threadIdx.x], v);
            else if (v != 0.0 && dst)
                atomicAdd(dst, float(v));
        }
        __syncthreads();  // red is reused by the next tile of a persistent block

        const Ray ray = setup_ray(f, px, py, inside && frag && c_primary != 0.0);
        const bool walk = ray.hit && c_primary != 0.0;
        const int n = frag ? r.n_primary : 0;
        if constexpr (kWindows)
            scatter_rays(a, L, walk, ray.xs, ray.dx, n, float(c_primary));
        else
            scatter_rays_cells(a, cells, walk, ray.xs, ray.dx, n, float(c_primary));
        return;
    }
    // shadow rays: from the surface point to the light origin, every sample
    double s[3] = {0, 0, 0}, sl[3] = {0, 0, 0};
    if (frag) {
        s[0] = r.sx; s[1] = r.sy; s[2] = r.sz;
        for (int k = 0; k < 3; ++k) sl[k] = a.light_texel[k] - s[k];
    }
    if (walks & kWalkShadow) {
        // samples past the volume's support carry no gradient: the walk stops
        // there (an upper bound on their count is enough, in_range does the rest)
        int n_shadow = 0;
        if (frag) {
            double lo, hi;
            support_interval(f, s, sl, &lo, &hi);
            if (hi >= 0.0 && lo <= hi)
                n_shadow = min(a.n_steps, int(fmin(hi, 2.0) / double(f.step_size) * 1.0001) + 2);
        }
        scatter_rays_cells(a, cells, frag && adsm_on && c_shadow != 0.0, s, sl, n_shadow, float(c_shadow));
    }
    if (!(walks & kWalkOcclusion)) return;
    // LAO taps: d ln(lao)/dD = -e / (8 - D), through min(v, clamp)
    const bool lao = frag && lao_on && G != 0.0;
    double v[8], D = 0.0;
    double tap[8][3];
    float taps[8] = {};
    if (lao) occlusion_taps<kFloats>(f.vol, s, f.ao_scaling, taps);
#pragma unroll
    for (int n = 0; n < 8; ++n) {
        tap[n][0] = s[0] + ((n & 1) ? 0.5 : -0.5) * f.ao_scaling;
        tap[n][1] = s[1] + (((n >> 1) & 1) ? 0.5 : -0.5) * f.ao_scaling;
        tap[n][2] = s[2] + ((n >> 2) ? 0.5 : -0.5) * f.ao_scaling;
        v[n] = lao ? double(taps[n]) : 0.0;
        D += fmin(v[n], f.ao_clamp);
    }
    const float cl = lao ? float(G * (-f.ao_exponent) / (8.0 - D)) : 0.0f;
#pragma unroll
    for (int n = 0; n < 8; ++n) {
        float w[3] = {0.0f, 0.0f, 0.0f};
        uint32_t cell = kNoCell;
        if (lao && v[n] < f.ao_clamp && in_range(f, tap[n])) cell = cell_of(f, tap[n], w);
        scatter_wave(a.cell_grad, cells, cell, w[0], w[1], w[2], cl);
    }
}

// blockIdx.z: 0 the primary rays and parameters, 1 the shadow rays, 2 the LAO
// taps (with windows 1 both).  In workgroups of their own the taps wait for neither
// walk: 64^3 / 24^2 / 16 steps 52 us against 67 behind the primary rays, 128^3 /
// 300^2 / 300 steps 289 against 302.
template <class Lds>
__device__ __forceinline__ void adjoint_block(const AdjointArgs& a) {
    __shared__ double red[4][256 / kWave];
    __shared__ Lds scatter[256 / kWave];
    const int x0 = int(blockIdx.x) * 16, y0 = int(blockIdx.y) * 16;
    if (blockIdx.z == 0)
        adjoint_tile(a, x0, y0, red, scatter, kWalkPrimary);
    else if (std::is_same<Lds, WindowLds>::value)
        adjoint_tile(a, x0, y0, red, scatter, kWalkShadow | kWalkOcclusion);
    else if (blockIdx.z == 1)
        adjoint_tile(a, x0, y0, red, scatter, kWalkShadow);
    else
        adjoint_tile(a, x0, y0, red, scatter, kWalkOcclusion);
}

__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
adjoint_windows_kernel(AdjointArgs) {
    adjoint_block<WindowLds>(kernel_args<AdjointArgs>());
}

__global__ void __launch_bounds__(256)
adjoint_cells_kernel(AdjointArgs) {
    adjoint_block<CellLds>(kernel_args<AdjointArgs>());
}

// ---------------------------------------------------------- batched form

struct AdjointBatchStyle {
    float* cell_grad;           // 8 floats per cell, owned by the batch
    float* texel_grad;          // what the windows are flushed to, in the cells' pitch, behind them (nullable)
    float* d_density;
    float* d_params;
    uint32_t nx, ny, nz;
    uint32_t reserved;
};

// A contiguous range [begin, end) of one style's accumulator floats, cells and
// texels (clear), or voxels (fold).
struct AdjointChunk {
    uint32_t style;
    uint32_t reserved;
    uint64_t begin, end;
};

struct AdjointBatchDevice {
    AdjointBatchStyle* styles;
    AdjointChunk* clear_chunks;
    AdjointChunk* fold_chunks;
    float** losses;             // per render, nullable entries
    uint32_t* order;            // the renders whose primary rays go through windows, then the others
    uint32_t n_windows;
    uint32_t n_styles, n_renders;
    uint32_t n_clear_chunks, n_fold_chunks;
    uint32_t tiles_x, tiles_per_render;
};

__global__ void __launch_bounds__(256)
adjoint_batch_clear_kernel(AdjointBatchDevice d) {
    if (blockIdx.x == 0) {
        for (uint32_t s = threadIdx.x; s < 3 * d.n_styles; s += blockDim.x) d.styles[s / 3].d_params[s % 3] = 0.0f;
        for (uint32_t r = threadIdx.x; r < d.n_renders; r += blockDim.x)
            if (d.losses[r]) *d.losses[r] = 0.0f;
    }
    for (uint32_t c = blockIdx.x; c < d.n_clear_chunks; c += gridDim.x) {
        const AdjointChunk ch = d.clear_chunks[c];
        float* cg = d.styles[ch.style].cell_grad;
        for (uint64_t i = ch.begin + threadIdx.x; i < ch.end; i += blockDim.x) cg[i] = 0.0f;
    }
}

// One block per (render, 16x16 tile): the recording forward.
__global__ void __launch_bounds__(256)
adjoint_batch_forward_kernel(AdjointBatchDevice d, const AdjointArgs* __restrict__ args) {
    __shared__ uint32_t occ_lds[1];  // float volumes carry no occupancy
    const uint32_t item = uint32_t(__builtin_amdgcn_readfirstlane(int(blockIdx.x)));
    const uint32_t r = item / d.tiles_per_render, tile = item % d.tiles_per_render;
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const int px = int(tile % d.tiles_x) * 16 + (wave & 1) * 8 + (lane & 7);
    const int py = int(tile / d.tiles_x) * 16 + (wave >> 1) * 8 + (lane >> 3);
    raymarch_pixel<true>(args[r].f, px, py, OccupancyView{occ_lds, false});
}

// One block per (render, 16x16 tile), the renders from order[first] on: the
// adjoint with the L2 loss gradient.
template <class Lds>
__device__ __forceinline__ void adjoint_batch_block(const AdjointBatchDevice& d, const AdjointArgs* __restrict__ args,
                                                    uint32_t first) {
    __shared__ double red[4][256 / kWave];
    __shared__ Lds scatter[256 / kWave];
    const uint32_t item = uint32_t(__builtin_amdgcn_readfirstlane(int(blockIdx.x)));
    const AdjointArgs& a = args[d.order[first + item / d.tiles_per_render]];
    const uint32_t tile = item % d.tiles_per_render;
    const int x0 = int(tile % d.tiles_x) * 16, y0 = int(tile / d.tiles_x) * 16;
    adjoint_tile(a, x0, y0, red, scatter, kWalkPrimary);
    adjoint_tile(a, x0, y0, red, scatter, kWalkShadow | kWalkOcclusion);
}

__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
adjoint_batch_windows_kernel(AdjointBatchDevice d, const AdjointArgs* __restrict__ args) {
    adjoint_batch_block<WindowLds>(d, args, 0u);
}

__global__ void __launch_bounds__(256)
adjoint_batch_cells_kernel(AdjointBatchDevice d, const AdjointArgs* __restrict__ args) {
    adjoint_batch_block<CellLds>(d, args, d.n_windows);
}

// d_density = the fold of each style's cells and texels (overwritten).
__global__ void __launch_bounds__(256)
adjoint_batch_fold_kernel(AdjointBatchDevice d) {
    for (uint32_t c = blockIdx.x; c < d.n_fold_chunks; c += gridDim.x) {
        const AdjointChunk ch = d.fold_chunks[c];
        const AdjointBatchStyle& st = d.styles[ch.style];
        const size_t cx = size_t(st.nx) + 1, cy = size_t(st.ny) + 1;
        for (uint64_t i = ch.begin + threadIdx.x; i < ch.end; i += blockDim.x) {
            const size_t x = i % st.nx, yz = i / st.nx, y = yz % st.ny, z = yz / st.ny;
            float sum = st.texel_grad ? st.texel_grad[x + cx * (y + cy * z)] : 0.0f;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const size_t cell = (x + 1 - (q & 1)) + cx * ((y + 1 - ((q >> 1) & 1)) + cy * (z + 1 - (q >> 2)));
                sum += st.cell_grad[cell * 8u + size_t(q)];
            }
            st.d_density[i] = sum;
        }
    }
}

}  // namespace
}  // namespace vkhr

using namespace vkhr;

extern "C" size_t vkhr_march_record_bytes(uint32_t width, uint32_t height) {
    return size_t(width) * height * sizeof(MarchRecord);
}

static int diff_args(const vkhr_volume* volume, const vkhr_camera* camera, const vkhr_light* light,
                     const vkhr_strand_params* strand, const vkhr_render_params* params, const vkhr_diff_params* diff,
                     uint32_t width, uint32_t height, RaymarchArgs* a) {
    int rc = make_raymarch_args(volume, camera, light, strand, params, width, height, a);
    if (rc) return rc;
    if (diff) {
        VKHR_REQUIRE(diff->absorption >= 0.0f && diff->absorption < 1.0f, VKHR_ERR_INVALID, "absorption %g",
                     diff->absorption);
        a->alpha = diff->absorption;
        a->adsm_k = diff->adsm_thickness;
        a->shininess = diff->shininess;
    }
    return VKHR_OK;
}

// Whether the primary rays' samples go through windows: when a wave's rays
// share texels but not one texel, and its chunk of steps fits a window.  The
// pitch of the pixels and the step are in texels (of the mean side, at the
// volume's centre); 16 pixels span a wave.  Measured (us of the adjoint, cells
// / windows; hair, steps in brackets): pitch 0.036 (0.22) 331 / 436, 0.08
// (0.45) 211 / 171, 0.23 (0.45) 140 / 97 at 64^3, 0.36 (0.9) 316 / 251 at
// 128^3; 0.58 (0.9) 269 / 600, 1.4 (0.9) 215 / 730, 2.8 (3.6) 107 / 1000.
static bool window_scatter(const RaymarchArgs& f, const vkhr_camera& camera) {
    double away2 = 0.0, texels = 1.0, volume = 1.0;
    for (int c = 0; c < 3; ++c) {
        const double d = f.origin[c] + 0.5 * f.size[c] - f.eye[c];
        away2 += d * d;
        volume *= f.size[c];
        texels *= f.nres[c];
    }
    const double texel = std::cbrt(volume / texels);
    const double focal = std::sqrt(std::fabs(double(camera.projection[0]) * double(camera.projection[5])));
    const double pitch = 2.0 * std::sqrt(away2 / (double(f.width) * f.height)) / (focal * texel);
    const double step = double(f.radius) * double(f.step_size) / texel;
    const double across = 16.0 * pitch + 2.0, along = std::fmin(16.0 * step, 8.0) + 2.0;
    return pitch >= 0.18 && step <= 1.2 && across * across * along <= 850.0;
}

// The per-launch constants of the adjoint derived from the forward's.
static void finish_adjoint_args(AdjointArgs* a) {
    int n = 0;
    for (float t = 0.0f; t < 1.0f; t += a->f.step_size) ++n;
    a->n_steps = n;
    a->ln_transmit = std::log(1.0 - a->f.alpha);
    for (int c = 0; c < 3; ++c)
        a->light_texel[c] = (a->f.light_origin[c] - a->f.origin[c]) / a->f.size[c] * a->f.nres[c] - 0.5;
}

extern "C" int vkhr_raymarch_record(const vkhr_volume* volume, const vkhr_camera* camera, const vkhr_light* light,
                                    const vkhr_strand_params* strand, const vkhr_render_params* params,
                                    const vkhr_diff_params* diff, uint32_t width, uint32_t height,
                                    const float* depth_buffer, float* rgba, float* depth, void* record,
                                    vkhr_stream stream) {
    clear_error();
    int rc = ensure_device();
    if (rc) return rc;
    VKHR_REQUIRE(rgba && record, VKHR_ERR_INVALID, "rgba/record is null");
    RaymarchArgs a;
    if ((rc = diff_args(volume, camera, light, strand, params, diff, width, height, &a))) return rc;
    a.depth_buffer = depth_buffer;
    a.rgba = reinterpret_cast<float4*>(rgba);
    a.depth = depth;
    a.record = static_cast<MarchRecord*>(record);
    launch_raymarch(a, as_stream(stream));
    VKHR_CHECK_LAUNCH();
    return VKHR_OK;
}

extern "C" int vkhr_raymarch_adjoint(const vkhr_volume* volume, const vkhr_camera* camera, const vkhr_light* light,
                                     const vkhr_strand_params* strand, const vkhr_render_params* params,
                                     const vkhr_diff_params* diff, uint32_t width, uint32_t height,
                                     const void* record, const float* d_rgba, float* d_density, float* d_params,
                                     vkhr_stream stream) {
    clear_error();
    int rc = ensure_device();
    if (rc) return rc;
    VKHR_REQUIRE(record && d_rgba && d_density && d_params, VKHR_ERR_INVALID, "null argument");
    VKHR_REQUIRE(volume && volume->density_f32, VKHR_ERR_INVALID, "the adjoint needs the float density volume");
    AdjointArgs* a = new AdjointArgs();
    std::memset(a, 0, sizeof(AdjointArgs));
    if ((rc = diff_args(volume, camera, light, strand, params, diff, width, height, &a->f))) {
        delete a;
        return rc;
    }
    a->record = static_cast<const MarchRecord*>(record);
    a->d_rgba = reinterpret_cast<const float4*>(d_rgba);
    a->d_params = d_params;
    finish_adjoint_args(a);
    const bool windows = window_scatter(a->f, *camera);
    // the cells, then with windows the texels (in the cells' pitch)
    const size_t n_cells = (size_t(volume->nx) + 1) * (size_t(volume->ny) + 1) * (size_t(volume->nz) + 1);
    const size_t sums = (n_cells * (windows ? 9 : 8) + 1) / 2 * 2, words = sums + 8;   // and the parameter sums
    void* cg = nullptr;
    hipStream_t st = as_stream(stream);
    if ((rc = stream_scratch(words * sizeof(float), st, &cg))) {
        delete a;
        return rc;
    }
    a->cell_grad = static_cast<float*>(cg);
    a->texel_grad = windows ? a->cell_grad + n_cells * 8 : nullptr;
    a->param_sums = reinterpret_cast<double*>(a->cell_grad + sums);
    a->texel_row = size_t(volume->nx) + 1;
    a->texel_slice = a->texel_row * (size_t(volume->ny) + 1);
    if ((rc = fill_u32(static_cast<uint32_t*>(cg), words, 0u, st))) {
        delete a;
        return rc;
    }
    // each walk family in workgroups of its own
    dim3 grid((width + 15) / 16, (height + 15) / 16, windows ? 2 : 3);
    if (windows)
        adjoint_windows_kernel<<<grid, 256, 0, st>>>(*a);
    else
        adjoint_cells_kernel<<<grid, 256, 0, st>>>(*a);
    const dim3 fold((volume->nx + kWave - 1) / kWave,
                    (volume->ny + kFoldRows * (256 / kWave) - 1) / (kFoldRows * (256 / kWave)),
                    (volume->nz + kFoldLevels - 1) / kFoldLevels);
    (windows ? gather_cells_kernel<true> : gather_cells_kernel<false>)<<<fold, 256, 0, st>>>(
        a->cell_grad, a->texel_grad, d_density, int(volume->nx), int(volume->ny), int(volume->nz), a->param_sums,
        d_params);
    delete a;
    VKHR_CHECK_LAUNCH();
    return VKHR_OK;
}

// ------------------------------------------------------------ batched form

struct vkhr_adjoint_batch {
    AdjointBatchDevice d;
    AdjointArgs* args = nullptr;      // device, per render
    std::vector<void*> allocations;
    uint32_t n_items = 0;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
};

namespace {

void release_adjoint_batch(vkhr_adjoint_batch* b) {
    if (b->exec) (void)hipGraphExecDestroy(b->exec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    for (void* p : b->allocations) (void)hipFree(p);
    b->allocations.clear();
}

template <class T>
int upload_table(vkhr_adjoint_batch* b, const std::vector<T>& host, T** out) {
    void* p = nullptr;
    VKHR_CHECK_HIP(hipMalloc(&p, std::max<size_t>(host.size() * sizeof(T), 16)));
    b->allocations.push_back(p);
    if (!host.empty()) VKHR_CHECK_HIP(hipMemcpy(p, host.data(), host.size() * sizeof(T), hipMemcpyHostToDevice));
    *out = static_cast<T*>(p);
    return VKHR_OK;
}

int build_adjoint_batch(vkhr_adjoint_batch* b, const vkhr_adjoint_style* styles, uint32_t n_styles,
                        const vkhr_adjoint_render* renders, uint32_t n_renders, uint32_t width, uint32_t height) {
    int rc = VKHR_OK;
    std::vector<AdjointBatchStyle> st(n_styles);
    std::vector<AdjointChunk> clear, fold;
    std::vector<uint64_t> n_cells(n_styles);
    std::vector<bool> windows(n_styles, false);   // some render of the style takes them
    const uint64_t kChunk = 1u << 16;
    for (uint32_t s = 0; s < n_styles; ++s) {
        const vkhr_adjoint_style& in = styles[s];
        VKHR_REQUIRE(in.volume.density_f32 && in.volume.tangents && in.d_density && in.d_params, VKHR_ERR_INVALID,
                     "style %u: the float density, tangents, d_density and d_params are required", s);
        if ((rc = check_volume(in.volume.nx, in.volume.ny, in.volume.nz, true, "adjoint style volume"))) return rc;
        const uint64_t cells = (uint64_t(in.volume.nx) + 1) * (uint64_t(in.volume.ny) + 1) * (uint64_t(in.volume.nz) + 1);
        n_cells[s] = cells;
        st[s] = {nullptr, nullptr, in.d_density, in.d_params, in.volume.nx, in.volume.ny, in.volume.nz, 0};
        const uint64_t vox = uint64_t(in.volume.nx) * in.volume.ny * in.volume.nz;
        for (uint64_t a = 0; a < vox; a += kChunk) fold.push_back({s, 0, a, std::min(vox, a + kChunk)});
    }
    std::vector<AdjointArgs> args(n_renders);
    std::vector<float*> losses(n_renders, nullptr);
    std::vector<uint32_t> order, in_cells;
    for (uint32_t r = 0; r < n_renders; ++r) {
        const vkhr_adjoint_render& in = renders[r];
        VKHR_REQUIRE(in.style < n_styles, VKHR_ERR_INVALID, "render %u: style %u of %u", r, in.style, n_styles);
        VKHR_REQUIRE(in.target && in.rgba && in.record, VKHR_ERR_INVALID, "render %u: target/rgba/record is null", r);
        AdjointArgs& a = args[r];
        std::memset(&a, 0, sizeof(a));
        if ((rc = diff_args(&styles[in.style].volume, &in.camera, &in.light, &in.strand, &in.params, &in.diff, width,
                            height, &a.f)))
            return rc;
        a.f.rgba = reinterpret_cast<float4*>(in.rgba);
        a.f.record = static_cast<MarchRecord*>(in.record);
        a.record = static_cast<const MarchRecord*>(in.record);
        a.target = reinterpret_cast<const float4*>(in.target);
        a.loss = in.loss;
        a.d_params = styles[in.style].d_params;
        a.texel_row = size_t(a.f.nx) + 1;
        a.texel_slice = a.texel_row * (size_t(a.f.ny) + 1);
        finish_adjoint_args(&a);
        losses[r] = in.loss;
        const bool in_windows = window_scatter(a.f, in.camera);
        if (in_windows) windows[in.style] = true;
        (in_windows ? order : in_cells).push_back(r);
    }
    // the accumulators: atomics go to memory of the batch's own (float atomics
    // to a caller's fine-grained memory would be lost)
    for (uint32_t s = 0; s < n_styles; ++s) {
        const uint64_t floats = n_cells[s] * (windows[s] ? 9 : 8);
        void* cg = nullptr;
        VKHR_CHECK_HIP(hipMalloc(&cg, floats * sizeof(float)));
        b->allocations.push_back(cg);
        st[s].cell_grad = static_cast<float*>(cg);
        if (windows[s]) st[s].texel_grad = st[s].cell_grad + n_cells[s] * 8;
        for (uint64_t a = 0; a < floats; a += kChunk) clear.push_back({s, 0, a, std::min(floats, a + kChunk)});
    }
    for (uint32_t r = 0; r < n_renders; ++r) {
        args[r].cell_grad = st[renders[r].style].cell_grad;
        args[r].texel_grad = st[renders[r].style].texel_grad;
    }
    const uint32_t n_windows = uint32_t(order.size());
    order.insert(order.end(), in_cells.begin(), in_cells.end());
    AdjointBatchDevice& d = b->d;
    if ((rc = upload_table(b, st, &d.styles)) || (rc = upload_table(b, clear, &d.clear_chunks)) ||
        (rc = upload_table(b, fold, &d.fold_chunks)) || (rc = upload_table(b, losses, &d.losses)) ||
        (rc = upload_table(b, args, &b->args)) || (rc = upload_table(b, order, &d.order)))
        return rc;
    d.n_styles = n_styles;
    d.n_renders = n_renders;
    d.n_windows = n_windows;
    d.n_clear_chunks = uint32_t(clear.size());
    d.n_fold_chunks = uint32_t(fold.size());
    d.tiles_x = (width + 15) / 16;
    d.tiles_per_render = d.tiles_x * ((height + 15) / 16);
    b->n_items = d.tiles_per_render * n_renders;
    return VKHR_OK;
}

}  // namespace

extern "C" int vkhr_adjoint_batch_create(const vkhr_adjoint_style* styles, uint32_t n_styles,
                                         const vkhr_adjoint_render* renders, uint32_t n_renders, uint32_t width,
                                         uint32_t height, vkhr_adjoint_batch** out) {
    clear_error();
    int rc = ensure_device();
    if (rc) return rc;
    VKHR_REQUIRE(styles && n_styles && renders && n_renders && out, VKHR_ERR_INVALID, "no styles or renders");
    VKHR_REQUIRE(width && height, VKHR_ERR_INVALID, "empty image");
    VKHR_REQUIRE(uint64_t(n_renders) * ((width + 15) / 16) * ((height + 15) / 16) < (uint64_t(1) << 31),
                 VKHR_ERR_INVALID, "too many tiles");
    vkhr_adjoint_batch* b = new vkhr_adjoint_batch();
    std::memset(&b->d, 0, sizeof(b->d));
    if ((rc = build_adjoint_batch(b, styles, n_styles, renders, n_renders, width, height))) {
        release_adjoint_batch(b);
        delete b;
        return rc;
    }
    *out = b;
    return VKHR_OK;
}

extern "C" int vkhr_adjoint_batch_launch(vkhr_adjoint_batch* b, vkhr_stream stream) {
    clear_error();
    VKHR_REQUIRE(b, VKHR_ERR_INVALID, "null batch");
    VKHR_REQUIRE(stream, VKHR_ERR_INVALID, "the batched launch is graph-captured: pass a created stream, not NULL");
    hipStream_t s = as_stream(stream);
    if (!b->exec) {
        VKHR_CHECK_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
        adjoint_batch_clear_kernel<<<4096, 256, 0, s>>>(b->d);
        adjoint_batch_forward_kernel<<<b->n_items, 256, 0, s>>>(b->d, b->args);
        const uint32_t in_windows = b->d.n_windows * b->d.tiles_per_render, in_cells = b->n_items - in_windows;
        if (in_windows) adjoint_batch_windows_kernel<<<in_windows, 256, 0, s>>>(b->d, b->args);
        if (in_cells) adjoint_batch_cells_kernel<<<in_cells, 256, 0, s>>>(b->d, b->args);
        adjoint_batch_fold_kernel<<<4096, 256, 0, s>>>(b->d);
        hipError_t e = hipStreamEndCapture(s, &b->graph);
        VKHR_CHECK_HIP(e);
        VKHR_CHECK_HIP(hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0));
    }
    VKHR_CHECK_HIP(hipGraphLaunch(b->exec, s));
    return VKHR_OK;
}

extern "C" int vkhr_adjoint_batch_destroy(vkhr_adjoint_batch* b) {
    clear_error();
    if (!b) return VKHR_OK;
    release_adjoint_batch(b);
    delete b;
    return VKHR_OK;
}
