// ReduceMean, Concat and Resize(nearest): the HBM-bound shape / reduction operators around the convolution path
// (lib_reduction_math.zig:30-268, lib_shape_math.zig:22-160, 307-630 in the reference).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "common.h"
#include "zant_hip.h"

namespace {

constexpr int kThreads = 256;

static inline unsigned grid_for(int64_t items, int per_block, int num_cus) {
    int64_t b = ceil_div64(items, per_block);
    const int64_t cap = int64_t(num_cus) * 32;
    if (b > cap) b = cap;
    return unsigned(b < 1 ? 1 : b);
}

// ---- ReduceMean --------------------------------------------------------------------------------
// Adjacent axes of the same kind (kept / reduced) are merged on the host, so at most four groups of each kind remain,
// outermost first.
struct ReduceGeom {
    int nk, nr;
    int64_t ksize[4], kstride[4];  // kept groups
    int64_t rsize[4], rstride[4];  // reduced groups
    int64_t outputs, count;        // number of results, elements per result
};

__device__ __forceinline__ int64_t kept_base(const ReduceGeom &g, int64_t o) {
    int64_t base = 0;
    for (int i = g.nk - 1; i > 0; --i) {
        const int64_t q = o / g.ksize[i];
        base += (o - q * g.ksize[i]) * g.kstride[i];
        o = q;
    }
    return g.nk ? base + o * g.kstride[0] : base;  // (what is left indexes the outermost group)
}

// The innermost group is reduced (unit stride): LANES lanes share one result and walk the contiguous run together.
// `seg` > 1 splits the run of a result into segments (few results, long runs); partial sums go to `part`.
// Bound by memory where a wave has enough of it in flight and few instructions around it: the usual form, planes of one kept group,
// takes no 64-bit division (each is some hundred instructions), and what does not fill a round of loads is asked for all at once too.
template <int LANES>
__global__ void __launch_bounds__(kThreads) reduce_mean_lanes_kernel(const float *__restrict__ x, float *__restrict__ y,
                                                                    ReduceGeom g, int seg, int64_t seg_len, int vec4) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    const int lane = threadIdx.x % LANES;
    const int64_t step = int64_t(gridDim.x) * (kThreads / LANES);
    const int64_t items = g.outputs * seg;
    const int64_t inner = g.rsize[g.nr - 1];
    int64_t outer = 1;
    for (int i = 0; i < g.nr - 1; ++i) outer *= g.rsize[i];
    for (int64_t it = int64_t(blockIdx.x) * (kThreads / LANES) + threadIdx.x / LANES; it < items; it += step) {
        const int64_t o = seg > 1 ? it / seg : it;
        const int s = int(it - o * seg);
        const float *row = x + kept_base(g, o);
        const int64_t lo = s * seg_len, hi = lo + seg_len < inner ? lo + seg_len : inner;
        float sum = 0.0f;
        for (int64_t c = 0; c < outer; ++c) {  // outer reduced groups (none in the common trailing-axes case)
            int64_t off = 0, r = c;
            for (int i = g.nr - 2; i > 0; --i) {
                const int64_t q = r / g.rsize[i];
                off += (r - q * g.rsize[i]) * g.rstride[i];
                r = q;
            }
            if (g.nr > 1) off += r * g.rstride[0];
            const float *p = row + off;
            if (vec4) {  // the host checked: base 16-byte aligned, every run start and length a multiple of 4
                const f4 *p4 = reinterpret_cast<const f4 *>(p);
                float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f, a3 = 0.0f;
                int64_t j = (lo >> 2) + lane;
                const int64_t j_end = hi >> 2;
                for (; j + 3 * LANES < j_end; j += 4 * LANES) {  // four loads in flight per lane
                    const f4 v0 = __builtin_nontemporal_load(p4 + j), v1 = __builtin_nontemporal_load(p4 + j + LANES);
                    const f4 v2 = __builtin_nontemporal_load(p4 + j + 2 * LANES), v3 = __builtin_nontemporal_load(p4 + j + 3 * LANES);
                    a0 += (v0.x + v1.x) + (v2.x + v3.x); a1 += (v0.y + v1.y) + (v2.y + v3.y);
                    a2 += (v0.z + v1.z) + (v2.z + v3.z); a3 += (v0.w + v1.w) + (v2.w + v3.w);
                }
                f4 v[3];  // (zeros where the run has ended: they change no sum)
#pragma unroll
                for (int i = 0; i < 3; ++i) v[i] = j + i * LANES < j_end ? __builtin_nontemporal_load(p4 + j + i * LANES) : f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int i = 0; i < 3; ++i) { a0 += v[i].x; a1 += v[i].y; a2 += v[i].z; a3 += v[i].w; }
                sum += (a0 + a1) + (a2 + a3);
            } else {
                for (int64_t j = lo + lane; j < hi; j += 8 * LANES) {  // eight loads in flight per lane
                    float v[8];
#pragma unroll
                    for (int i = 0; i < 8; ++i) v[i] = j + i * LANES < hi ? p[j + i * LANES] : 0.0f;
#pragma unroll
                    for (int i = 0; i < 8; ++i) sum += v[i];
                }
            }
        }
#pragma unroll
        for (int m = LANES / 2; m >= 1; m >>= 1) sum += __shfl_xor(sum, m, 64);
        if (lane == 0) y[it] = seg > 1 ? sum : sum / float(g.count);
    }
}

// Planes: one kept group, one contiguous run of `inner` elements per result, at most U loads of a lane.  A wave takes 256 / LANES
// results at once, four to a group of LANES lanes, and asks for all of their elements before it adds any: with one result at a time a
// plane of some hundred elements leaves one or two loads in flight and the six exchanges of its sum behind each.  The four sums of a
// group of 64 lanes meet in one register on the way (two half-wave swaps, one row swap), so four exchanges are left for four results.
// Each result is the same sum, in the same order, as reduce_mean_lanes_kernel's.  Means of 270000 planes of 13x13: 92 us one at a time, 64
// without the divisions, 41 here (4.4 TB/s); of 64064 planes of 26x26 34, 29 and 26.5 (6.5 TB/s).
template <int LANES, int U, typename V>
__global__ void __launch_bounds__(kThreads) reduce_mean_planes_kernel(const V *__restrict__ x, float *__restrict__ y, int64_t outputs,
                                                                      int inner, float count) {
    constexpr int GROUPS = 64 / LANES, ROWS = 4 * GROUPS;  // a wave's
    const int lane = threadIdx.x % LANES, group = threadIdx.x % 64 / LANES;
    const int64_t row0 = (int64_t(blockIdx.x) * (kThreads / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x / 64)) * ROWS;
    if (row0 >= outputs) return;
    V v[4][U];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int64_t row = row0 + group * 4 + r;
        const V *p = x + (row < outputs ? row : outputs - 1) * inner;  // (behind the last result: read again, not written)
#pragma unroll
        for (int u = 0; u < U; ++u) {
            v[r][u] = V{};
            if (u * LANES < inner && u * LANES + lane < inner) {
                if constexpr (sizeof(V) == 16) v[r][u] = __builtin_nontemporal_load(p + u * LANES + lane);
                else v[r][u] = p[u * LANES + lane];  // (rows share cache lines)
            }
        }
    }
    float sum[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if constexpr (sizeof(V) == 16) {
            V a = v[r][0];
#pragma unroll
            for (int u = 1; u < U; ++u) a += v[r][u];
            sum[r] = 0.0f + ((a.x + a.y) + (a.z + a.w));  // (+0 for a plane of -0, as from a sum that starts at +0)
        } else {
            sum[r] = 0.0f;
#pragma unroll
            for (int u = 0; u < U; ++u) sum[r] += v[r][u];
        }
    }
    if constexpr (LANES == 64) {
        auto both = [](auto sw) { return __uint_as_float(sw[0]) + __uint_as_float(sw[1]); };
        const float s02 = both(__builtin_amdgcn_permlane32_swap(__float_as_uint(sum[0]), __float_as_uint(sum[2]), false, false));
        const float s13 = both(__builtin_amdgcn_permlane32_swap(__float_as_uint(sum[1]), __float_as_uint(sum[3]), false, false));
        float s = both(__builtin_amdgcn_permlane16_swap(__float_as_uint(s02), __float_as_uint(s13), false, false));
#pragma unroll
        for (int m = 8; m >= 1; m >>= 1) s += __shfl_xor(s, m, 64);
        const int64_t row = row0 + lane / 16;  // (16 lanes hold one result each)
        if (lane % 16 == 0 && row < outputs) y[row] = s / count;
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t row = row0 + group * 4 + r;
#pragma unroll
            for (int m = LANES / 2; m >= 1; m >>= 1) sum[r] += __shfl_xor(sum[r], m, 64);
            if (lane == 0 && row < outputs) y[row] = sum[r] / count;
        }
    }
}

// Second pass of a segmented reduction: `seg` partial sums per result.
__global__ void __launch_bounds__(kThreads) reduce_mean_finish_kernel(const float *__restrict__ part, float *__restrict__ y,
                                                                     int64_t outputs, int seg, float count) {
    const int64_t o = int64_t(blockIdx.x) * (kThreads / 64) + threadIdx.x / 64;
    if (o >= outputs) return;
    float sum = 0.0f;
    for (int j = threadIdx.x % 64; j < seg; j += 64) sum += part[o * seg + j];
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) sum += __shfl_xor(sum, m, 64);
    if (threadIdx.x % 64 == 0) y[o] = sum / count;
}

// The innermost group is kept: one thread per result, neighbouring threads read neighbouring addresses.
__global__ void __launch_bounds__(kThreads) reduce_mean_threads_kernel(const float *__restrict__ x, float *__restrict__ y,
                                                                      ReduceGeom g) {
    const int64_t step = int64_t(gridDim.x) * kThreads;
    for (int64_t o = int64_t(blockIdx.x) * kThreads + threadIdx.x; o < g.outputs; o += step) {
        const float *row = x + kept_base(g, o);
        float sum = 0.0f;
        for (int64_t c = 0; c < g.count; ++c) {
            int64_t off = 0, r = c;
            for (int i = g.nr - 1; i >= 0; --i) {
                const int64_t q = r / g.rsize[i];
                off += (r - q * g.rsize[i]) * g.rstride[i];
                r = q;
            }
            sum += row[off];
        }
        y[o] = sum / float(g.count);
    }
}

// ---- Concat ------------------------------------------------------------------------------------
// One launch per input: `slices` chunks of `chunk` units each go to pitch-strided places in the output.
// Units narrower than 16 bytes are of pieces that start anywhere in a cache line, and a wave's store through the L2 at once (kept) leaves parts of
// lines to be written twice: of 4 bytes, [1001, 33, 13, 13] f32 twice 28.4 us that way and 22.4 nontemporal, 44.9 and 40.8 with the operator
// that reads them, [700, 30, 27, 27] 62.9 and 53.7; of 16, [1001, 33, 26, 26] 61.9 and 69.1.
template <typename U, typename I>
__global__ void __launch_bounds__(kThreads) concat_copy_kernel(const U *__restrict__ x, U *__restrict__ y, I total, I chunk,
                                                              int64_t pitch, int64_t offset, bool kept) {
    // streaming pattern: ZANT_STREAM_U x 256 consecutive units per workgroup, all loads before the stores
    const I base = I(blockIdx.x) * I(kThreads * ZANT_STREAM_U) + threadIdx.x;
    U v[ZANT_STREAM_U];
#pragma unroll
    for (int k = 0; k < ZANT_STREAM_U; ++k) {
        const I u = base + I(k * kThreads);
        if (u < total) v[k] = __builtin_nontemporal_load(x + u);
    }
#pragma unroll
    for (int k = 0; k < ZANT_STREAM_U; ++k) {
        const I u = base + I(k * kThreads);
        if (u < total) {
            const I sl = u / chunk, r = u - sl * chunk;
            U *to = y + (int64_t(sl) * pitch + offset + int64_t(r));
            if constexpr (sizeof(U) == 16) zant_store_out(v[k], to, kept);
            else __builtin_nontemporal_store(v[k], to);
        }
    }
}

// ---- Resize (nearest) --------------------------------------------------------------------------
struct ResizeGeom {
    int rank;
    int64_t xdim[8], ydim[8], xstride[8];
    int64_t tab_off[8];  // where each axis starts in the offset table
    int64_t tab_total, total;
    int coord_mode;
    FastDiv ydiv[8];  // division by ydim[d] (the vector kernel, whose indices stay below 2^31)
    FastDiv owdiv;    // ... by the number of vectors in an output row
};

// Input index of output coordinate o of an axis, in the reference's f32 arithmetic (lib_shape_math.zig:128-145):
// scale = out / in; half_pixel (o + 0.5) / scale - 0.5; align_corners o (in-1) / (out-1); otherwise o / scale; round half
// away from zero; clamp.  Never decreases with o.
__device__ __forceinline__ int64_t resize_source(int64_t o, int64_t in, int64_t out, int coord_mode) {
    const float scale = float(out) / float(in);
    float pos;
    if (coord_mode == 0) pos = (float(o) + 0.5f) / scale - 0.5f;
    else if (coord_mode == 1) pos = float(o) * float(in - 1) / float(out - 1);
    else pos = float(o) / scale;
    if (!(pos == pos)) pos = 0.0f;  // 0 / 0 of a one-element axis under align_corners
    int64_t i = int64_t(roundf(pos));
    i = i < 0 ? 0 : i;
    return i > in - 1 ? in - 1 : i;
}

// Input offset (index * stride) of every output coordinate of every axis.
// Written twice: as 64-bit offsets, and (for inputs of fewer than 2^31 elements) as 32-bit ones behind them.
__global__ void __launch_bounds__(kThreads) resize_table_kernel(int64_t *__restrict__ tab, ResizeGeom g) {
    const int64_t t = int64_t(blockIdx.x) * kThreads + threadIdx.x;
    if (t >= g.tab_total) return;
    int d = 0;
    while (d + 1 < g.rank && t >= g.tab_off[d + 1]) ++d;
    const int64_t o = t - g.tab_off[d];
    const int64_t i = resize_source(o, g.xdim[d], g.ydim[d], g.coord_mode);
    tab[t] = i * g.xstride[d];
    reinterpret_cast<int *>(tab + g.tab_total)[t] = int(i * g.xstride[d]);
}

template <typename U>
__global__ void __launch_bounds__(kThreads) resize_gather_kernel(const U *__restrict__ x, U *__restrict__ y,
                                                                const int64_t *__restrict__ tab, ResizeGeom g) {
    const int64_t step = int64_t(gridDim.x) * kThreads;
    for (int64_t o = int64_t(blockIdx.x) * kThreads + threadIdx.x; o < g.total; o += step) {
        int64_t r = o, off = 0;
        if (g.total < (int64_t(1) << 31)) {
            unsigned r32 = unsigned(r);
            for (int d = g.rank - 1; d >= 0; --d) {
                const unsigned n = unsigned(g.ydim[d]), q = r32 / n;
                off += tab[g.tab_off[d] + (r32 - q * n)];
                r32 = q;
            }
        } else {
            for (int d = g.rank - 1; d >= 0; --d) {
                const int64_t q = r / g.ydim[d];
                off += tab[g.tab_off[d] + (r - q * g.ydim[d])];
                r = q;
            }
        }
        y[o] = x[off];
    }
}

// VEC consecutive outputs of the innermost axis per thread (one 16-byte store); the outer axes are decoded once per thread.
// Streaming pattern: a workgroup takes ZANT_STREAM_U x 256 consecutive output vectors and issues all its gathers before its
// stores.  Stores are what this kernel is built around: whole, aligned, consecutive vectors (a variant that loaded whole
// input vectors and wrote each to its repeated places was twice as slow on rows that are not multiples of a cache line).
// What then bounds it is the address unit of the vector memory path, which takes every lane of every load whatever the
// lanes point at: so the tables of the innermost `lds_axes` axes (kResizeLdsEntries entries at most, 32-bit) are first
// copied to LDS and looked up there, and only the VEC gathers and the outer axes' 32-bit lookups go through it.
constexpr int kResizeLdsEntries = 2048;
template <typename U, int VEC>
__global__ void __launch_bounds__(kThreads) resize_gather_vec_kernel(const U *__restrict__ x, U *__restrict__ y,
                                                                    const int *__restrict__ tab, ResizeGeom g,
                                                                    unsigned nvec, unsigned ow_vec, int lds_axes, unsigned n_chunks) {
    typedef U UV __attribute__((ext_vector_type(VEC)));
    const bool kept = zant_out_kept(int64_t(nvec) * int64_t(sizeof(UV)));
    __shared__ __attribute__((aligned(16))) int tab_lds[kResizeLdsEntries];
    const int first = g.rank - lds_axes;  // axes first .. rank-1 are looked up in LDS
    const int lds_base = first < g.rank ? int(g.tab_off[first]) : int(g.tab_total);
    for (int c = threadIdx.x; c < int(g.tab_total) - lds_base; c += kThreads) tab_lds[c] = tab[lds_base + c];
    __syncthreads();
    const int *tw = tab + g.tab_off[g.rank - 1];
    const int tw_lds = int(g.tab_off[g.rank - 1]) - lds_base;
    // a workgroup stays for several chunks so that the table copy above is paid once and its waves drift apart
    for (unsigned chunk = blockIdx.x; chunk < n_chunks; chunk += gridDim.x) {
    const unsigned base = chunk * unsigned(kThreads * ZANT_STREAM_U) + threadIdx.x;
    UV out[ZANT_STREAM_U];
#pragma unroll
    for (int u = 0; u < ZANT_STREAM_U; ++u) {
        const unsigned v = base + unsigned(u * kThreads);
        if (v < nvec) {
            unsigned r = fastdiv(v, g.owdiv);
            const unsigned cv = v - r * ow_vec;
            int off = 0;  // below 2^31: the input has fewer elements than that
            for (int d = g.rank - 2; d >= 0; --d) {
                const unsigned n = unsigned(g.ydim[d]), q = fastdiv(r, g.ydiv[d]);
                const int e = int(g.tab_off[d]) + int(r - q * n);
                off += d >= first ? tab_lds[e - lds_base] : tab[e];
                r = q;
            }
            const U *row = x + off;
            if (lds_axes > 0) {
                int col[VEC];
#pragma unroll
                for (int k = 0; k < VEC; ++k) col[k] = tab_lds[tw_lds + int(cv) * VEC + k];
                bool wide = false;
                if constexpr (VEC <= 4) {
                    // up-sampling: the VEC sources lie within VEC consecutive input elements, so one (unaligned) 16-byte
                    // load and a register select replace VEC gathers -- a 4-byte gather at an 8-byte lane stride makes
                    // some thirty cache accesses per wave, a contiguous load four
                    int lo = col[0], hi = col[0];
#pragma unroll
                    for (int k = 1; k < VEC; ++k) { lo = min(lo, col[k]); hi = max(hi, col[k]); }
                    const int row_len = int(g.xdim[g.rank - 1]);
                    if (hi - lo < VEC && row_len >= VEC) {
                        wide = true;
                        const int b0 = min(lo, row_len - VEC);  // keep the window inside the row
                        UV w;
                        __builtin_memcpy(&w, row + b0, sizeof(UV));
#pragma unroll
                        for (int k = 0; k < VEC; ++k) {
                            const int sel = col[k] - b0;
                            U e = w[0];
#pragma unroll
                            for (int j = 1; j < VEC; ++j) e = sel == j ? w[j] : e;
                            out[u][k] = e;
                        }
                    }
                }
                if (!wide) {
#pragma unroll
                    for (int k = 0; k < VEC; ++k) out[u][k] = row[col[k]];
                }
            } else {
#pragma unroll
                for (int k = 0; k < VEC; ++k) out[u][k] = row[tw[cv * VEC + k]];
            }
        }
    }
#pragma unroll
    for (int u = 0; u < ZANT_STREAM_U; ++u) {
        const unsigned v = base + unsigned(u * kThreads);
        if (v < nvec) zant_store_out(out[u], reinterpret_cast<UV *>(y) + v, kept);
    }
    }
}

// The two innermost axes resized, the others kept (planes of H x W -> OH x OW).  A workgroup writes ZANT_STREAM_U x 256
// consecutive 16-byte vectors of the flat output, so stores are whole and aligned whatever the row length; the sources of
// consecutive outputs lie in one run of consecutive input elements (no axis' source index decreases), which is copied to
// LDS by coalesced loads and gathered there, each element read from memory once.  Row offsets and column indices are
// computed here: no table launch.  A run that does not fit `span_cap` elements is gathered from memory instead.
// HBM-bound: 1001x32x13x13 -> 26x26, 108 MB of f32, 26 us (4.2 TB/s; one output per thread through the tables: 93 us);
// as u8 13.6 us (82 us).
struct ResizePlanes {
    int H, W, OH, OW;
    unsigned total;
    int span_cap, rows_cap;  // LDS capacities: input elements, output rows
    int coord_mode;
    FastDiv d_oh, d_ow;
};
template <typename U, int VEC>
__global__ void __launch_bounds__(kThreads) resize_planes_kernel(const U *__restrict__ x, U *__restrict__ y, ResizePlanes g) {
    typedef U UV __attribute__((ext_vector_type(VEC)));
    const bool kept = zant_out_kept(int64_t(g.total) * int64_t(sizeof(U)));
    extern __shared__ __attribute__((aligned(16))) char lds[];
    U *span = reinterpret_cast<U *>(lds);
    int *rows = reinterpret_cast<int *>(lds + ((size_t(g.span_cap) * sizeof(U) + 15) & ~size_t(15)));
    int *cols = rows + g.rows_cap;
    constexpr unsigned CHUNK = kThreads * ZANT_STREAM_U * VEC;
    auto row_start = [&](unsigned r) -> unsigned {  // input offset of the row that output row r (of all planes) is made of
        const unsigned p = fastdiv(r, g.d_oh);
        return (p * unsigned(g.H) + unsigned(resize_source(int64_t(r - p * unsigned(g.OH)), g.H, g.OH, g.coord_mode))) * unsigned(g.W);
    };
    const unsigned o0 = blockIdx.x * CHUNK, o1 = min(o0 + CHUNK, g.total) - 1;  // first and last output
    const unsigned r0 = fastdiv(o0, g.d_ow), r1 = fastdiv(o1, g.d_ow);
    const unsigned s0 = row_start(r0), n_span = row_start(r1) + unsigned(g.W) - s0;
    const U *src = x + s0;
    const bool staged = n_span <= unsigned(g.span_cap);
    if (staged)
        for (unsigned e = threadIdx.x; e < n_span; e += kThreads) span[e] = __builtin_nontemporal_load(src + e);
    for (unsigned r = threadIdx.x; r <= r1 - r0; r += kThreads) rows[r] = int(row_start(r0 + r) - s0);
    for (int c = threadIdx.x; c < g.OW; c += kThreads) cols[c] = int(resize_source(c, g.W, g.OW, g.coord_mode));
    __syncthreads();
    auto gather = [&](auto from) {
#pragma unroll
        for (int u = 0; u < ZANT_STREAM_U; ++u) {
            const unsigned o = o0 + unsigned(u * kThreads + int(threadIdx.x)) * VEC;
            if (o > o1) break;
            const unsigned rel = o - r0 * unsigned(g.OW), r = fastdiv(rel, g.d_ow);
            int col = int(rel - r * unsigned(g.OW));
            int at = rows[r];
            const int next = rows[min(r + 1, r1 - r0)];
            UV v;
#pragma unroll
            for (int k = 0; k < VEC; ++k) {  // at most one row end inside a vector: OW >= VEC
                if (col == g.OW) { col = 0; at = next; }
                v[k] = from[at + cols[col]];
                ++col;
            }
            if (o + VEC - 1 <= o1) zant_store_out(v, reinterpret_cast<UV *>(y + o), kept);
            else
                for (int k = 0; k < VEC; ++k)
                    if (o + k <= o1) y[o + k] = v[k];
        }
    };
    if (staged) gather(span);
    else gather(src);
}

// Takes the call if it is one for resize_planes_kernel: kept outer axes (an axis of 2^21 and more could map to a neighbour
// in f32), rows of at least one vector, and a mean run of inputs per workgroup that fits LDS with several workgroups a CU.
// Rows of whole vectors of four or two elements stay with resize_gather_vec_kernel, whose one load and register select per
// vector is the faster there (512x32x32x32 -> 64x64 f32: 64 against 71 us; with 16 elements a vector it gathers each: the
// same as u8 41 against 34 us, 1001x32x12x12 -> 24x24 66 against 13 us).
template <typename U>
bool launch_resize_planes(zant_ctx *ctx, const void *x, void *y, const ResizeGeom &g) {
    constexpr int VEC = 16 / int(sizeof(U));
    constexpr int64_t CHUNK = int64_t(kThreads) * ZANT_STREAM_U * VEC;
    constexpr int64_t kLds = 40 << 10;  // four workgroups a CU
    const int64_t W = g.xdim[g.rank - 1], OW = g.ydim[g.rank - 1];
    const int64_t H = g.rank > 1 ? g.xdim[g.rank - 2] : 1, OH = g.rank > 1 ? g.ydim[g.rank - 2] : 1;
    int64_t in_total = H * W;
    for (int d = 0; d + 2 < g.rank; ++d) {
        if (g.xdim[d] != g.ydim[d] || g.xdim[d] >= (1 << 21)) return false;
        in_total *= g.xdim[d];
    }
    if (VEC <= 4 && OW % VEC == 0) return false;
    if ((reinterpret_cast<uintptr_t>(y) & 15) != 0 || OW < VEC || OW > 4096 || g.total + CHUNK >= (int64_t(1) << 31) || in_total >= (int64_t(1) << 31))
        return false;
    const int64_t rows = std::min((CHUNK - 1) / OW + 2, g.total / OW);
    const int64_t span = std::min(in_total, W * (ceil_div64(rows * H, OH) + 3));
    const int64_t span_bytes = (span * int64_t(sizeof(U)) + 15) & ~int64_t(15);
    const int64_t lds_bytes = span_bytes + (rows + OW) * int64_t(sizeof(int));
    if (lds_bytes > kLds) return false;
    // Every input row of the run is copied, needed or not, an element a thread at a time.  Down to 22 rounds of that a workgroup's
    // latency is no longer than the table launch it saves (60x200 -> 30x401 f32, 60 planes, 8.4 against 8.3 us of kernels; u8 12 to 29
    // against 6 to 8 from 40 rounds on); longer runs need two workgroups per CU to hide it (u8 800 planes of 60x200 -> 30x401, 587
    // workgroups, 27 against 36 us; -> 24x401, 470 workgroups, 34 against 30) and at most 1.6 inputs an output (f32 8000 planes of
    // 60x76 -> 20x149 85 against 100 us, -> 15x149 93 against 78).
    if (span > 22 * kThreads && (ceil_div64(g.total, CHUNK) < 2 * ctx->num_cus || 5 * H * W > 8 * OH * OW)) return false;
    ResizePlanes p;
    p.H = int(H); p.W = int(W); p.OH = int(OH); p.OW = int(OW);
    p.total = unsigned(g.total);
    p.span_cap = int(span); p.rows_cap = int(rows);
    p.coord_mode = g.coord_mode;
    p.d_oh = make_fastdiv(unsigned(OH)); p.d_ow = make_fastdiv(unsigned(OW));
    ZANT_KERNEL_NAME(ctx, "resize_planes_kernel<%d,%d>", int(sizeof(U)), VEC);
    hipLaunchKernelGGL((resize_planes_kernel<U, VEC>), dim3(unsigned(ceil_div64(g.total, CHUNK))), dim3(kThreads), size_t(lds_bytes), ctx->stream,
                       static_cast<const U *>(x), static_cast<U *>(y), p);
    return true;
}

template <typename U>
int launch_resize(zant_ctx *ctx, const void *x, void *y, ResizeGeom &g) {
    constexpr int VEC = 16 / int(sizeof(U));
    const int64_t ow = g.ydim[g.rank - 1];
    {
        KernelTimer kt(ctx);
        if (launch_resize_planes<U>(ctx, x, y, g)) {
            ZANT_LAUNCH_CHECK(ctx);
            return ZANT_OK;
        }
    }
    void *ws = nullptr;
    const int rc = zant_workspace(ctx, size_t(g.tab_total) * (sizeof(int64_t) + sizeof(int)), &ws);
    if (rc != ZANT_OK) return rc;
    int64_t *tab = static_cast<int64_t *>(ws);
    hipLaunchKernelGGL(resize_table_kernel, dim3(unsigned(ceil_div64(g.tab_total, kThreads))), dim3(kThreads), 0, ctx->stream, tab, g);
    ZANT_LAUNCH_CHECK(ctx);
    int64_t in_total = 1;
    for (int d = 0; d < g.rank; ++d) in_total *= g.xdim[d];
    KernelTimer kt(ctx);
    if (ow % VEC == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0 && g.total / VEC < (int64_t(1) << 31) &&
        in_total < (int64_t(1) << 31) && g.tab_total < (int64_t(1) << 31)) {
        for (int d = 0; d < g.rank; ++d) g.ydiv[d] = make_fastdiv(unsigned(g.ydim[d]));  // ydim[d] <= total / VEC here for d < rank - 1
        g.owdiv = make_fastdiv(unsigned(ow / VEC));
        int lds_axes = 0;  // as many innermost axes as fit
        while (lds_axes < g.rank && g.tab_total - g.tab_off[g.rank - 1 - lds_axes] <= kResizeLdsEntries) ++lds_axes;
        const unsigned n_chunks = zant_stream_grid(g.total / VEC);
        hipLaunchKernelGGL((resize_gather_vec_kernel<U, VEC>), dim3(std::min(n_chunks, unsigned(ctx->num_cus) * 8u)), dim3(kThreads), 0,
                           ctx->stream, static_cast<const U *>(x), static_cast<U *>(y), reinterpret_cast<const int *>(tab + g.tab_total),
                           g, unsigned(g.total / VEC), unsigned(ow / VEC), lds_axes, n_chunks);
    } else
        hipLaunchKernelGGL(resize_gather_kernel<U>, dim3(grid_for(g.total, kThreads, ctx->num_cus)), dim3(kThreads), 0, ctx->stream,
                           static_cast<const U *>(x), static_cast<U *>(y), tab, g);
    ZANT_LAUNCH_CHECK(ctx);
    return ZANT_OK;
}

template <typename U>
int launch_concat(zant_ctx *ctx, const void *x, void *y, int64_t slices, int64_t chunk, int64_t pitch, int64_t offset) {
    const int64_t total = slices * chunk;
    const bool kept = zant_out_kept(slices * pitch * int64_t(sizeof(U)));
    if (total < (int64_t(1) << 31))
        hipLaunchKernelGGL((concat_copy_kernel<U, unsigned>), dim3(zant_stream_grid(total)), dim3(kThreads), 0,
                           ctx->stream, static_cast<const U *>(x), static_cast<U *>(y), unsigned(total), unsigned(chunk), pitch,
                           offset, kept);
    else
        hipLaunchKernelGGL((concat_copy_kernel<U, int64_t>), dim3(zant_stream_grid(total)), dim3(kThreads), 0,
                           ctx->stream, static_cast<const U *>(x), static_cast<U *>(y), total, chunk, pitch, offset, kept);
    ZANT_LAUNCH_CHECK(ctx);
    return ZANT_OK;
}

typedef unsigned u4 __attribute__((ext_vector_type(4)));

}  // namespace

// -------------------------------------------------------------------------------------------------

extern "C" int zant_hip_reduce_mean_f32(zant_ctx *ctx, const float *x, const int64_t *xdim, int rank, const int64_t *axes,
                                        int n_axes, int keepdims, int noop_with_empty_axes, float *y, int64_t *ydim_out,
                                        int *y_rank_out) {
    if (!xdim || !ydim_out || !y_rank_out) return ZANT_NullPointer;
    if (rank < 0 || rank > 8) return ZANT_InvalidDimensions;
    for (int i = 0; i < rank; ++i)
        if (xdim[i] < 0) return ZANT_InvalidDimensions;
    const int64_t size = prod_dims(xdim, rank);
    bool reduced[8] = {false, false, false, false, false, false, false, false};
    if (!axes || n_axes == 0) {  // lib_reduction_math.zig:35-46, 111-128
        if (noop_with_empty_axes) {
            for (int i = 0; i < rank; ++i) ydim_out[i] = xdim[i];
            *y_rank_out = rank;
            if (!y || size == 0) return ZANT_OK;
            if (!ctx || !x) return ZANT_NullPointer;
            if (y != x) ZANT_HIP_TRY(ctx, hipMemcpyAsync(y, x, size_t(size) * sizeof(float), hipMemcpyDeviceToDevice, ctx->stream));
            return ZANT_OK;
        }
        if (keepdims) {
            for (int i = 0; i < rank; ++i) ydim_out[i] = 1;
            *y_rank_out = rank;
        } else {
            ydim_out[0] = 1;
            *y_rank_out = 1;
        }
        for (int i = 0; i < rank; ++i) reduced[i] = true;
    } else {
        if (n_axes > 8) return ZANT_InvalidAxes;
        for (int i = 0; i < n_axes; ++i) {  // :131-141; a repeated axis is rejected (the reference would read out of bounds)
            const int64_t a = axes[i] < 0 ? axes[i] + rank : axes[i];
            if (a < 0 || a >= rank || reduced[a]) return ZANT_InvalidAxes;
            reduced[a] = true;
        }
        int out_rank = 0;
        for (int i = 0; i < rank; ++i)  // :62-76
            if (!reduced[i] || keepdims) ydim_out[out_rank++] = reduced[i] ? 1 : xdim[i];
        *y_rank_out = out_rank;
    }
    if (!y) return ZANT_OK;
    if (!ctx || !x) return ZANT_NullPointer;
    if (size == 0) return ZANT_ZeroSizeTensor;

    // merge neighbouring axes of one kind; axes of extent 1 join whatever is next to them
    ReduceGeom g = {};
    g.outputs = 1;
    g.count = 1;
    int64_t stride[8], st = 1;
    for (int i = rank - 1; i >= 0; --i) { stride[i] = st; st *= xdim[i]; }
    int last_kind = -1;  // 0 kept, 1 reduced
    for (int i = 0; i < rank; ++i) {
        if (xdim[i] == 1) continue;
        const int kind = reduced[i] ? 1 : 0;
        if (kind == last_kind) {
            if (kind) { g.rsize[g.nr - 1] *= xdim[i]; g.rstride[g.nr - 1] = stride[i]; }
            else { g.ksize[g.nk - 1] *= xdim[i]; g.kstride[g.nk - 1] = stride[i]; }
        } else if (kind) {
            g.rsize[g.nr] = xdim[i]; g.rstride[g.nr++] = stride[i];
        } else {
            g.ksize[g.nk] = xdim[i]; g.kstride[g.nk++] = stride[i];
        }
        last_kind = kind;
        if (kind) g.count *= xdim[i]; else g.outputs *= xdim[i];
    }
    if (g.nr == 0) {  // only axes of extent 1 were reduced: a copy
        if (y != x) ZANT_HIP_TRY(ctx, hipMemcpyAsync(y, x, size_t(size) * sizeof(float), hipMemcpyDeviceToDevice, ctx->stream));
        return ZANT_OK;
    }
    if (last_kind == 0) {
        KernelTimer kt(ctx);
        hipLaunchKernelGGL(reduce_mean_threads_kernel, dim3(grid_for(g.outputs, kThreads, ctx->num_cus)), dim3(kThreads), 0,
                           ctx->stream, x, y, g);
        ZANT_LAUNCH_CHECK(ctx);
        return ZANT_OK;
    }
    const int64_t inner = g.rsize[g.nr - 1];
    // few results with long runs: cut each run into segments so the whole chip reads, then add the partial sums
    int seg = 1;
    int64_t seg_len = inner;
    if (g.nr == 1 && g.outputs < int64_t(ctx->num_cus) * 16 && inner >= (1 << 16)) {
        int64_t want = ceil_div64(int64_t(ctx->num_cus) * 32, g.outputs);
        const int64_t most = inner >> 14;  // at least 16 Ki elements per segment
        if (want > most) want = most;
        if (want > 4096) want = 4096;
        if (want > 1) {
            seg_len = ceil_div64(ceil_div64(inner, want), 4) * 4;
            seg = int(ceil_div64(inner, seg_len));
        }
    }
    bool vec4 = (reinterpret_cast<uintptr_t>(x) & 15) == 0 && inner % 4 == 0 && inner >= 256;
    for (int i = 0; i < g.nk && vec4; ++i) vec4 = g.kstride[i] % 4 == 0;
    for (int i = 0; i + 1 < g.nr && vec4; ++i) vec4 = g.rstride[i] % 4 == 0;
    float *dst = y;
    if (seg > 1) {
        void *ws = nullptr;
        const int rc = zant_workspace(ctx, size_t(g.outputs) * seg * sizeof(float), &ws);
        if (rc != ZANT_OK) return rc;
        dst = static_cast<float *>(ws);
    }
    const int64_t items = g.outputs * seg;
    const int64_t per_lane_run = vec4 ? inner / 4 : inner;
    // planes that a group of lanes reads in few loads each (three of vectors, eight of elements): four of them at once.  Longer runs fill
    // a lane's loads by themselves; runs under 16 elements are left to the four-lane groups.
    const int64_t groups = per_lane_run >= 64 ? 1 : 4;
    const int64_t blocks = ceil_div64(g.outputs, groups * 4 * (kThreads / 64));
    if (g.nk == 1 && g.nr == 1 && seg == 1 && per_lane_run >= 16 && per_lane_run <= (vec4 ? 192 : 512) && blocks <= ZANT_MAX_BLOCKS_256) {
        typedef float f4 __attribute__((ext_vector_type(4)));
        KernelTimer kt(ctx);
#define ZANT_PLANES(LANES, U, V)                                                                                                    \
    hipLaunchKernelGGL((reduce_mean_planes_kernel<LANES, U, V>), dim3(unsigned(blocks)), dim3(kThreads), 0, ctx->stream,            \
                       reinterpret_cast<const V *>(x), y, g.outputs, int(per_lane_run), float(g.count))
        if (vec4) ZANT_PLANES(64, 3, f4);
        else if (groups == 4) ZANT_PLANES(16, 4, float);
        else if (inner <= 256) ZANT_PLANES(64, 4, float);
        else ZANT_PLANES(64, 8, float);
#undef ZANT_PLANES
        ZANT_LAUNCH_CHECK(ctx);
        return ZANT_OK;
    }
    {
        KernelTimer kt(ctx);
        if (per_lane_run >= 64)
            hipLaunchKernelGGL(reduce_mean_lanes_kernel<64>, dim3(grid_for(items, kThreads / 64, ctx->num_cus)), dim3(kThreads), 0,
                               ctx->stream, x, dst, g, seg, seg_len, vec4 ? 1 : 0);
        else if (per_lane_run >= 16)
            hipLaunchKernelGGL(reduce_mean_lanes_kernel<16>, dim3(grid_for(items, kThreads / 16, ctx->num_cus)), dim3(kThreads), 0,
                               ctx->stream, x, dst, g, seg, seg_len, vec4 ? 1 : 0);
        else
            hipLaunchKernelGGL(reduce_mean_lanes_kernel<4>, dim3(grid_for(items, kThreads / 4, ctx->num_cus)), dim3(kThreads), 0,
                               ctx->stream, x, dst, g, seg, seg_len, vec4 ? 1 : 0);
    }
    ZANT_LAUNCH_CHECK(ctx);
    if (seg > 1) {
        hipLaunchKernelGGL(reduce_mean_finish_kernel, dim3(unsigned(ceil_div64(g.outputs, kThreads / 64))), dim3(kThreads), 0,
                           ctx->stream, dst, y, g.outputs, seg, float(g.count));
        ZANT_LAUNCH_CHECK(ctx);
    }
    return ZANT_OK;
}

extern "C" int zant_hip_concatenate(zant_ctx *ctx, const void *const *xs, const int64_t *const *dims, const int *ranks, int n,
                                    int64_t axis, size_t elem_size, void *y, int64_t *ydim_out, int *y_rank_out) {
    if (n <= 0) return ZANT_EmptyTensorList;  // lib_shape_math.zig:308
    if (!dims || !ranks || !ydim_out || !y_rank_out) return ZANT_NullPointer;
    if (n > 16) return ZANT_InvalidDimensions;
    int rank = 0;
    for (int t = 0; t < n; ++t) {
        if (ranks[t] < 0 || ranks[t] > 8 || !dims[t]) return ZANT_InvalidDimensions;
        if (ranks[t] > rank) rank = ranks[t];  // :314-320
    }
    if (axis < 0) axis += rank;  // :363-370
    if (axis < 0 || axis >= rank) return ZANT_AxisOutOfBounds;
    int64_t shp[16][8];
    for (int t = 0; t < n; ++t) {  // lower ranks get leading ones (:335-358)
        const int off = rank - ranks[t];
        for (int d = 0; d < rank; ++d) shp[t][d] = d < off ? 1 : dims[t][d - off];
    }
    int64_t total_cd = 0;
    for (int t = 0; t < n; ++t) {  // :374-380
        for (int d = 0; d < rank; ++d)
            if (d != axis && shp[t][d] != shp[0][d]) return ZANT_MismatchedShape;
        total_cd += shp[t][axis];
    }
    for (int d = 0; d < rank; ++d) ydim_out[d] = d == axis ? total_cd : shp[0][d];
    *y_rank_out = rank;
    if (!y) return ZANT_OK;
    if (!ctx || !xs) return ZANT_NullPointer;
    if (elem_size != 1 && elem_size != 2 && elem_size != 4 && elem_size != 8) return ZANT_InvalidInput;
    int64_t slices = 1, inner = 1;
    for (int d = 0; d < axis; ++d) slices *= shp[0][d];
    for (int d = int(axis) + 1; d < rank; ++d) inner *= shp[0][d];
    const int64_t pitch_b = total_cd * inner * int64_t(elem_size);
    int64_t off_b = 0;
    KernelTimer kt(ctx);
    for (int t = 0; t < n; ++t) {
        const int64_t chunk_b = shp[t][axis] * inner * int64_t(elem_size);
        if (chunk_b > 0 && slices > 0) {
            if (!xs[t]) return ZANT_NullPointer;
            const uintptr_t a = reinterpret_cast<uintptr_t>(xs[t]) | reinterpret_cast<uintptr_t>(y) | uintptr_t(chunk_b) |
                                uintptr_t(pitch_b) | uintptr_t(off_b);
            int rc;
            if (slices == 1) {  // one contiguous block
                ZANT_HIP_TRY(ctx, hipMemcpyAsync(static_cast<char *>(y) + off_b, xs[t], size_t(chunk_b), hipMemcpyDeviceToDevice,
                                                 ctx->stream));
                rc = ZANT_OK;
            } else if ((a & 15) == 0) rc = launch_concat<u4>(ctx, xs[t], y, slices, chunk_b / 16, pitch_b / 16, off_b / 16);
            else if ((a & 3) == 0) rc = launch_concat<uint32_t>(ctx, xs[t], y, slices, chunk_b / 4, pitch_b / 4, off_b / 4);
            else rc = launch_concat<uint8_t>(ctx, xs[t], y, slices, chunk_b, pitch_b, off_b);
            if (rc != ZANT_OK) return rc;
        }
        off_b += chunk_b;
    }
    return ZANT_OK;
}

extern "C" int zant_hip_resize_nearest(zant_ctx *ctx, const void *x, const int64_t *xdim, int rank, size_t elem_size,
                                       const float *scales, const int64_t *sizes, int n_param, int coord_mode, void *y,
                                       int64_t *ydim_out) {
    if ((!scales && !sizes) || (scales && sizes)) return ZANT_InvalidInput;  // lib_shape_math.zig:23-28
    if (!xdim || !ydim_out) return ZANT_NullPointer;
    if (n_param != rank || rank < 1 || rank > 8) return ZANT_InvalidInput;  // :35-37, 43-45
    ResizeGeom g = {};
    g.rank = rank;
    g.coord_mode = coord_mode;
    g.total = 1;
    for (int i = 0; i < rank; ++i) {
        if (xdim[i] < 0) return ZANT_InvalidDimensions;
        ydim_out[i] = scales ? int64_t(floorf(float(xdim[i]) * scales[i])) : sizes[i];  // :38-40
        if (ydim_out[i] < 0) return ZANT_InvalidInput;
        g.xdim[i] = xdim[i];
        g.ydim[i] = ydim_out[i];
        g.tab_off[i] = g.tab_total;
        g.tab_total += ydim_out[i];
        g.total *= ydim_out[i];
    }
    if (!y) return ZANT_OK;
    if (g.total == 0) return ZANT_OK;
    if (!ctx || !x) return ZANT_NullPointer;
    if (prod_dims(xdim, rank) == 0) return ZANT_ZeroSizeTensor;
    if (elem_size != 1 && elem_size != 2 && elem_size != 4 && elem_size != 8) return ZANT_InvalidInput;
    int64_t st = 1;
    for (int i = rank - 1; i >= 0; --i) { g.xstride[i] = st; st *= xdim[i]; }
    switch (elem_size) {
    case 1: return launch_resize<uint8_t>(ctx, x, y, g);
    case 2: return launch_resize<uint16_t>(ctx, x, y, g);
    case 4: return launch_resize<uint32_t>(ctx, x, y, g);
    default: return launch_resize<uint64_t>(ctx, x, y, g);
    }
}
