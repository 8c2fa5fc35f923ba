// Small kernels of the paged flow-LM KV cache: block-table patches and plan pulls, the standalone
// append of t rows, shifting-ring eviction, page copies, raw row I/O and voice loading.
#include "kernels_common.h"

namespace xnp {

// ---------------------------------------------------------------------------------------------
// block-table patches (pages taken since the previous batch)

__global__ void k_patch_tables(int32_t *tables, const TablePatch *patches, int n, int mbps) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) tables[(size_t)patches[i].sid * mbps + patches[i].blk] = patches[i].page;
}

hipError_t launch_patch_tables(const PoolView &pv, const TablePatch *patches, int n, hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_patch_tables, dim3((n + 255) / 256), dim3(256), 0, stream, pv.tables, patches, n,
                       pv.mbps);
    return hipGetLastError();
}

// The batch plan, read straight from the pinned staging buffer the host composed it in, and the
// block-table patches staged behind it: one launch, where copies would take a copy engine per
// part plus a patch kernel, with a hand-off between engines before each.  The launch boundary
// makes the host's writes to the buffer visible.
__global__ __launch_bounds__(256) void k_pull_plan(const uint4 *src, uint4 *dst, int n16, const TablePatch *patches,
                                                   int np, int32_t *tables, int mbps) {
    const int stride = gridDim.x * blockDim.x, i0 = blockIdx.x * blockDim.x + threadIdx.x;
    for (int i = i0; i < n16; i += stride) dst[i] = src[i];
    for (int i = i0; i < np; i += stride) {
        const TablePatch t = patches[i];
        tables[(size_t)t.sid * mbps + t.blk] = t.page;
    }
}

hipError_t launch_pull_plan(const PoolView &pv, const void *src, void *dst, size_t bytes, const TablePatch *patches,
                            int np, hipStream_t stream) {
    const int n16 = (int)((bytes + 15) / 16), work = std::max(n16, np);
    if (work <= 0) return hipSuccess;
    const int blocks = std::min((work + 255) / 256, 1024);
    hipLaunchKernelGGL(k_pull_plan, dim3(blocks), dim3(256), 0, stream, (const uint4 *)src, (uint4 *)dst, n16, patches,
                       np, pv.tables, pv.mbps);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// standalone append of t rows per stream, f32 and bf16 pools: a work group per (stream, row), one wave
// per kv head.  (A page's rows in turn by one wave took 8.3 us for one stream's 64 rows, a round trip
// each; a wave per row and head 3.4 us.)  A launch holds fewer than 2^32 threads: more rows than
// kAppendGroups take several launches, from row r0 on.
constexpr int kAppendGroups = 1 << 20;

template <int CDT, bool ABF>
__global__ __launch_bounds__(1024) void k_append(PoolView pv, BatchView bv, int layer, const void *k, const void *v, int r0) {
    const int t = bv.t, r = r0 + (int)blockIdx.x, b = r / t, i = r % t;
    const StreamPlan P = bv.plans[b];
    const int j = threadIdx.x >> 6; // kv head
    const int slot = P.write_slot + i;
    const int page = pv.tables[(size_t)P.sid * pv.mbps + (slot >> 4)];
    if (page < 0 || page >= pv.NB) return; // begin took this page; never index the pool without one
    constexpr int AE = ABF ? 2 : 4;
    const size_t arow = ((size_t)P.out_row * t + i) * pv.KVH + j;
    append_row_wave<CDT, ABF>(pv, layer, page, slot & 15, j, P.key_pos + i, (const char *)k + arow * kHeadDim * AE,
                              (const char *)v + arow * kHeadDim * AE, false);
}

// The int8 append of a step's rows, one wave per (stream, page the rows touch, kv head, keys or
// values) with the whole tile in registers: lane l holds dims 16 (l % 4) .. + 15 of the page's row
// l / 4, so a tile's rows load at once and its codes leave in one coalesced 1 KB store.
//
// The result is that of appending the rows one by one (append_row_wave): row r is quantized with the
// scale in effect after it, s_r = max(s_(r-1), amax_r / 127), and requantized at every later row that
// raises the scale.  So: every row's amax / 127 (one division a lane), the scales s_r in row order
// (scalars), each row's codes at its own s_r (all rows together), then one requantization of the
// rows before it per scale increase (about 2.4 a page for N(0, 1) rows).
//
// What bounded the row-by-row form was the correctly rounded division in front of each rint: about
// 138 a lane and page, in a chain of one round trip per row.  Here a code is rint(y * (1 / s)), which
// is rint(y / s) unless the quotient lies near a half (code16 below); 16 rows' first codes cost what
// one row's did.  48 prompts of 250 rows, 8 heads, append and attention: 86.4 -> 45.4 us a layer, of
// which the attention is 20.7.
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
constexpr float kHalfBand = 0.5f - 6e-5f;

// 16 values to codes rint(y / s), as floats: |y| <= 127 s up to rounding.  The product y * inv, inv =
// 1 / s rounded, lies within 2^-23 |y / s| (1 + 2^-24) < 1.6e-5 of the exact quotient, and the division
// rounds it by at most 3.9e-6 more; away from a half by more than 6e-5 both round to the same integer.
// Where any of the 16 is nearer, or not finite, or s is outside the range where 1 / s is normal, the
// division is taken.
__device__ __forceinline__ void code16(float (&y)[16], float s) {
    const float inv = 1.0f / s;
    bool far = s > 1e-30f && s < 1e30f;
    float q[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const float p = y[i] * inv;
        q[i] = __builtin_rintf(p);
        far = far && fabsf(p - q[i]) < kHalfBand;
    }
    if (!far) {
#pragma unroll
        for (int i = 0; i < 16; ++i) q[i] = (float)quant(y[i], s);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) y[i] = q[i];
}

template <bool ABF>
__global__ __launch_bounds__(128) void k_append_i8(PoolView pv, BatchView bv, int layer, const void *k, const void *v,
                                                   int nseg) {
    const int j = blockIdx.x % pv.KVH, seg = blockIdx.x / pv.KVH % nseg, b = blockIdx.x / pv.KVH / nseg; // j: kv head
    const StreamPlan P = bv.plans[b];
    const int t = bv.t, ws = P.write_slot, blk = (ws >> 4) + seg;
    const int i0 = max(0, blk * kBlock - ws), i1 = min(t, (blk + 1) * kBlock - ws);
    if (i0 >= i1) return;
    const int page = pv.tables[(size_t)P.sid * pv.mbps + blk];
    if (page < 0 || page >= pv.NB) return; // begin took this page; never index the pool without one
    const int kv = threadIdx.x >> 6, lane = threadIdx.x & 63, row = lane >> 2, c = lane & 3;
    const int r0 = (ws + i0) & 15, r1 = r0 + (i1 - i0); // the page's rows written
    const bool mine = row >= r0 && row < r1;
    const bool fresh = P.ring ? P.fresh != 0 : r0 == 0; // the page holds no other row
    const int i = i0 + min(max(row - r0, 0), i1 - i0 - 1); // the lane's input row (clamped; used where mine)
    const size_t arow = (((size_t)P.out_row * t + i) * pv.KVH + j) * kHeadDim + 16 * c;
    const void *src = kv ? v : k;
    const size_t tile = tile_index(pv, layer, kv, page, j);
    uint4 *codes = (uint4 *)((int8_t *)pv.pages + tile * (kBlock * kHeadDim)) + lane;
    uint4 old = make_uint4(0, 0, 0, 0);
    float s = 0.f;
    if (!fresh) {
        old = *codes;
        s = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(pv.scales[tile])));
    }
    float y[16];
    if constexpr (ABF) {
        uint4 raw[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) { // rows need word alignment only, as append_row_wave's loads do
            const u32x4_a4 u = ((const u32x4_a4 *)((const uint16_t *)src + arow))[h];
            raw[h] = make_uint4(u.x, u.y, u.z, u.w);
        }
        if (kv == 0) {
            const uint4 *cs = (const uint4 *)(pv.rope16 + (size_t)(P.key_pos + i) * (kHeadDim / 2) + 8 * c);
#pragma unroll
            for (int h = 0; h < 2; ++h) raw[h] = rotate8(raw[h], cs[h]);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t u = ((const uint32_t *)&raw[e >> 2])[e & 3];
            y[2 * e] = bf16_value(u & 0xffffu);
            y[2 * e + 1] = bf16_value(u >> 16);
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            float2 x = ((const float2 *)((const float *)src + arow))[e];
            if (kv == 0) {
                const float2 cs = pv.rope[(size_t)(P.key_pos + i) * (kHeadDim / 2) + 8 * c + e];
                const float a = x.x * cs.x, bb = x.y * cs.y, d = x.x * cs.y, f = x.y * cs.x;
                x = make_float2(a - bb, d + f);
            }
            y[2 * e] = x.x;
            y[2 * e + 1] = x.y;
        }
    }
    float amax = fabsf(y[0]);
#pragma unroll
    for (int e = 1; e < 16; ++e) amax = fmaxf(amax, fabsf(y[e]));
    amax = fmaxf(amax, dpp_move<0xB1>(amax)); // the row's 4 lanes
    amax = fmaxf(amax, dpp_move<0x4E>(amax));
    const float srow = amax / 127.0f;
    // the scale after each written row: its own row's in the lanes of that row, every scale increase
    // past the first row in `raised` (bit r), the rows' scales as scalars in after[]
    float after[kBlock], own = 1.f;
    const float s0 = s;
    uint32_t raised = 0;
#pragma unroll
    for (int r = 0; r < kBlock; ++r) {
        after[r] = s;
        if (r < r0 || r >= r1) continue;
        const float sr = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(srow), 4 * r));
        const bool first = fresh && r == r0;
        const float sn = first ? sr : fmaxf(s, sr);
        if (!first && sn > s) raised |= 1u << r;
        s = sn;
        after[r] = s;
        if (row == r) own = s;
    }
    if (mine) code16(y, own);
    if (!mine) {
#pragma unroll
        for (int e = 0; e < 16; ++e) y[e] = (float)(int8_t)((((const uint32_t *)&old)[e >> 2] >> (8 * (e & 3))) & 0xffu);
    }
    const bool held = !mine && !fresh && (P.ring || row < r0); // a row the page held before
    if (raised) {
#pragma unroll
        for (int r = 0; r < kBlock; ++r) {
            if (!((raised >> r) & 1u)) continue; // uniform
            const float so = r > 0 ? (r == r0 ? s0 : after[r - 1]) : s0, sn = after[r];
            if (held || (mine && row < r)) {
#pragma unroll
                for (int e = 0; e < 16; ++e) y[e] *= so;
                code16(y, sn);
            }
        }
    }
    if (mine || (held && raised)) {
        uint32_t w[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            w[e] = ((uint32_t)(int)y[4 * e] & 0xffu) | ((uint32_t)(int)y[4 * e + 1] & 0xffu) << 8 |
                   ((uint32_t)(int)y[4 * e + 2] & 0xffu) << 16 | ((uint32_t)(int)y[4 * e + 3] & 0xffu) << 24;
        *codes = make_uint4(w[0], w[1], w[2], w[3]);
    }
    if (lane == 0) pv.scales[tile] = s;
}

// The same a row after another, one wave per kv head and a work group per (stream, page), for steps of one or
// two rows, and of three in large batches: k_append_i8 takes the page's tile whole whatever the rows.  1000
// streams, 8 kv heads, new pages / 37 held rows: one row 20.2 (k_append_i8) and 7.1 us / 20.6 and 7.1, two rows
// 25.2 and 22.0 / 22.2 and 9.9, three 28.9 and 33.4 / 23.3 and 12.9, four 31.8 and 42.2 / 24.8 and 16.3; 8 streams:
// two rows 5.3 and 6.0 / 4.7 and 4.4, three 6.4 and 8.4 / 4.7 and 4.9.
template <bool ABF>
__global__ __launch_bounds__(1024) void k_append_i8_few(PoolView pv, BatchView bv, int layer, const void *k, const void *v,
                                                        int nseg) {
    const int b = blockIdx.x / nseg, seg = blockIdx.x % nseg;
    const StreamPlan P = bv.plans[b];
    const int j = threadIdx.x >> 6, t = bv.t, ws = P.write_slot, blk = (ws >> 4) + seg; // j: kv head
    const int i0 = max(0, blk * kBlock - ws), i1 = min(t, (blk + 1) * kBlock - ws);
    if (i0 >= i1) return;
    const int page = pv.tables[(size_t)P.sid * pv.mbps + blk];
    if (page < 0 || page >= pv.NB) return; // begin took this page; never index the pool without one
    constexpr int AE = ABF ? 2 : 4;
    for (int i = i0; i < i1; ++i) {
        const size_t arow = ((size_t)P.out_row * t + i) * pv.KVH + j;
        const bool fresh = P.ring ? (P.fresh != 0) : (((ws + i) & 15) == 0);
        append_row_wave<DT_I8, ABF>(pv, layer, page, (ws + i) & 15, j, P.key_pos + i, (const char *)k + arow * kHeadDim * AE,
                                    (const char *)v + arow * kHeadDim * AE, fresh);
        __syncthreads(); // the row's codes and scale before the next row reads them
    }
}
static bool append_i8_few(const PoolView &pv, const BatchView &bv) {
    return bv.t <= 2 || (bv.t == 3 && (int64_t)bv.n * pv.KVH >= 2048);
}

template <int CDT, bool ABF>
static hipError_t append_impl(const PoolView &pv, const BatchView &bv, int layer, const void *k,
                              const void *v, hipStream_t stream) {
    if constexpr (CDT == DT_I8) {
        const int nseg = (bv.t + kBlock - 1) / kBlock + 1; // the most pages a stream's rows touch
        if (append_i8_few(pv, bv))
            hipLaunchKernelGGL(k_append_i8_few<ABF>, dim3(bv.n * nseg), dim3(64 * pv.KVH), 0, stream, pv, bv, layer, k, v, nseg);
        else
            hipLaunchKernelGGL(k_append_i8<ABF>, dim3(bv.n * nseg * pv.KVH), dim3(128), 0, stream, pv, bv, layer, k, v, nseg);
    } else {
        for (int r0 = 0; r0 < bv.n * bv.t; r0 += kAppendGroups)
            hipLaunchKernelGGL((k_append<CDT, ABF>), dim3(std::min(bv.n * bv.t - r0, kAppendGroups)), dim3(64 * pv.KVH), 0, stream,
                               pv, bv, layer, k, v, r0);
    }
    return hipGetLastError();
}

hipError_t launch_append(const PoolView &pv, const BatchView &bv, int layer, const void *k, const void *v,
                         hipStream_t stream) {
    if (bv.n == 0) return hipSuccess;
    switch (pv.cache_dt * 2 + pv.act_dt) {
    case DT_F32 * 2 + DT_F32: return append_impl<DT_F32, false>(pv, bv, layer, k, v, stream);
    case DT_BF16 * 2 + DT_BF16: return append_impl<DT_BF16, true>(pv, bv, layer, k, v, stream);
    case DT_I8 * 2 + DT_BF16: return append_impl<DT_I8, true>(pv, bv, layer, k, v, stream);
    case DT_I8 * 2 + DT_F32: return append_impl<DT_I8, false>(pv, bv, layer, k, v, stream);
    default: return hipErrorInvalidValue;
    }
}

// ---------------------------------------------------------------------------------------------
// A window step's rows into the held windows after its attention (Mimi's chunk where query heads share a kv
// head, bf16 and f32 pools): slot s takes the step's last row i with (p + i) % window == s; a row that a later row of the
// step overwrites is never written.  One work group per (stream, page of the window), one wave per
// kv head for the page's 16 slots.
//   bf16: lane l takes 16-byte unit l % 8 of the K and V rows of slots l / 8 and l / 8 + 8, and
//         each slot's row comes from the lane's own arithmetic: four 16-byte loads and the RoPE
//         pieces of its two keys, all issued unconditionally (a slot the step leaves alone loads
//         row 0, never stored), then rotate8 on the keys (the packed bf16 table the prefill
//         kernels rotate with: the same products and roundings as append_row_wave) and four
//         16-byte stores.
//   f32:  each lane one pair of dims (keys in lanes 0-31, values in 32-63, as append_row_wave),
//         every slot's loads first, then the rotations and stores.
// A loop of append_row_wave calls took 96 us per layer at 256 streams x 250 rows (each slot's loads
// waited for the previous slot's stores), and one slot per step of a scalar loop 68 us (two
// integer divisions per slot on the scalar unit).

template <int CDT, bool ABF>
__global__ __launch_bounds__(1024) void k_window_append(PoolView pv, BatchView bv, int layer, const void *k,
                                                        const void *v) {
    static_assert((CDT == DT_BF16 && ABF) || (CDT == DT_F32 && !ABF), "bf16 and f32 windows; int8 ones append row by row");
    const int b = blockIdx.x / pv.mbps, blk = blockIdx.x % pv.mbps;
    const StreamPlan P = bv.plans[b];
    const int W = P.window, t = bv.t, j = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (W <= 0 || kBlock * blk >= W || P.pos_pre == 0) return; // (a fresh window's: written by k_prefill_window)
    const int page = pv.tables[(size_t)P.sid * pv.mbps + blk];
    if (page < 0 || page >= pv.NB) return; // begin took this page; never index the pool without one
    const int rb = ((kBlock * blk - P.pos) % W + W) % W; // the first row of the step in the page's slot 0
    // the last row of the step in slot kBlock * blk + n, or -1
    auto last_row = [&](int n) {
        const int s = kBlock * blk + n, r = (rb + n) % W;
        return s < W && r < t ? (t <= W ? r : r + W * ((t - 1 - r) / W)) : -1;
    };
    if constexpr (CDT == DT_BF16) {
        const int unit = lane & 7;
        int row[2];
        uint4 kx[2], vx[2], cs[2];
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
            row[hf] = last_row((lane >> 3) + 8 * hf);
            const int i = max(row[hf], 0);
            const size_t arow = (((size_t)P.out_row * t + i) * pv.KVH + j) * kHeadDim + 8 * unit;
            kx[hf] = ld_stream((const uint16_t *)k + arow); // read once: streamed past the caches
            vx[hf] = ld_stream((const uint16_t *)v + arow);
            cs[hf] = *(const uint4 *)(pv.rope16 + (size_t)(P.key_pos + i) * (kHeadDim / 2) + 4 * unit);
        }
        uint16_t *kt = (uint16_t *)pv.pages + tile_index(pv, layer, 0, page, j) * (kBlock * kHeadDim);
        uint16_t *vt = (uint16_t *)pv.pages + tile_index(pv, layer, 1, page, j) * (kBlock * kHeadDim);
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
            if (row[hf] < 0) continue;
            const int o = ((lane >> 3) + 8 * hf) * kHeadDim + 8 * unit;
            *(uint4 *)(kt + o) = rotate8(kx[hf], cs[hf]);
            *(uint4 *)(vt + o) = vx[hf];
        }
    } else {
        const int kv = lane >> 5, pr = lane & 31;
        const char *src = (const char *)(kv ? v : k);
        int row[kBlock];
        float2 x[kBlock], cs[kBlock];
#pragma unroll
        for (int n = 0; n < kBlock; ++n) {
            row[n] = last_row(n);
            const int i = max(row[n], 0);
            x[n] = load_pair<false>(src + (((size_t)P.out_row * t + i) * pv.KVH + j) * kHeadDim * 4, pr);
            cs[n] = pv.rope[(size_t)(P.key_pos + i) * (pv.D / 2) + pr];
        }
        const size_t tile = tile_index(pv, layer, kv, page, j);
#pragma unroll
        for (int n = 0; n < kBlock; ++n) {
            if (row[n] < 0) continue;
            float2 y = x[n];
            if (kv == 0) { // the key rotated at its position (rope.rs:74-95), as append_row_wave rotates it
                const float a = y.x * cs[n].x, bb = y.y * cs[n].y, e = y.x * cs[n].y, f = y.y * cs[n].x;
                y.x = a - bb;
                y.y = e + f;
            }
            ((float2 *)pv.pages)[tile * (kBlock * kHeadDim / 2) + n * (kHeadDim / 2) + pr] = y;
        }
    }
}

hipError_t launch_window_append(const PoolView &pv, const BatchView &bv, int layer, const void *k, const void *v,
                                hipStream_t stream) {
    if (bv.n == 0) return hipSuccess;
    const dim3 grid(bv.n * pv.mbps), block(64 * pv.KVH);
    switch (pv.cache_dt * 2 + pv.act_dt) {
    case DT_F32 * 2 + DT_F32: hipLaunchKernelGGL((k_window_append<DT_F32, false>), grid, block, 0, stream, pv, bv, layer, k, v); break;
    case DT_BF16 * 2 + DT_BF16: hipLaunchKernelGGL((k_window_append<DT_BF16, true>), grid, block, 0, stream, pv, bv, layer, k, v); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// eviction on a shifting ring: rotate one kept key row by -count in place (transformer.rs:905-926)

template <int CDT, bool ABF>
__global__ void k_evict_rotate(PoolView pv, const EvictRow *rows, const float2 *cs_row) {
    const EvictRow R = rows[blockIdx.x / pv.L];
    const int layer = blockIdx.x % pv.L;
    const int j = threadIdx.x >> 5, pr = threadIdx.x & 31; // kv head, dim pair
    const int page = pv.tables[(size_t)R.sid * pv.mbps + (R.slot >> 4)];
    if (page < 0 || page >= pv.NB) return;
    const size_t e = tile_index(pv, layer, 0, page, j) * (kBlock * kHeadDim) + (R.slot & 15) * kHeadDim + 2 * pr;
    float2 x;
    if constexpr (CDT == DT_F32) {
        x = *(const float2 *)((const float *)pv.pages + e);
    } else {
        uint32_t w = *(const uint32_t *)((const uint16_t *)pv.pages + e);
        x = make_float2(bf16_value(w & 0xffffu), bf16_value(w >> 16));
    }
    const float2 cs = cs_row[pr];
    float a = x.x * cs.x, b = x.y * cs.y, ee = x.x * cs.y, f = x.y * cs.x;
    x.x = round_act<ABF>(a - b);
    x.y = round_act<ABF>(ee + f);
    if constexpr (CDT == DT_F32)
        *(float2 *)((float *)pv.pages + e) = x;
    else
        *(uint32_t *)((uint16_t *)pv.pages + e) = bf16_bits(x.x) | (bf16_bits(x.y) << 16);
}

hipError_t launch_evict_rotate(const PoolView &pv, const EvictRow *rows, int n, const float *cs,
                               const float *, hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    const dim3 grid(n * pv.L), block(32 * pv.KVH);
    const float2 *csr = (const float2 *)cs;
    switch (pv.cache_dt * 2 + pv.act_dt) {
    case DT_F32 * 2 + DT_F32: hipLaunchKernelGGL((k_evict_rotate<DT_F32, false>), grid, block, 0, stream, pv, rows, csr); break;
    case DT_BF16 * 2 + DT_BF16: hipLaunchKernelGGL((k_evict_rotate<DT_BF16, true>), grid, block, 0, stream, pv, rows, csr); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// page copy (fork of a partial last page, unsharing before a ring): every layer, K and V, scales

__global__ void k_copy_page(PoolView pv, int src, int dst, int tile_u4) {
    const int layer = blockIdx.x >> 1, kv = blockIdx.x & 1;
    const uint4 *s = (const uint4 *)pv.pages + tile_index(pv, layer, kv, src, 0) * tile_u4;
    uint4 *d = (uint4 *)pv.pages + tile_index(pv, layer, kv, dst, 0) * tile_u4;
    const int n = tile_u4 * pv.KVH;
    for (int i = threadIdx.x; i < n; i += blockDim.x) d[i] = s[i];
    if (pv.scales && threadIdx.x < pv.KVH)
        pv.scales[tile_index(pv, layer, kv, dst, threadIdx.x)] = pv.scales[tile_index(pv, layer, kv, src, threadIdx.x)];
}

hipError_t launch_copy_page(const PoolView &pv, int src_page, int dst_page, hipStream_t stream) {
    const int es = pv.cache_dt == DT_F32 ? 4 : pv.cache_dt == DT_BF16 ? 2 : 1;
    const int tile_u4 = kBlock * kHeadDim * es / 16;
    hipLaunchKernelGGL(k_copy_page, dim3(pv.L * 2), dim3(256), 0, stream, pv, src_page, dst_page, tile_u4);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// raw row I/O: rows [n][H][D] in the cache dtype <-> the stream's pages; int8 scales per page

__global__ void k_rows_io(PoolView pv, int sid, int layer, int kv, int slot0, void *rows, float *scales,
                          int write, int row_u4) {
    const int s = blockIdx.x;
    const int slot = slot0 + s;
    const int page = pv.tables[(size_t)sid * pv.mbps + (slot >> 4)];
    if (page < 0 || page >= pv.NB) return;
    const int per_head = row_u4 / pv.KVH;
    for (int i = threadIdx.x; i < row_u4; i += blockDim.x) {
        const int h = i / per_head, w = i % per_head;
        uint4 *pg = (uint4 *)pv.pages + tile_index(pv, layer, kv, page, h) * (kBlock * per_head) + (slot & 15) * per_head + w;
        uint4 *rw = (uint4 *)rows + (size_t)s * row_u4 + i;
        if (write)
            *pg = *rw;
        else
            *rw = *pg;
    }
    if (scales && ((slot & 15) == 0 || s == 0) && threadIdx.x < pv.KVH) {
        const int bi = (slot >> 4) - (slot0 >> 4);
        float *ps = pv.scales + tile_index(pv, layer, kv, page, threadIdx.x);
        float *us = scales + (size_t)bi * pv.KVH + threadIdx.x;
        if (write)
            *ps = *us;
        else
            *us = *ps;
    }
}

hipError_t launch_rows_io(const PoolView &pv, int sid, int layer, int kv, int slot0, int n, void *rows,
                          float *scales, bool write, hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    const int es = pv.cache_dt == DT_F32 ? 4 : pv.cache_dt == DT_BF16 ? 2 : 1;
    const int row_u4 = pv.KVH * kHeadDim * es / 16;
    hipLaunchKernelGGL(k_rows_io, dim3(n), dim3(256), 0, stream, pv, sid, layer, kv, slot0, rows,
                       pv.cache_dt == DT_I8 ? scales : nullptr, write ? 1 : 0, row_u4);
    return hipGetLastError();
}

// A voice stored as the KV cache (voice_from_kv_cache, ptts-wasm/src/lib.rs:291-325): rows
// [0, n) of one layer from an f32 [2][n][H][D] tensor (keys, already rotated, then values),
// converted to the cache dtype: f32 as is, bf16 rounded to nearest even, int8 with one scale per
// (page, head), amax / 127 over the rows the page receives, and codes rint(x / s).  One wave per
// (page, head, keys or values); lane d holds dimension d of each of the page's 16 rows, so every
// row is one coalesced 256 B read.  Rows past n in the last page are left as they are.
template <int CDT>
__global__ __launch_bounds__(64) void k_load_kv(PoolView pv, int sid, int layer, const float *kv, int n) {
    const int b = blockIdx.x, j = blockIdx.y, which = blockIdx.z, lane = threadIdx.x;
    const int h = j * (pv.H / pv.KVH); // the voice repeats kv head j over its group's query heads
    const int page = pv.tables[(size_t)sid * pv.mbps + b];
    if (page < 0 || page >= pv.NB) return;
    const int rows = min(kBlock, n - b * kBlock);
    float x[kBlock];
#pragma unroll
    for (int r = 0; r < kBlock; ++r) { // all 16 loads in flight; rows past n re-read the last one
        const int slot = b * kBlock + min(r, rows - 1);
        x[r] = kv[(((size_t)which * n + slot) * pv.H + h) * kHeadDim + lane];
    }
    const size_t tile = tile_index(pv, layer, which, page, j);
    if constexpr (CDT == DT_F32) {
        float *pg = (float *)pv.pages + tile * (kBlock * kHeadDim);
#pragma unroll
        for (int r = 0; r < kBlock; ++r)
            if (r < rows) pg[r * kHeadDim + lane] = x[r];
    } else if constexpr (CDT == DT_BF16) {
        uint16_t *pg = (uint16_t *)pv.pages + tile * (kBlock * kHeadDim);
#pragma unroll
        for (int r = 0; r < kBlock; ++r)
            if (r < rows) pg[r * kHeadDim + lane] = (uint16_t)bf16_bits(x[r]);
    } else {
        float amax = 0.f;
#pragma unroll
        for (int r = 0; r < kBlock; ++r)
            if (r < rows) amax = fmaxf(amax, fabsf(x[r]));
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o));
        const float sc = amax / 127.0f;
        int8_t *pg = (int8_t *)pv.pages + tile * (kBlock * kHeadDim);
#pragma unroll
        for (int r = 0; r < kBlock; ++r)
            if (r < rows) pg[r * kHeadDim + lane] = (int8_t)quant(x[r], sc);
        if (lane == 0) pv.scales[tile] = sc;
    }
}

hipError_t launch_load_kv(const PoolView &pv, int sid, int layer, const float *kv, int n, hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    const dim3 grid((n + kBlock - 1) / kBlock, pv.KVH, 2);
    switch (pv.cache_dt) {
    case DT_F32: hipLaunchKernelGGL(k_load_kv<DT_F32>, grid, dim3(64), 0, stream, pv, sid, layer, kv, n); break;
    case DT_BF16: hipLaunchKernelGGL(k_load_kv<DT_BF16>, grid, dim3(64), 0, stream, pv, sid, layer, kv, n); break;
    case DT_I8: hipLaunchKernelGGL(k_load_kv<DT_I8>, grid, dim3(64), 0, stream, pv, sid, layer, kv, n); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

} // namespace xnp
