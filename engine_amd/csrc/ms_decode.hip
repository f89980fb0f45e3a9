// ms_decode.hip -- read side of the compression-aware path on gfx950:
//   * fused decompress + select + agg_sum (decompress_and_process_batch with
//     the select core feeding the agg_sum core, format.h:164-195,
//     select_compr.h:80-89, agg_sum_compr.h:57-71) for every format,
//   * decompression (morph_t<ve, uncompr_f, F>, morph.h:203-241),
//   * select's position list (select_compr.h:100-260) as count + compact.
//
// Mapping: a wave decodes a 512-value unit.  For a vertical-bit-packed
// layout with S lanes, thread t handles lane j = t % S and the 8 codes
// k = 8g .. 8g+7 with g = unit*(64/S) + t/S (values S*k + j).
#include <map>
#include <mutex>


#include "ms_lookback.hpp"
#include "ms_units.hpp"

namespace ms {

__global__ void k_fill_u64(uint64_t *p, uint64_t n, uint64_t v)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

int launch_fill_u64(uint64_t *p, uint64_t n, uint64_t v, hipStream_t s)
{
    if (n == 0) return MS_OK;
    hipLaunchKernelGGL(k_fill_u64, dim3(grid_for(n, WG * 4ull, 2048)), dim3(WG), 0, s, p, n, v);
    MS_HIP(hipGetLastError());
    return MS_OK;
}

// The meta of the uncompr_f column whose one value is at `value`, the sum of
// a column of format kind `of` (sizeCompr: agg_sum_compr.h:148-150 vs
// agg_sum_uncompr.h:126).
__device__ __forceinline__ void set_meta_one(uint64_t *value, uint32_t of)
{
    ms_dev_meta *om = (ms_dev_meta *)((uint8_t *)value - COL_META_BYTES);
    om->count = 1;
    om->size_used = 8;
    om->size_compr = of == MS_UNCOMPR ? 0 : 8;
    om->status = 0;
    for (int k = 0; k < 4; k++) om->aux[k] = 0;
}

// How a select + sum kernel ends.  Short columns run in one workgroup that
// also takes the raw rest and writes the result, since the second launch
// costs more than the sum (dynamic_vbp_f calls one after the other, two
// launches / one: 1000 values 5.8 / 3.5 us, 8192 5.7 / 4.1, 16384 6.1 / 6.0;
// delta_f at 16384 6.2 / 5.9).  Longer ones leave a partial sum per workgroup
// to k_sum_finish.  One word says which, so that the launches of longer sums
// carry no more arguments than their own: the address of the partial sums or
// of the result, SS_RESULT for the latter and SS_META if that is the value of
// a column (addresses have 57 bits at most).  48 bytes of arguments more in
// the two launches cost 0.6 to 0.9 us of 8 where the host is the slower side
// (100,000 values of static_vbp_f<20, 8>: 8.5 -> 9.1 us, now 8.4).
typedef uint64_t ss_end;
constexpr uint64_t SS_RESULT = 1ull << 63, SS_META = 1ull << 62;
constexpr uint64_t SS_SINGLE = 8192;
// Layouts read value by value (k_select_sum_generic) are bound by the reads
// themselves: beyond what one workgroup of their two launches takes, a second
// one is worth more than the launch (two launches / one: dynamic_vbp_f<64, 8,
// 1> 4096 values 12.4 / 10.2 us, 4608 9.2 / 11.2, 8192 12.6 / 18.3; for_f over
// uncompr_f 4096 14.9 / 12.4, 4608 10.8 / 13.7, 8192 15.2 / 22.8).
constexpr uint64_t SS_SINGLE_GENERIC = WG * 16;

__device__ __forceinline__ void ss_finish(const ms_colv &c, const ms_pred &p, ss_end end, uint64_t acc)
{
    uint64_t *dst = (uint64_t *)(end & ~(SS_RESULT | SS_META));
    if ((end & SS_RESULT) && c.g.kind != MS_UNCOMPR && c.g.kind != MS_RLE) {
        const ms_parts pt = parts_of(c);
        const uint64_t *x = (const uint64_t *)(c.data + pt.rest_off);
        for (uint64_t i = threadIdx.x; i < pt.n_rest; i += WG) acc += pred_eval(p, x[i]) ? x[i] : 0;
    }
    wg_partial(acc, dst);   // one workgroup: its sum is the result
    if ((end & SS_META) && threadIdx.x == 0) set_meta_one(dst, c.g.kind);
}

// One wave decodes one 512-value unit per iteration (grid-stride); the
// next unit's index entry is fetched one iteration ahead.  Unit -> block
// and block -> for_f block are shifts (the host only takes this path when
// the ratios are powers of two).  dynamic_vbp takes its per-bit-width
// predicate from a table built on the host; for_f specialises it per block
// around the block's reference value.
template <bool IS_FOR, bool LEFORM>
__global__ __launch_bounds__(WG) void k_select_sum_blocks(ms_colv c, ms_pred p, ms_bwtab tab, ss_end end)
{
    const ms_parts pt = parts_of(c);
    const uint32_t lg_spb = c.g.lg_spb;
    const uint32_t lg_ipo = c.g.lg_ipo;
    const uint64_t n = pt.n_compr >> 9;
    const uint64_t nq = (n + 3) >> 2;   // groups of 4 units
    const uint32_t t = threadIdx.x & 63;
    const uint32_t j = t & 7, gl = t >> 3;
    const uint64_t W = (uint64_t)gridDim.x * WAVES;
    const uint64_t mask = (1ull << lg_spb) - 1ull;
    uint64_t acc = 0;
    uint64_t q = (uint64_t)blockIdx.x * WAVES + wave_index();
    // lanes 0..3 hold the group's index entries (and for_f references),
    // requested one group ahead
    uint64_t my_e = 0, my_r = 0;
    if (q < nq && t < 4 && q * 4 + t < n) {
        my_e = gload(c.index + ((q * 4 + t) >> lg_spb));
        if (IS_FOR) my_r = gload(c.refs + (((q * 4 + t) >> lg_spb) >> lg_ipo));
    }
    for (; q < nq; q += W) {
        const uint64_t u0 = q * 4;
        const uint32_t cnt = n - u0 < 4 ? (uint32_t)(n - u0) : 4u;
        uint64_t e[4], r[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            e[u] = readlane64(my_e, u);
            r[u] = IS_FOR ? readlane64(my_r, u) : 0ull;
        }
        const uint64_t un = u0 + 4 * W + t;
        my_e = my_r = 0;
        if (q + W < nq && t < 4 && un < n) {
            my_e = gload(c.index + (un >> lg_spb));
            if (IS_FOR) my_r = gload(c.refs + ((un >> lg_spb) >> lg_ipo));
        }
        vbp_units_ss<IS_FOR, LEFORM>(c.data, e, r, cnt, u0, mask, p, tab, j, gl, acc);
    }
    ss_finish(c, p, end, acc);
}

// static_vbp_f<vbp_l<BW, S>> with 64 % S == 0.
template <int BW>
__global__ __launch_bounds__(WG) void k_select_sum_static(ms_colv c, ms_pred p, ss_end end)
{
    const ms_parts pt = parts_of(c);
    const uint32_t S = c.g.lanes, lgS = c.g.lg_lanes;
    const uint64_t gpu = 64 >> lgS;
    const uint64_t ngroups = pt.n_compr >> (lgS + 3);
    const uint64_t nunits = (ngroups + gpu - 1) >> (6 - lgS);
    const uint32_t t = threadIdx.x & 63;
    const uint32_t j = t & (S - 1);
    const uint64_t maxcode = BW >= 64 ? ~0ull : (1ull << BW) - 1ull;
    const ms_cpred cp = code_pred(p, 0, maxcode);
    const uint64_t nwaves = (uint64_t)gridDim.x * WAVES;
    uint64_t acc = 0;
    if (cp.mode != PM_NONE) {
        const uint64_t *base = (const uint64_t *)c.data;
        uint64_t u = (uint64_t)blockIdx.x * WAVES + wave_index();
        // four units a step, every unit's words requested before the first is cut
        constexpr int NW = vbp_traits<BW>::NW;
        for (; u + 3 * nwaves < nunits; u += 4 * nwaves) {
            uint64_t w0[NW], w1[NW], w2[NW], w3[NW];   // named arrays: they stay in registers
            uint32_t s0 = 0, s1 = 0, s2 = 0, s3 = 0;
            const uint64_t g0 = u * gpu + (t >> lgS), g1 = g0 + nwaves * gpu, g2 = g1 + nwaves * gpu,
                           g3 = g2 + nwaves * gpu;
            if (g0 < ngroups) vbp_load<BW>(base, S, j, g0, w0, s0);
            if (g1 < ngroups) vbp_load<BW>(base, S, j, g1, w1, s1);
            if (g2 < ngroups) vbp_load<BW>(base, S, j, g2, w2, s2);
            if (g3 < ngroups) vbp_load<BW>(base, S, j, g3, w3, s3);
            if (g0 < ngroups) ss_loaded<BW>(w0, s0, cp, 0, acc);
            if (g1 < ngroups) ss_loaded<BW>(w1, s1, cp, 0, acc);
            if (g2 < ngroups) ss_loaded<BW>(w2, s2, cp, 0, acc);
            if (g3 < ngroups) ss_loaded<BW>(w3, s3, cp, 0, acc);
        }
        for (; u < nunits; u += nwaves) {
            const uint64_t g = u * gpu + (t >> lgS);
            if (g < ngroups) ss_unit<BW>(base, S, j, g, cp, 0, acc);
        }
    }
    ss_finish(c, p, end, acc);
}

// Uncompressed values: the whole of an uncompr_f column, or the rest part.
__global__ __launch_bounds__(WG) void k_select_sum_uncompr(ms_colv c, ms_pred p, ss_end end)
{
    const ms_parts pt = parts_of(c);
    const uint64_t *x = (const uint64_t *)(c.data + pt.rest_off);
    const uint64_t n = pt.n_rest;
    uint64_t acc = 0;
    const uint64_t stride = (uint64_t)gridDim.x * WG;
    uint64_t i = (uint64_t)blockIdx.x * WG + threadIdx.x;
    for (; 2 * i + 1 < n; i += stride) {
        const u64x2 v = __builtin_nontemporal_load((const u64x2 *)x + i);
        acc += pred_eval(p, v.x) ? v.x : 0;
        acc += pred_eval(p, v.y) ? v.y : 0;
    }
    if (2 * i < n && 2 * i + 1 == n) {
        const uint64_t v = x[2 * i];
        acc += pred_eval(p, v) ? v : 0;
    }
    ss_finish(c, p, end, acc);
}

// *d_n decompressed values.
__global__ __launch_bounds__(WG) void k_select_sum_values(const uint64_t *x, const uint64_t *d_n, ms_pred p,
                                                          uint64_t *res)
{
    const uint64_t n = *d_n;
    uint64_t acc = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * WG + threadIdx.x; i < n; i += (uint64_t)gridDim.x * WG)
        acc += pred_eval(p, x[i]) ? x[i] : 0ull;
    wg_partial(acc, res);
}

// Any layout readable by read_compr, one value per thread.
__global__ __launch_bounds__(WG) void k_select_sum_generic(ms_colv c, ms_pred p, ss_end end)
{
    const ms_parts pt = parts_of(c);
    uint64_t acc = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * WG + threadIdx.x; i < pt.n_compr; i += (uint64_t)gridDim.x * WG) {
        const uint64_t x = read_compr(c, i);
        if (pred_eval(p, x)) acc += x;
    }
    ss_finish(c, p, end, acc);
}

// rle_f: a run of `len` copies of v contributes len * v when v passes.
static constexpr uint64_t RLE_CHUNK = 512;   // runs per wave and step

__global__ __launch_bounds__(WG) void k_select_sum_rle(ms_colv c, ms_pred p, ss_end end)
{
    const uint64_t runs = c.meta->size_used / 16;
    const u64x2 *w = (const u64x2 *)c.data;
    const uint64_t nch = (runs + RLE_CHUNK - 1) / RLE_CHUNK;
    const uint64_t W = (uint64_t)gridDim.x * WAVES;
    const uint32_t t = threadIdx.x & 63;
    uint64_t acc = 0;
    for (uint64_t ch = (uint64_t)blockIdx.x * WAVES + wave_index(); ch < nch; ch += W) {
        const uint64_t r0 = ch * RLE_CHUNK, r1 = r0 + RLE_CHUNK < runs ? r0 + RLE_CHUNK : runs;
        acc += rle_runs_ss(w, r0, r1, p, t);
    }
    ss_finish(c, p, end, acc);
}

// ------------------------------------------------------------------
// delta_f: x = lane-wise running sum of the decoded deltas (delta.h:
// 229-261).  The column's derived index holds, per 2048-value tile, the
// running sums of the S lanes at the tile's start (its "carries"), so every
// tile decodes independently: a workgroup (4 waves x 512 values) scans its
// tile locally and adds the carries.  SRC 0 decodes 8-lane indexed blocks,
// SRC 1 reads deltas already decoded into `arr`, whose n need not end with a
// unit of 512 (blocks of fewer values).
// ------------------------------------------------------------------
static constexpr uint64_t DELTA_TILE = MS_DELTA_TILE;
static_assert(MS_DELTA_TILE == WAVES * 512, "a delta tile is one workgroup's 4 units");

template <int SRC>
// e_v: unit u's index entry (SRC 0), loaded by the caller.
__device__ __forceinline__ void delta_load(const ms_colv &c, const uint64_t *arr, uint64_t n, uint64_t u,
                                           uint64_t nunits, uint32_t S, uint32_t j, uint32_t gl, uint64_t e_v,
                                           uint64_t (&d)[8])
{
    if (u >= nunits) {
#pragma unroll
        for (int m = 0; m < 8; m++) d[m] = 0;
        return;
    }
    if (SRC == 0) {
        const uint64_t sub = u & ((1ull << c.g.lg_spb) - 1);
        const uint64_t e = uniform64(e_v);
        dec_dispatch((uint32_t)(e & 0xff), (const uint64_t *)(c.data + (e >> 8)), 8, j, sub * 8 + gl, d);
    } else {
        const uint64_t *a = arr + u * 512;
        if ((u + 1) * 512 <= n) {
#pragma unroll
            for (int m = 0; m < 8; m++) d[m] = a[S * (8 * gl + m) + j];
        } else {
            const uint32_t left = (uint32_t)(n - u * 512);
#pragma unroll
            for (int m = 0; m < 8; m++) d[m] = S * (8 * gl + m) + j < left ? a[S * (8 * gl + m) + j] : 0;
        }
    }
}

// Lane-wise scan of one 2048-value tile: returns, per thread, the
// exclusive prefix of its 8 values inside the tile (d[] becomes the
// inclusive prefix within the thread).  tile_tot receives lane j's total.
__device__ __forceinline__ uint64_t delta_tile_scan(uint64_t (&d)[8], uint32_t S, uint32_t j, uint32_t t,
                                                    uint32_t wv, uint64_t (*s_wtot)[8], uint64_t &tile_tot)
{
#pragma unroll
    for (int m = 1; m < 8; m++) d[m] += d[m - 1];
    const uint64_t tot = d[7];
    uint64_t incl = tot;
    for (uint32_t o = S; o < 64; o <<= 1) {
        const uint64_t v = __shfl_up(incl, o, MS_WAVE);
        if (t >= o) incl += v;
    }
    if (t >= 64 - S) s_wtot[wv][j] = incl;
    __syncthreads();
    uint64_t wpre = 0;
    tile_tot = 0;
    for (uint32_t w = 0; w < WAVES; w++) {
        const uint64_t v = s_wtot[w][j];
        if (w < wv) wpre += v;
        tile_tot += v;
    }
    __syncthreads();
    return wpre + incl - tot;
}

// MODE 0 writes x, MODE 1 folds select + sum into per-workgroup partials.
template <int MODE, int SRC>
__global__ __launch_bounds__(WG) void k_delta_tiles(ms_colv c, const uint64_t *arr, uint64_t *out, ms_pred p,
                                                    uint64_t *part)
{
    __shared__ uint64_t s_wtot[WAVES][8];
    const ms_parts pt = parts_of(c);
    const uint32_t S = c.g.dstep;
    const uint64_t nunits = (pt.n_compr + 511) >> 9;   // SRC 0: all of them full
    const uint64_t ntiles = (nunits + WAVES - 1) / WAVES;
    const uint32_t wv = wave_index();
    const uint32_t t = threadIdx.x & 63;
    const uint32_t j = t & (S - 1), gl = t >> c.g.lg_dstep;
    uint64_t acc = 0;
    // SRC 0: each unit's index entry is requested one tile ahead
    uint64_t e_n = 0;
    if (SRC == 0 && blockIdx.x * WAVES + wv < nunits) e_n = gload(c.index + ((blockIdx.x * WAVES + wv) >> c.g.lg_spb));
    for (uint64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const uint64_t u = tile * WAVES + wv;
        const uint64_t carry = gload(c.refs + tile * 8 + j);   // needed after the scan: requested first
        const uint64_t e_v = e_n;
        const uint64_t un = (tile + gridDim.x) * WAVES + wv;
        if (SRC == 0) e_n = un < nunits ? gload(c.index + (un >> c.g.lg_spb)) : 0ull;
        uint64_t d[8];
        delta_load<SRC>(c, arr, pt.n_compr, u, nunits, S, j, gl, e_v, d);
        uint64_t tile_tot;
        const uint64_t base = carry + delta_tile_scan(d, S, j, t, wv, s_wtot, tile_tot);
        if (u < nunits) {
            const uint32_t left = SRC == 0 || (u + 1) * 512 <= pt.n_compr ? 512u : (uint32_t)(pt.n_compr - u * 512);
            if (MODE == 0) {
                uint64_t *o = out + u * 512;
                if (left == 512) {
#pragma unroll
                    for (int m = 0; m < 8; m++) o[S * (8 * gl + m) + j] = base + d[m];
                } else {
#pragma unroll
                    for (int m = 0; m < 8; m++)
                        if (S * (8 * gl + m) + j < left) o[S * (8 * gl + m) + j] = base + d[m];
                }
            } else {
#pragma unroll
                for (int m = 0; m < 8; m++) {
                    const uint64_t x = base + d[m];
                    acc += S * (8 * gl + m) + j < left && pred_eval(p, x) ? x : 0;
                }
            }
        }
    }
    if (MODE == 1) wg_partial(acc, part);
}

// Select + sum over a delta_f column with 8 lanes and indexed 8-lane
// inner blocks: one wave per tile, no workgroup synchronisation.
__global__ __launch_bounds__(WG) void k_delta_select_sum(ms_colv c, ms_pred p, ss_end end)
{
    const ms_parts pt = parts_of(c);
    const uint64_t nunits = pt.n_compr >> 9;
    const uint64_t ntiles = (nunits + 3) >> 2;
    const uint32_t t = threadIdx.x & 63;
    const uint32_t j = t >> 3, gl = t & 7;   // delta lane j in 8 consecutive threads
    const uint64_t W = (uint64_t)gridDim.x * WAVES;
    uint64_t acc = 0;
    uint64_t tile = (uint64_t)blockIdx.x * WAVES + wave_index();
    // each tile's index entries are requested one tile ahead
    uint64_t my_e = tile < ntiles ? delta_tile_entries(c.index, c.g.lg_spb, tile, nunits, t) : 0ull;
    for (; tile < ntiles; tile += W) {
        const uint64_t e_next =
            tile + W < ntiles ? delta_tile_entries(c.index, c.g.lg_spb, tile + W, nunits, t) : 0ull;
        delta_tile_ss<false>(c.data, my_e, c.refs, c.g.lg_spb, p, tile, nunits, t, j, gl, acc);
        my_e = e_next;
    }
    ss_finish(c, p, end, acc);
}

// Per-tile lane totals, lane-major: sums[j * ntb + tile].
template <int SRC>
__global__ __launch_bounds__(WG) void k_delta_tile_sums(ms_colv c, const uint64_t *arr, uint64_t *sums, uint64_t ntb)
{
    __shared__ uint64_t s_wtot[WAVES][8];
    const ms_parts pt = parts_of(c);
    const uint32_t S = c.g.dstep;
    const uint64_t nunits = (pt.n_compr + 511) >> 9;
    const uint32_t wv = wave_index();
    const uint32_t t = threadIdx.x & 63;
    const uint32_t j = t & (S - 1), gl = t >> c.g.lg_dstep;
    for (uint64_t tile = blockIdx.x; tile < ntb; tile += gridDim.x) {
        const uint64_t u = tile * WAVES + wv;
        const uint64_t e_v = SRC == 0 && u < nunits ? gload(c.index + (u >> c.g.lg_spb)) : 0ull;
        uint64_t d[8];
        delta_load<SRC>(c, arr, pt.n_compr, u, nunits, S, j, gl, e_v, d);
        uint64_t tile_tot;
        (void)delta_tile_scan(d, S, j, t, wv, s_wtot, tile_tot);
        if (threadIdx.x < S) sums[(uint64_t)threadIdx.x * ntb + tile] = tile_tot;
    }
}

__global__ __launch_bounds__(WG) void k_delta_carries(const uint64_t *scan, uint64_t ntb, uint32_t S, uint64_t *refs)
{
    for (uint64_t i = (uint64_t)blockIdx.x * WG + threadIdx.x; i < ntb * 8; i += (uint64_t)gridDim.x * WG) {
        const uint64_t tile = i / 8, j = i % 8;
        refs[i] = j < S ? scan[j * ntb + tile] : 0;
    }
}

// ------------------------------------------------------------------
// Decompression kernels.
// ------------------------------------------------------------------
// 8-lane indexed layouts (dynamic_vbp_f, for_f's inner blocks) and
// static_vbp_f<vbp_l<bw, 8>> (LAYOUT 2: unit u's payload is 64 bw bytes at
// u * 64 bw, no index): one resident wave of workgroups, grid-stride over
// groups of 4 units; a group's index entries (and for_f references) are
// loaded lane-parallel one group ahead, and its 4 units' words are all
// requested before the first is decoded.
enum { DL_BLOCKS = 0, DL_FOR = 1, DL_STATIC8 = 2 };

// The end of a decompression kernel: the raw rest behind the compressed
// part (grid-stride), and, when om is given, the output column's whole
// meta (count, 8 bytes a value, status and append slots cleared).
__device__ __forceinline__ void decomp_tail(const ms_colv &c, const ms_parts &pt, uint64_t *out, ms_dev_meta *om)
{
    const uint64_t *rx = (const uint64_t *)(c.data + pt.rest_off);
    for (uint64_t i = (uint64_t)blockIdx.x * WG + threadIdx.x; i < pt.n_rest; i += (uint64_t)gridDim.x * WG)
        out[pt.n_compr + i] = gload(rx + i);
    if (om && blockIdx.x == 0 && threadIdx.x == 0) {
        om->count = pt.n;
        om->size_used = 8 * pt.n;
        om->size_compr = 0;
        om->status = 0;
        for (int k = 0; k < 4; k++) om->aux[k] = 0;
    }
}

__global__ void k_set_meta_uncompr(const ms_dev_meta *in, ms_dev_meta *om)
{
    const uint64_t n = in->count;
    om->count = n;
    om->size_used = 8 * n;
    om->size_compr = 0;
    om->status = 0;
    for (int k = 0; k < 4; k++) om->aux[k] = 0;
}

template <int LAYOUT, bool NT>
__global__ __launch_bounds__(WG) void k_decomp_units(ms_colv c, uint64_t *out, ms_dev_meta *om)
{
    const ms_parts pt = parts_of(c);
    const uint32_t lg_spb = LAYOUT == DL_STATIC8 ? 0 : c.g.lg_spb;
    const uint32_t lg_ipo = c.g.lg_ipo;
    const uint64_t n = pt.n_compr >> 9;
    const uint64_t nq = (n + 3) >> 2;
    const uint32_t t = threadIdx.x & 63;
    const uint32_t j = t & 7, gl = t >> 3;
    const uint64_t W = (uint64_t)gridDim.x * WAVES;
    const uint64_t mask = (1ull << lg_spb) - 1ull;
    const uint64_t bw8 = c.g.bw;
    uint64_t q = (uint64_t)blockIdx.x * WAVES + wave_index();
    const auto entry = [&](uint64_t u, uint64_t &e, uint64_t &r) {
        e = r = 0;
        if (LAYOUT == DL_STATIC8) return;
        e = gload(c.index + (u >> lg_spb));
        if (LAYOUT == DL_FOR) r = gload(c.refs + ((u >> lg_spb) >> lg_ipo));
    };
    uint64_t my_e = 0, my_r = 0;
    if (q < nq && t < 4 && q * 4 + t < n) entry(q * 4 + t, my_e, my_r);
    for (; q < nq; q += W) {
        const uint64_t u0 = q * 4;
        const uint32_t cnt = n - u0 < 4 ? (uint32_t)(n - u0) : 4u;
        uint64_t e[4], r[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            if (LAYOUT == DL_STATIC8) {
                e[u] = (((u0 + u) * 64ull * bw8) << 8) | bw8;
                r[u] = 0;
            } else {
                e[u] = readlane64(my_e, u);
                r[u] = LAYOUT == DL_FOR ? readlane64(my_r, u) : 0ull;
            }
        }
        const uint64_t un = u0 + 4 * W + t;
        my_e = my_r = 0;
        if (q + W < nq && t < 4 && un < n) entry(un, my_e, my_r);
        dec_units<NT>(c.data, e, r, cnt, u0, mask, j, gl, out);
    }
    decomp_tail(c, pt, out, om);
}

// delta_f with 8 lanes over indexed 8-lane inner blocks: one wave per
// 2048-value tile (lane-major threads, 8 per delta lane), the tile's index
// entries requested one tile ahead.
template <bool NT>
__global__ __launch_bounds__(WG) void k_delta_decomp(ms_colv c, uint64_t *out, ms_dev_meta *om)
{
    const ms_parts pt = parts_of(c);
    const uint64_t nunits = pt.n_compr >> 9;
    const uint64_t ntiles = (nunits + 3) >> 2;
    const uint32_t t = threadIdx.x & 63;
    const uint32_t j = t >> 3, gl = t & 7;
    const uint64_t W = (uint64_t)gridDim.x * WAVES;
    uint64_t tile = (uint64_t)blockIdx.x * WAVES + wave_index();
    uint64_t my_e = tile < ntiles ? delta_tile_entries(c.index, c.g.lg_spb, tile, nunits, t) : 0ull;
    for (; tile < ntiles; tile += W) {
        const uint64_t e_next =
            tile + W < ntiles ? delta_tile_entries(c.index, c.g.lg_spb, tile + W, nunits, t) : 0ull;
        delta_tile_store<NT>(c.data, my_e, c.refs, c.g.lg_spb, tile, nunits, t, j, gl, out);
        my_e = e_next;
    }
    decomp_tail(c, pt, out, om);
}

template <int BW>
__global__ __launch_bounds__(WG) void k_decomp_static(ms_colv c, uint64_t *out)
{
    const ms_parts pt = parts_of(c);
    const uint32_t S = c.g.lanes, lgS = c.g.lg_lanes;
    const uint64_t gpu = 64 >> lgS;
    const uint64_t ngroups = pt.n_compr >> (lgS + 3);
    const uint64_t nunits = (ngroups + gpu - 1) >> (6 - lgS);
    const uint32_t t = threadIdx.x & 63;
    const uint32_t j = t & (S - 1);
    const uint64_t nwaves = (uint64_t)gridDim.x * WAVES;
    for (uint64_t u = (uint64_t)blockIdx.x * WAVES + wave_index(); u < nunits; u += nwaves) {
        const uint64_t g = u * gpu + (t >> lgS);
        if (g >= ngroups) continue;
        uint64_t d[8];
        dec_unit<BW>((const uint64_t *)c.data, S, j, g, d);
#pragma unroll
        for (int m = 0; m < 8; m++) out[S * (8 * g + m) + j] = d[m];
    }
}

// read_compr per value: the fallback for every other layout (and deltas
// of a delta_f whose inner format is not an 8-lane indexed layout).
__global__ __launch_bounds__(WG) void k_decomp_generic(ms_colv c, uint64_t *out)
{
    const ms_parts pt = parts_of(c);
    for (uint64_t i = (uint64_t)blockIdx.x * WG + threadIdx.x; i < pt.n_compr; i += (uint64_t)gridDim.x * WG)
        out[i] = read_compr(c, i);
}

__global__ __launch_bounds__(WG) void k_copy_rest(ms_colv c, uint64_t *out)
{
    const ms_parts pt = parts_of(c);
    const uint64_t *x = (const uint64_t *)(c.data + pt.rest_off);
    for (uint64_t i = (uint64_t)blockIdx.x * WG + threadIdx.x; i < pt.n_rest; i += (uint64_t)gridDim.x * WG)
        out[pt.n_compr + i] = x[i];
}

// rle_f expansion by output tiles of RLE_XT values, a wave per tile, so that
// neither short nor long runs leave lanes or waves idle (a wave per chunk of
// runs wrote one run at a time with half-empty stores, and a column of few
// runs with a few waves).  k_rle_starts sums the lengths of every chunk of
// 64 runs, places the chunks by a look-back and notes for every output tile
// the chunk that holds its first value.  k_rle_expand then takes a tile's
// runs 64 at a time: their heads become bits of a bitmap of the tile, and a
// value's run is the number of heads up to it.
// Bound by the output's stores.  Measured for 5 10^7 values in runs of 64 on
// average, the kernels before and now: 169 -> 97 us; 2^26 values in one
// run 26.2 ms -> 117 us, 2^25 runs of one value 1.57 ms -> 0.36 ms.
constexpr uint32_t RLE_XCH = 64;        // runs per chunk
constexpr uint32_t RLE_XT = 2048;       // values per output tile
constexpr uint32_t RLE_SCH = 64;        // chunks per tile of k_rle_starts
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Clears the look-back state and sets the expanded column's meta.
__global__ __launch_bounds__(WG) void k_rle_begin(const ms_dev_meta *in, uint64_t *state, uint64_t words,
                                                  ms_dev_meta *om)
{
    for (uint64_t i = (uint64_t)blockIdx.x * WG + threadIdx.x; i < words; i += (uint64_t)gridDim.x * WG) state[i] = 0;
    if (om && blockIdx.x == 0 && threadIdx.x == 0) {
        const uint64_t n = in->count;
        om->count = n;
        om->size_used = 8 * n;
        om->size_compr = 0;
        om->status = 0;
        for (int k = 0; k < 4; k++) om->aux[k] = 0;
    }
}

// cstart[ch]: the first value of chunk ch; tchunk[b]: the chunk that holds
// value b RLE_XT.
__global__ __launch_bounds__(WG) void k_rle_starts(ms_colv c, uint64_t *state, uint64_t *cstart, uint32_t *tchunk,
                                                   uint64_t tiles_bound)
{
    constexpr uint32_t PER = RLE_SCH / WAVES;   // chunks per wave
    __shared__ uint64_t s_len[RLE_SCH], s_start[RLE_SCH], s_ticket;
    __shared__ unsigned long long s_many;
    const uint64_t runs = c.meta->size_used / 16;
    const uint64_t nch = (runs + RLE_XCH - 1) / RLE_XCH, nst = (nch + RLE_SCH - 1) / RLE_SCH;
    const uint32_t t = threadIdx.x & 63, w = wave_index();
    const uint64_t *pairs = (const uint64_t *)c.data;
    if (blockIdx.x >= nst) return;   // as many workgroups as tiles take tickets
    for (;;) {
        if (threadIdx.x == 0) s_ticket = lb_ticket(state);
        __syncthreads();
        const uint64_t st = readlane64(s_ticket, 0);
        if (st >= nst) return;
        uint64_t len[PER];
#pragma unroll
        for (uint32_t i = 0; i < PER; i++) {
            const uint64_t r = (st * RLE_SCH + w * PER + i) * RLE_XCH + t;
            len[i] = r < runs ? gload(pairs + 2 * r + 1) : 0ull;
        }
#pragma unroll
        for (uint32_t i = 0; i < PER; i++) {
            const uint64_t sum = dpp_scan_u64(len[i]);
            if (t == 63) s_len[w * PER + i] = sum;
        }
        if (threadIdx.x == 0) s_many = 0;
        __syncthreads();
        if (w == 0) {
            const uint64_t v = s_len[t], incl = dpp_scan_u64(v);
            const uint64_t total = readlane64(incl, 63) & LB_VALUE;
            uint64_t words[LB_SPAN];
            lb_publish(state + 1, st, total);
            lb_request(state + 1, (int64_t)st - 1, words);
            const uint64_t start = lb_exclusive(state + 1, st, total, words) + incl - v;
            s_start[t] = start;
            const uint64_t ch = st * RLE_SCH + t;
            if (ch < nch) cstart[ch] = start;
        }
        __syncthreads();
        // four threads per chunk note its tiles; a chunk of long runs is
        // left to all of them
        static_assert(WG == 4 * RLE_SCH, "four threads per chunk");
        const auto tiles_of = [&](uint32_t k, uint64_t &b0, uint64_t &b1) {
            b0 = (s_start[k] + RLE_XT - 1) / RLE_XT;
            b1 = (s_start[k] + s_len[k] + RLE_XT - 1) / RLE_XT;
            if (b1 > tiles_bound) b1 = tiles_bound;
        };
        uint64_t b0, b1;
        tiles_of(threadIdx.x / 4, b0, b1);
        const bool many = b1 > b0 && b1 - b0 > 64;
        if (!many)
            for (uint64_t b = b0 + threadIdx.x % 4; b < b1; b += 4)
                tchunk[b] = (uint32_t)(st * RLE_SCH + threadIdx.x / 4);
        if (threadIdx.x % 4 == 0 && many) atomicOr(&s_many, 1ull << (threadIdx.x / 4));
        __syncthreads();
        for (uint64_t left = readlane64(s_many, 0); left; left &= left - 1) {
            const uint32_t k = (uint32_t)__builtin_ctzll(left);
            tiles_of(k, b0, b1);
            for (uint64_t b = b0 + threadIdx.x; b < b1; b += WG) tchunk[b] = (uint32_t)(st * RLE_SCH + k);
        }
        __syncthreads();   // s_ticket, s_len and s_start are rewritten
    }
}

template <bool NT>
__global__ __launch_bounds__(WG) void k_rle_expand(ms_colv c, const uint64_t *cstart, const uint32_t *tchunk,
                                                   uint64_t *out)
{
    __shared__ uint64_t s_val[WAVES][RLE_XCH];
    __shared__ uint32_t s_bits[WAVES][RLE_XT / 32];
    __shared__ u32x2 s_word[WAVES][RLE_XT / 32];   // a word of the bitmap and the heads before it
    static_assert(RLE_XT / 32 == 64, "a word of the bitmap per lane");
    const uint64_t runs = c.meta->size_used / 16, n = c.meta->count;
    const uint64_t nch = (runs + RLE_XCH - 1) / RLE_XCH, nt = (n + RLE_XT - 1) / RLE_XT;
    const u64x2 *pairs = (const u64x2 *)c.data;
    const uint32_t t = threadIdx.x & 63, w = wave_index();
    for (uint64_t b = (uint64_t)blockIdx.x * WAVES + w; b < nt; b += (uint64_t)gridDim.x * WAVES) {
        const uint64_t o0 = b * RLE_XT;
        const uint32_t size = n - o0 < RLE_XT ? (uint32_t)(n - o0) : RLE_XT;   // writes stay inside the tile
        uint64_t ch = __builtin_amdgcn_readfirstlane(gload(tchunk + b));
        if (ch >= nch) continue;                     // lengths that end before the count
        uint64_t pos = uniform64(gload(cstart + ch));
        for (; ch < nch; ch++) {
            const uint64_t r = ch * RLE_XCH + t;
            const u64x2 vl = r < runs ? gload(pairs + r) : u64x2{0, 0};
            s_bits[w][t] = 0;
            const uint64_t end = pos + dpp_scan_u64(vl.y), start = end - vl.y;
            const bool in = vl.y && end > o0 && start < o0 + size;
            const uint64_t m = __ballot(in);
            pos = readlane64(end, 63);
            if (m == 0) {
                if (pos >= o0 + size) break;
                continue;
            }
            wave_lds_sync();
            const uint32_t p0 = start > o0 ? (uint32_t)(start - o0) : 0u;
            if (in) {
                const uint32_t k = lanes_below(m);
                s_val[w][k] = vl.x;
                atomicOr(&s_bits[w][p0 >> 5], 1u << (p0 & 31));
            }
            // the values this batch writes: [lo, hi) of the tile
            const uint32_t lo = __builtin_amdgcn_readlane(p0, __builtin_ctzll(m));
            const uint32_t hi = pos - o0 < size ? (uint32_t)(pos - o0) : size;
            wave_lds_sync();
            const uint32_t bits = s_bits[w][t];
            const uint32_t own = (uint32_t)__builtin_popcount(bits);
            const uint32_t heads = dpp_scan_u32(own, op_add{});
            s_word[w][t] = u32x2{bits, heads - own};
            wave_lds_sync();
            for (uint32_t row = lo / 128; row * 128 < hi; row++) {
                const uint32_t p = row * 128 + 2 * t;
                const u32x2 wd = s_word[w][p >> 5];
                const uint32_t sh = p & 31;
                // heads up to p, up to p + 1: at least one for p >= lo
                const uint32_t ka = wd.y + (uint32_t)__builtin_popcount(wd.x & ((2u << sh) - 1u));
                const uint32_t kb = ka + ((wd.x >> sh) >> 1 & 1u);
                u64x2 v;
                v.x = s_val[w][(ka - 1) & (RLE_XCH - 1)];
                v.y = s_val[w][(kb - 1) & (RLE_XCH - 1)];
                uint64_t *o = out + o0 + p;
                if (p >= lo && p + 1 < hi) {
                    if (NT) __builtin_nontemporal_store(v, (u64x2 *)o);
                    else *(u64x2 *)o = v;
                } else {
                    if (p >= lo && p < hi) *o = v.x;
                    if (p + 1 >= lo && p + 1 < hi) o[1] = v.y;
                }
            }
            if (pos >= o0 + size) break;
            wave_lds_sync();
        }
    }
}

// ------------------------------------------------------------------
// Host launchers
// ------------------------------------------------------------------
static bool fast_blocks(const ms_colv &v)
{
    // 8-lane indexed layouts whose blocks hold a power-of-two multiple of
    // 512 values (and, for cascades, a power-of-two number of blocks per
    // outer block)
    return (v.g.kind == MS_DYNAMIC_VBP || v.g.kind == MS_FOR || v.g.kind == MS_DELTA) &&
           v.g.leaf == MS_DYNAMIC_VBP && v.g.lanes == 8 && v.g.lg_spb != 0xff &&
           (v.g.kind == MS_DYNAMIC_VBP || v.g.lg_ipo != 0xff);
}

static bool fast_static(const ms_colv &v)
{
    return v.g.kind == MS_STATIC_VBP && v.g.lg_lanes != 0xff && v.g.lanes <= 64;
}

typedef void (*static_kernel_t)(ms_colv, ms_pred, ss_end);
typedef void (*static_dec_t)(ms_colv, uint64_t *);

static static_kernel_t static_sum_kernel(uint32_t bw)
{
    switch (bw) {
#define MS_CASE(B) \
    case B: return k_select_sum_static<B>;
        MS_BW_CASES(MS_CASE)
#undef MS_CASE
    default: return nullptr;
    }
}

static static_dec_t static_dec_kernel(uint32_t bw)
{
    switch (bw) {
#define MS_CASE(B) \
    case B: return k_decomp_static<B>;
        MS_BW_CASES(MS_CASE)
#undef MS_CASE
    default: return nullptr;
    }
}

__global__ void k_set_meta_one(uint64_t *value, uint32_t of) { set_meta_one(value, of); }

// Sums the per-workgroup partials and the uncompressed rest (select + sum
// over the rest part, the vectorised and scalar loops of
// agg_sum_compr.h:110-146 folded into one) and writes the result.
__global__ __launch_bounds__(WG) void k_sum_finish(ms_colv c, ms_pred p, const uint64_t *part, uint32_t nparts,
                                                   int with_rest, ss_end end)
{
    uint64_t acc = 0;
    for (uint32_t i = threadIdx.x; i < nparts; i += WG) acc += part[i];
    if (with_rest) {
        const ms_parts pt = parts_of(c);
        const uint64_t *x = (const uint64_t *)(c.data + pt.rest_off);
        for (uint64_t i = threadIdx.x; i < pt.n_rest; i += WG) acc += pred_eval(p, x[i]) ? x[i] : 0;
    }
    __shared__ uint64_t s_part[WAVES];
    acc = wave_sum_u64(acc);
    if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint64_t sum = 0;
        for (int w = 0; w < WAVES; w++) sum += s_part[w];
        uint64_t *result = (uint64_t *)(end & ~SS_META);
        *result = sum;
        if (end & SS_META) set_meta_one(result, c.g.kind);
    }
}

static bool delta_fast(const ms_colv &v) { return fast_blocks(v) && v.g.dstep == 8; }
static bool delta_shiftable(const ms_colv &v) { return v.g.lg_dstep != 0xff && v.g.dstep <= 8; }

// Deltas of a delta_f column whose inner layout has no fast decoder,
// decoded per value into a temporary.
static int delta_src(const ms_col *in, const ms_colv &v, temps &sc, const uint64_t **arr,
                     const ss_buffers *bufs = nullptr)
{
    *arr = nullptr;
    if (delta_fast(v)) return MS_OK;
    uint64_t *tmp;
    if (bufs) {
        if (in->count_bound > bufs->tmp_values)
            return ms_fail(MS_ERR_CAPACITY, "delta_f column of %llu values without a unit decoder exceeds the "
                           "%llu-value temporary of the caller's buffers",
                           (unsigned long long)in->count_bound, (unsigned long long)bufs->tmp_values);
        tmp = bufs->tmp;
    } else {
        tmp = (uint64_t *)sc.get(in->count_bound * 8 + 64);
    }
    if (!tmp) return ms_fail(MS_ERR_NOMEM, "delta scratch");
    hipLaunchKernelGGL(k_decomp_generic, dim3(grid_for(in->count_bound, WG * 8ull)), dim3(WG), 0, sc.s, v, tmp);
    MS_HIP(hipGetLastError());
    *arr = tmp;
    return MS_OK;
}

int launch_delta_carries(const ms_col *in, temps &sc)
{
    ms_colv v;
    MS_TRY(colv_of(in, v));
    const uint64_t ntb = in->count_bound / DELTA_TILE + 1;
    if (!in->refs || in->refs_cap < ntb * 8) return ms_fail(MS_ERR_CAPACITY, "delta carries capacity");
    const uint64_t *arr;
    MS_TRY(delta_src(in, v, sc, &arr));
    uint64_t *sums = (uint64_t *)sc.get(ntb * 8 * 8 + 64);
    uint64_t *scan = (uint64_t *)sc.get(ntb * 8 * 8 + 64);
    if (!sums || !scan) return ms_fail(MS_ERR_NOMEM, "delta carries scratch");
    const uint32_t S = in->g.dstep;
    const dim3 grid(grid_for(ntb, 1, 65536));
    if (arr) hipLaunchKernelGGL(k_delta_tile_sums<1>, grid, dim3(WG), 0, sc.s, v, arr, sums, ntb);
    else hipLaunchKernelGGL(k_delta_tile_sums<0>, grid, dim3(WG), 0, sc.s, v, arr, sums, ntb);
    MS_HIP(hipGetLastError());
    for (uint32_t j = 0; j < S; j++) MS_TRY(launch_exclusive_scan(sums + j * ntb, scan + j * ntb, ntb, sc));
    hipLaunchKernelGGL(k_delta_carries, dim3(grid_for(ntb * 8, WG)), dim3(WG), 0, sc.s, scan, ntb, S, in->refs);
    MS_HIP(hipGetLastError());
    return MS_OK;
}

static uint32_t units_grid(uint64_t count_bound) { return grid_for(count_bound / 512 + 1, WAVES * 8ull, 2048); }

// Occupancy per CU times CUs: grid-stride kernels that prefetch their next
// piece of work run best as one resident wave of workgroups.
uint32_t resident_grid(const void *kernel, uint32_t wg)
{
    static std::mutex mu;
    static std::map<std::pair<int, const void *>, uint32_t> cache;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 2048;
    std::lock_guard<std::mutex> lk(mu);
    const auto key = std::make_pair(dev, kernel);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    int cus = 0, blocks = 0;
    uint32_t g = 2048;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, kernel, (int)wg, 0) == hipSuccess && cus > 0 && blocks > 0)
        g = (uint32_t)(cus * blocks);
    cache[key] = g;
    return g;
}

// Grid of a grid-stride kernel over `items` pieces of one wave each.
static uint32_t stride_grid(const void *kernel, uint64_t items)
{
    const uint32_t r = resident_grid(kernel, WG);
    return grid_for(items, WAVES, r < 8192 ? r : 8192);
}

int launch_select_sum(const ms_col *in, const ms_pred &p, uint64_t *d_result, bool accumulate, hipStream_t s,
                      const ss_buffers *bufs, bool column)
{
    ms_colv v;
    MS_TRY(colv_of(in, v));
    if (v.g.kind == MS_BLOCKWISE_INDIVIDUAL) {
        if (bufs) return ms_fail(MS_ERR_INVALID, "blockwise_individual_f: select_sum needs temporaries of its own");
        MS_TRY(launch_bwi_select_sum(in, p, d_result, accumulate, s));
        if (column) hipLaunchKernelGGL(k_set_meta_one, dim3(1), dim3(1), 0, s, d_result, v.g.kind);
        MS_HIP(hipGetLastError());
        return MS_OK;
    }
    temps sc(s);
    const uint64_t nb = in->count_bound;
    uint32_t grid = 1;
    int with_rest = 1;
    // kinds whose kernels end with ss_finish (delta_f without a unit decoder
    // and the formats read through decompression leave partial sums)
    const bool ends = v.g.kind == MS_UNCOMPR || v.g.kind == MS_RLE || v.g.kind == MS_STATIC_VBP ||
                      v.g.kind == MS_DYNAMIC_VBP || v.g.kind == MS_FOR || (v.g.kind == MS_DELTA && delta_fast(v));
    const bool by_value = v.g.kind == MS_STATIC_VBP ? !fast_static(v)
                        : (v.g.kind == MS_DYNAMIC_VBP || v.g.kind == MS_FOR) && !fast_blocks(v);
    const bool single = ends && nb <= (by_value ? SS_SINGLE_GENERIC : SS_SINGLE);
    uint64_t *part = single ? nullptr : bufs ? bufs->part : (uint64_t *)sc.get(SS_MAX_PARTS * 8);
    if (!part && !single) return ms_fail(MS_ERR_NOMEM, "select_sum scratch");
    const ss_end meta = column ? SS_META : 0;
    const ss_end end = single ? (uint64_t)d_result | SS_RESULT | meta : (uint64_t)part;
    switch (v.g.kind) {
    case MS_UNCOMPR:
        grid = grid_for(nb, WG * 32ull, 2048);
        hipLaunchKernelGGL(k_select_sum_uncompr, dim3(single ? 1 : grid), dim3(WG), 0, s, v, p, end);
        with_rest = 0;
        break;
    case MS_RLE:
        grid = stride_grid((const void *)k_select_sum_rle, in->size_alloc / 16 / RLE_CHUNK + 1);
        hipLaunchKernelGGL(k_select_sum_rle, dim3(single ? 1 : grid), dim3(WG), 0, s, v, p, end);
        with_rest = 0;
        break;
    case MS_STATIC_VBP:
        if (fast_static(v)) {
            grid = units_grid(nb);
            hipLaunchKernelGGL(static_sum_kernel(v.g.bw), dim3(single ? 1 : grid), dim3(WG), 0, s, v, p, end);
        } else {
            grid = grid_for(nb, WG * 16ull, 2048);
            hipLaunchKernelGGL(k_select_sum_generic, dim3(single ? 1 : grid), dim3(WG), 0, s, v, p, end);
        }
        break;
    case MS_DYNAMIC_VBP:
    case MS_FOR:
        if (fast_blocks(v)) {
            const ms_bwtab tab = make_bwtab(p);
            const uint64_t quads = nb / 2048 + 1;   // groups of 4 units
            auto k = v.g.kind == MS_FOR && pred_le_form(p) ? k_select_sum_blocks<true, true>
                   : v.g.kind == MS_FOR                    ? k_select_sum_blocks<true, false>
                                                           : k_select_sum_blocks<false, false>;
            grid = stride_grid((const void *)k, quads);
            hipLaunchKernelGGL(k, dim3(single ? 1 : grid), dim3(WG), 0, s, v, p, tab, end);
        } else {
            grid = grid_for(nb, WG * 16ull, 2048);
            hipLaunchKernelGGL(k_select_sum_generic, dim3(single ? 1 : grid), dim3(WG), 0, s, v, p, end);
        }
        break;
    case MS_DELTA: {
        const uint64_t *arr;
        MS_TRY(delta_src(in, v, sc, &arr, bufs));
        if (!arr && v.g.lg_spb != 0xff) {
            grid = stride_grid((const void *)k_delta_select_sum, nb / DELTA_TILE + 1);
            hipLaunchKernelGGL(k_delta_select_sum, dim3(single ? 1 : grid), dim3(WG), 0, s, v, p, end);
            break;
        }
        grid = grid_for(nb / DELTA_TILE + 1, 2, 2048);
        if (arr) hipLaunchKernelGGL((k_delta_tiles<1, 1>), dim3(grid), dim3(WG), 0, s, v, arr, nullptr, p, part);
        else hipLaunchKernelGGL((k_delta_tiles<1, 0>), dim3(grid), dim3(WG), 0, s, v, arr, nullptr, p, part);
        break;
    }
    case MS_STATIC_VBP_PAD:
    case MS_K_WISE_NS:
    case MS_GROUP_SIMPLE: {
        // these layouts are read through decompression into a temporary
        uint64_t *tmp;
        if (bufs) {
            if (nb > bufs->tmp_values)
                return ms_fail(MS_ERR_CAPACITY, "a column of %llu values exceeds the %llu-value temporary of the "
                               "caller's buffers", (unsigned long long)nb, (unsigned long long)bufs->tmp_values);
            tmp = bufs->tmp;
        } else {
            tmp = (uint64_t *)sc.get(nb * 8 + 64);
        }
        if (!tmp) return ms_fail(MS_ERR_NOMEM, "select_sum temporary");
        MS_TRY(launch_decompress(in, tmp, s));
        grid = grid_for(nb, WG * 32ull, 2048);
        hipLaunchKernelGGL(k_select_sum_values, dim3(grid), dim3(WG), 0, s, (const uint64_t *)tmp, &in->meta->count,
                           p, part);
        with_rest = 0;
        break;
    }
    default:
        return ms_fail(MS_ERR_INVALID, "select_sum: unsupported format");
    }
    MS_HIP(hipGetLastError());
    if (single) return MS_OK;
    static_assert(SS_MAX_PARTS >= 8192, "every grid above is capped at 8192 workgroups");
    hipLaunchKernelGGL(k_sum_finish, dim3(1), dim3(WG), 0, s, v, p, (const uint64_t *)part, grid, with_rest,
                       (uint64_t)d_result | meta);
    MS_HIP(hipGetLastError());
    return MS_OK;
}

// Decompressed values are written once, far more of them than any cache
// holds: they are stored non-temporally (measured: dynamic_vbp 334 ->
// 247 us, delta 400 -> 232 us for 2^27 values with the paired 16-byte
// stores).
#ifndef MS_DECOMP_NT
#define MS_DECOMP_NT 1
#endif
static constexpr bool DECOMP_NT = MS_DECOMP_NT != 0;

int launch_decompress(const ms_col *in, uint64_t *d_out, hipStream_t s, ms_dev_meta *om)
{
    ms_colv v;
    MS_TRY(colv_of(in, v));
    const uint64_t nb = in->count_bound;
    if (nb == 0) {
        if (om) hipLaunchKernelGGL(k_set_meta_uncompr, dim3(1), dim3(1), 0, s, (const ms_dev_meta *)in->meta, om);
        return om ? (hipGetLastError() == hipSuccess ? MS_OK : ms_fail(MS_ERR_HIP, "decompress meta")) : MS_OK;
    }
    const uint32_t grid_units = grid_for(nb / 512 + 1, WAVES * 4ull, 8192);
    const uint64_t quads = nb / 2048 + 1;   // groups of 4 units
    switch (v.g.kind) {
    case MS_UNCOMPR:
        break;
    case MS_RLE: {
        temps sc(s);
        const uint64_t nch_bound = (in->size_alloc / 16 + 1) / RLE_XCH + 1;
        const uint64_t nst_bound = nch_bound / RLE_SCH + 1, nt_bound = nb / RLE_XT + 1;
        if (nch_bound >= (1ull << 32)) return ms_fail(MS_ERR_CAPACITY, "rle: %llu chunks of runs",
                                                      (unsigned long long)nch_bound);
        uint64_t *state = (uint64_t *)sc.get((1 + nst_bound) * 8);
        uint64_t *cstart = (uint64_t *)sc.get(nch_bound * 8);
        uint32_t *tchunk = (uint32_t *)sc.get(nt_bound * 4);
        if (!state || !cstart || !tchunk) return ms_fail(MS_ERR_NOMEM, "rle scratch");
        hipLaunchKernelGGL(k_rle_begin, dim3(grid_for(1 + nst_bound, WG * 4ull, 256)), dim3(WG), 0, s,
                           (const ms_dev_meta *)in->meta, state, 1 + nst_bound, om);
        const uint32_t r = resident_grid((const void *)k_rle_starts, WG);
        hipLaunchKernelGGL(k_rle_starts, dim3(grid_for(nst_bound, 1, r)), dim3(WG), 0, s, v, state, cstart, tchunk,
                           nt_bound);
        MS_HIP(hipGetLastError());
        auto k = k_rle_expand<DECOMP_NT>;
        hipLaunchKernelGGL(k, dim3(stride_grid((const void *)k, nt_bound)), dim3(WG), 0, s, v,
                           (const uint64_t *)cstart, (const uint32_t *)tchunk, d_out);
        MS_HIP(hipGetLastError());
        return MS_OK;
    }
    case MS_STATIC_VBP:
        if (fast_static(v) && v.g.lanes == 8) {
            auto k = k_decomp_units<DL_STATIC8, DECOMP_NT>;
            hipLaunchKernelGGL(k, dim3(stride_grid((const void *)k, quads)), dim3(WG), 0, s, v, d_out, om);
            MS_HIP(hipGetLastError());
            return MS_OK;   // rest and meta written by the kernel
        } else if (fast_static(v)) {
            hipLaunchKernelGGL(static_dec_kernel(v.g.bw), dim3(grid_units), dim3(WG), 0, s, v, d_out);
        } else {
            hipLaunchKernelGGL(k_decomp_generic, dim3(grid_for(nb, WG * 8ull)), dim3(WG), 0, s, v, d_out);
        }
        break;
    case MS_DYNAMIC_VBP:
    case MS_FOR:
        if (fast_blocks(v)) {
            auto k = v.g.kind == MS_FOR ? k_decomp_units<DL_FOR, DECOMP_NT> : k_decomp_units<DL_BLOCKS, DECOMP_NT>;
            hipLaunchKernelGGL(k, dim3(stride_grid((const void *)k, quads)), dim3(WG), 0, s, v, d_out, om);
            MS_HIP(hipGetLastError());
            return MS_OK;   // rest and meta written by the kernel
        } else {
            hipLaunchKernelGGL(k_decomp_generic, dim3(grid_for(nb, WG * 8ull)), dim3(WG), 0, s, v, d_out);
        }
        break;
    case MS_DELTA: {
        temps sc(s);
        const uint64_t *arr;
        MS_TRY(delta_src(in, v, sc, &arr));
        if (!arr && v.g.lg_spb != 0xff) {
            auto k = k_delta_decomp<DECOMP_NT>;
            hipLaunchKernelGGL(k, dim3(stride_grid((const void *)k, nb / DELTA_TILE + 1)), dim3(WG), 0, s, v, d_out,
                               om);
            MS_HIP(hipGetLastError());
            return MS_OK;   // rest and meta written by the kernel
        }
        const dim3 grid(grid_for(nb / DELTA_TILE + 1, 1, 65536));
        if (arr) hipLaunchKernelGGL((k_delta_tiles<0, 1>), grid, dim3(WG), 0, s, v, arr, d_out, ms_pred{}, nullptr);
        else hipLaunchKernelGGL((k_delta_tiles<0, 0>), grid, dim3(WG), 0, s, v, arr, d_out, ms_pred{}, nullptr);
        break;
    }
    case MS_STATIC_VBP_PAD:
    case MS_K_WISE_NS:
    case MS_GROUP_SIMPLE:
        MS_TRY(launch_xfmt_decompress(in, d_out, s));
        break;
    case MS_BLOCKWISE_INDIVIDUAL:
        MS_TRY(launch_bwi_decompress(in, d_out, s));   // copies its rest itself
        if (om) hipLaunchKernelGGL(k_set_meta_uncompr, dim3(1), dim3(1), 0, s, (const ms_dev_meta *)in->meta, om);
        MS_HIP(hipGetLastError());
        return MS_OK;
    default:
        return ms_fail(MS_ERR_INVALID, "decompress: unsupported format");
    }
    MS_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_copy_rest, dim3(grid_for(nb, WG * 4ull, 4096)), dim3(WG), 0, s, v, d_out);
    if (om) hipLaunchKernelGGL(k_set_meta_uncompr, dim3(1), dim3(1), 0, s, (const ms_dev_meta *)in->meta, om);
    MS_HIP(hipGetLastError());
    return MS_OK;
}

// Flags of unit u's 512 values, a byte per thread (bit m of thread t's byte
// = value 64 * (t >> 3) + 8 * m + (t & 7) of the unit): decoded from the
// compressed part, or read raw from the rest.
// Index entry and for_f reference of unit u (left in vector registers, so
// that a caller can request them one unit ahead and wait only at use).
__device__ __forceinline__ void unit_entry(const ms_colv &c, uint64_t ncu, uint64_t u, uint64_t &e, uint64_t &r)
{
    e = r = 0;
    if (u < ncu && c.g.kind == MS_STATIC_VBP) {   // 8 lanes: 64 bw bytes per unit, no index
        e = ((u * 64 * c.g.bw) << 8) | c.g.bw;
    } else if (u < ncu) {
        const uint64_t b = u >> c.g.lg_spb;
        e = gload(c.index + b);
        if (c.g.kind == MS_FOR) r = gload(c.refs + (b >> c.g.lg_ipo));
    }
}

__device__ __forceinline__ uint32_t unit_flags(const ms_colv &c, const ms_parts &pt, const ms_pred &p, uint64_t u,
                                               uint64_t e_v, uint64_t r_v, uint32_t t)
{
    const uint32_t j = t & 7, gl = t >> 3;
    const uint64_t ncu = pt.n_compr >> 9;
    uint64_t d[8];
    uint32_t ok = 0xff;
    if (u < ncu) {
        const uint64_t sub = u & ((1ull << c.g.lg_spb) - 1);
        const uint64_t e = uniform64(e_v);
        const uint64_t ref = c.g.kind == MS_FOR ? uniform64(r_v) : 0ull;
        dec_dispatch((uint32_t)(e & 0xff), (const uint64_t *)(c.data + (e >> 8)), 8, j, sub * 8 + gl, d);
#pragma unroll
        for (int m = 0; m < 8; m++) d[m] += ref;
    } else {
        // the raw rest: value i of the unit is rest value (u - ncu) * 512 + i
        const uint64_t *x = (const uint64_t *)(c.data + pt.rest_off);
        const uint64_t r0 = (u - ncu) * 512;
        ok = 0;
#pragma unroll
        for (int m = 0; m < 8; m++) {
            const uint64_t r = r0 + 64 * gl + 8 * m + j;
            const bool in = r < pt.n_rest;
            d[m] = in ? gload(x + r) : 0ull;
            ok |= in ? 1u << m : 0u;
        }
    }
    uint32_t bits = 0;
#pragma unroll
    for (int m = 7; m >= 0; m--) bits = bits + bits + (pred_eval(p, d[m]) ? 1u : 0u);
    return bits & ok;
}

// The flags of a thread's 8 codes (at most 32 bits, cut from its words), bit
// m for code m, under the unit's predicate mode.
template <int BW>
__device__ __forceinline__ uint32_t flag_cut(const uint64_t (&w)[5], uint32_t g, uint32_t mode, uint32_t lo,
                                             uint32_t span)
{
    uint32_t c[8], bits = 0;
    vbp_cut32<BW>(w, ((g * BW) & 7) * 8, c);
    if (mode == SM_LE) {
#pragma unroll
        for (int m = 7; m >= 0; m--) bits = bits + bits + (c[m] <= span ? 1u : 0u);
    } else {
#pragma unroll
        for (int m = 7; m >= 0; m--) bits = bits + bits + ((uint32_t)(c[m] - lo) <= span ? 1u : 0u);
    }
    return bits;
}

__device__ __forceinline__ uint32_t flag_cut_dispatch(uint32_t bw, const uint64_t (&w)[5], uint32_t g, uint32_t mode,
                                                      uint32_t lo, uint32_t span)
{
    switch (bw) {
#define MS_CASE(X) \
    case X: return flag_cut<X>(w, g, mode, lo, span);
        MS_BW32_CASES(MS_CASE)
#undef MS_CASE
    default: return 0;
    }
}

// A unit's predicate mode and its words' request for k_sel_count_blocks: the
// fused sums' own, but that a wholly selected unit is not read either.
template <bool IS_FOR>
__device__ __forceinline__ void flag_prep(const uint8_t *data, uint64_t e, uint64_t r, bool valid, uint64_t u,
                                          uint64_t mask, const ms_pred &p, const ms_bwtab &tab, uint32_t j,
                                          uint32_t gl, uint32_t &mode, uint32_t &lo, uint32_t &span,
                                          uint64_t (&w)[5])
{
    mode = SM_NONE;
    lo = span = 0;
    if (!valid) return;
    const uint32_t bw = (uint32_t)(e & 0xff);
    if (bw > 32) {
        mode = SM_SLOW;
    } else if (IS_FOR) {
        const uint64_t maxcode = (1ull << bw) - 1ull;
        if (r + maxcode < r) {
            mode = SM_SLOW;
        } else {
            const ms_cpred cp = code_pred(p, r, maxcode);
            mode = cp.mode == PM_NONE ? SM_NONE : cp.mode == PM_ALL ? SM_ALL : cp.mode == PM_OUT ? SM_OUT
                 : cp.clo == 0 ? SM_LE : SM_IN;
            lo = (uint32_t)cp.clo;
            span = (uint32_t)cp.cspan;
        }
    } else {
        mode = tab.mode[bw];
        lo = tab.lo[bw];
        span = tab.span[bw];
    }
    if (mode == SM_LE || mode == SM_IN || mode == SM_OUT) {
        uint32_t g = (uint32_t)(u & mask) * 8 + gl;
        asm volatile("" : "+v"(g));   // keeps per-width offsets of g from being hoisted
        unit_words_dispatch(bw, (const uint64_t *)(data + (e >> 8)), j, g, w);
    }
}

// The flags of a thread's 8 wide (more than 32 bits) or wrapping codes.  Out
// of line, as the fused sums' rare path is, so that it does not set the
// kernel's register budget.
__device__ __attribute__((noinline, pure)) uint32_t slow_flags(const ms_pred p, const uint64_t *base, uint32_t bw, uint32_t j,
                                                         uint32_t g, uint64_t ref)
{
    uint64_t d[8];
    dec_dispatch(bw, base, 8, j, g, d);
    uint32_t bits = 0;
#pragma unroll
    for (int m = 7; m >= 0; m--) bits = bits + bits + (pred_eval(p, d[m] + ref) ? 1u : 0u);
    return bits;
}

// The flags of a thread's 8 codes of unit u.
template <bool IS_FOR>
__device__ __forceinline__ uint32_t flag_finish(const uint8_t *data, const ms_pred &p, uint64_t e, uint64_t r,
                                                bool valid, uint64_t u, uint64_t mask, uint32_t j, uint32_t gl,
                                                uint32_t mode, uint32_t lo, uint32_t span, const uint64_t (&w)[5])
{
    if (!valid || mode == SM_NONE) return 0;
    if (mode == SM_ALL) return 0xff;
    uint32_t g = (uint32_t)(u & mask) * 8 + gl;
    asm volatile("" : "+v"(g));
    const uint32_t bw = (uint32_t)(e & 0xff);
    if (mode == SM_SLOW) return slow_flags(p, (const uint64_t *)(data + (e >> 8)), bw, j, g, IS_FOR ? r : 0ull);
    const uint32_t bits = flag_cut_dispatch(bw, w, g, mode, lo, span);
    return mode == SM_OUT ? bits ^ 0xffu : bits;
}

// Decodes and tests every unit once: each thread's flag byte goes to byte t
// of the unit's flags (64 bytes per 512 values) and its selected count to
// cnt[u].  As the fused sums do, a wave takes 4 units at a time: each unit's
// predicate is reduced to its codes' range, the words of all 4 are requested
// before the first is cut (none for a unit that is selected wholly or not at
// all), and codes of up to 32 bits are tested in 32 bits.
// Bound by the decode's instructions (3-bit codes) or HBM (20 bits: 4.1
// TB/s).  Measured for 2^28 rows, one unit at a time in 64 bits with a ballot
// word per code before / now: 3-bit codes 164 / 102 us, 20-bit codes 226 /
// 163 us; for_f of 2^26 rows 47 / 38 us.
template <bool IS_FOR>
__global__ __launch_bounds__(WG) void k_sel_count_blocks(ms_colv c, ms_pred p, ms_bwtab tab, uint64_t *d_units,
                                                         uint64_t *cnt, uint64_t *flags)
{
    const ms_parts pt = parts_of(c);
    const uint64_t nunits = (pt.n + 511) / 512;
    const uint64_t ncu = pt.n_compr >> 9;
    const uint64_t nq = (ncu + 3) >> 2;   // groups of 4 packed units
    const uint32_t t = threadIdx.x & 63;
    const uint32_t j = t & 7, gl = t >> 3;
    const uint64_t W = (uint64_t)gridDim.x * WAVES;
    const uint64_t first = (uint64_t)blockIdx.x * WAVES + wave_index();
    const uint64_t mask = (1ull << c.g.lg_spb) - 1ull;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        *d_units = nunits;   // for the scan and the emission after this kernel
        cnt[nunits] = 0;     // the scan's total slot
    }
    uint64_t my_e = 0, my_r = 0;   // lanes 0..3: the next group's entries, requested one group ahead
    if (first < nq && t < 4) unit_entry(c, ncu, first * 4 + t, my_e, my_r);
    for (uint64_t q = first; q < nq; q += W) {
        const uint64_t u0 = q * 4;
        const uint32_t num = ncu - u0 < 4 ? (uint32_t)(ncu - u0) : 4u;
        uint64_t e[4], r[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            e[k] = readlane64(my_e, k);
            r[k] = IS_FOR ? readlane64(my_r, k) : 0ull;
        }
        my_e = my_r = 0;
        if (q + W < nq && t < 4) unit_entry(c, ncu, u0 + 4 * W + t, my_e, my_r);
        uint32_t mo0, mo1, mo2, mo3, lo0, lo1, lo2, lo3, sp0, sp1, sp2, sp3;
        uint64_t w0[5], w1[5], w2[5], w3[5];   // named arrays: they stay in registers
        flag_prep<IS_FOR>(c.data, e[0], r[0], num > 0, u0, mask, p, tab, j, gl, mo0, lo0, sp0, w0);
        flag_prep<IS_FOR>(c.data, e[1], r[1], num > 1, u0 + 1, mask, p, tab, j, gl, mo1, lo1, sp1, w1);
        flag_prep<IS_FOR>(c.data, e[2], r[2], num > 2, u0 + 2, mask, p, tab, j, gl, mo2, lo2, sp2, w2);
        flag_prep<IS_FOR>(c.data, e[3], r[3], num > 3, u0 + 3, mask, p, tab, j, gl, mo3, lo3, sp3, w3);
        const uint32_t f0 = flag_finish<IS_FOR>(c.data, p, e[0], r[0], num > 0, u0, mask, j, gl, mo0, lo0, sp0, w0);
        const uint32_t f1 = flag_finish<IS_FOR>(c.data, p, e[1], r[1], num > 1, u0 + 1, mask, j, gl, mo1, lo1, sp1, w1);
        const uint32_t f2 = flag_finish<IS_FOR>(c.data, p, e[2], r[2], num > 2, u0 + 2, mask, j, gl, mo2, lo2, sp2, w2);
        const uint32_t f3 = flag_finish<IS_FOR>(c.data, p, e[3], r[3], num > 3, u0 + 3, mask, j, gl, mo3, lo3, sp3, w3);
        uint8_t *fb = (uint8_t *)(flags + 8 * u0) + t;
        fb[0] = (uint8_t)f0;
        if (num > 1) fb[64] = (uint8_t)f1;
        if (num > 2) fb[128] = (uint8_t)f2;
        if (num > 3) fb[192] = (uint8_t)f3;
        const uint32_t n01 = dpp_sum_u32((uint32_t)__builtin_popcount(f0) + ((uint32_t)__builtin_popcount(f1) << 16));
        const uint32_t n23 = dpp_sum_u32((uint32_t)__builtin_popcount(f2) + ((uint32_t)__builtin_popcount(f3) << 16));
        const uint32_t pair = t & 2 ? n23 : n01;
        if (t < num) cnt[u0 + t] = t & 1 ? pair >> 16 : pair & 0xffffu;
    }
    for (uint64_t u = ncu + first; u < nunits; u += W) {   // the raw rest
        const uint32_t f = unit_flags(c, pt, p, u, 0, 0, t);
        ((uint8_t *)(flags + 8 * u))[t] = (uint8_t)f;
        const uint32_t n = dpp_sum_u32((uint32_t)__builtin_popcount(f));
        if (t == 0) cnt[u] = n;
    }
}

// ------------------------------------------------------------------
// Select positions: one pass over the rows, a wave per 1, 2 or 4 units of
// 512 rows (per_wave), a workgroup's units one tile of a look-back over the
// tiles' counts.
// A unit's flags go to LDS as a bit per row (row r's 64 bits in word r); the
// positions are written a tile later, when the tile's first rank is known
// (its look-back then waits for no straggler).  Codes are tested as they are
// decoded, so a bit-packed column is never expanded: SEL_LANES8 takes the
// 8-lane indexed layouts and static_vbp_f<vbp_l<bw, 8>>, SEL_LANES1
// static_vbp_f<vbp_l<bw, 1>>, SEL_RAW values (decompressed by the caller for
// every other format).
// Bound by the positions' stores and the tiles' tickets (about 20 ns each,
// one counter for all XCDs).  Measured over 2^24 values of 12 bits, half of
// them selected: 34 us from static_vbp_f<vbp_l<12, 1>> (decompression,
// count, two scan kernels, compaction, split, copy and append before:
// 200 us), 36 us from dynamic_vbp_f, 42 us from uncompr_f.
// ------------------------------------------------------------------
enum { SEL_LANES8 = 0, SEL_LANES1 = 1, SEL_RAW = 2 };
constexpr uint32_t SEL_WAVES = 16, SEL_UNITS = 4;          // waves per tile, units per wave at most

template <int SRC>
__global__ __launch_bounds__(SEL_WAVES * 64) void k_select_onepass(ms_colv c, const uint64_t *x, ms_pred p,
                                                                   uint64_t *state, uint64_t *pos, uint64_t *d_cnt,
                                                                   ms_dev_meta *om, uint32_t per_wave)
{
    __shared__ uint64_t s_rows[2][SEL_WAVES][SEL_UNITS][8], s_ticket, s_base;
    __shared__ uint32_t s_cnt[SEL_WAVES];
    const ms_parts pt = parts_of(c);
    const uint64_t nunits = (pt.n + 511) / 512, ncu = pt.n_compr >> 9;
    const uint32_t tile_units = SEL_WAVES * per_wave;
    const uint64_t ntiles = nunits ? (nunits + tile_units - 1) / tile_units : 1;
    const uint32_t t = threadIdx.x & 63, w = wave_index();
    uint64_t *tiles = state + 1;
    if (blockIdx.x >= ntiles) return;   // as many workgroups as tiles take tickets
    if (threadIdx.x == 0) s_ticket = lb_ticket(state);
    __syncthreads();
    uint64_t tile = readlane64(s_ticket, 0);
    __syncthreads();
    if (tile >= ntiles) return;
    uint64_t ptile = ~0ull;                 // the tile that waits for its first rank
    uint32_t pmine = 0, ptotal = 0;         // its rows of the waves before this one, of all
    for (uint32_t turn = 0;; turn ^= 1) {
        const bool have = tile < ntiles;
        uint32_t n = 0;
        if (have) {
            if (threadIdx.x == 0) s_ticket = lb_ticket(state);
            const uint64_t u0 = tile * tile_units + w * per_wave;
            uint64_t my_e = 0, my_r = 0;    // lanes 0..3: the units' index entries and references
            if (SRC == SEL_LANES8 && t < per_wave) unit_entry(c, ncu, u0 + t, my_e, my_r);
#pragma unroll 1
            for (uint32_t k = 0; k < per_wave; k++) {
                const uint64_t u = u0 + k;
                uint64_t *rows = s_rows[turn][w][k];
                if (u >= nunits) {
                    if (t < 8) rows[t] = 0;
                    continue;
                }
                if (SRC == SEL_LANES8) {
                    const uint32_t f = unit_flags(c, pt, p, u, readlane64(my_e, k), readlane64(my_r, k), t);
                    ((uint8_t *)rows)[t] = (uint8_t)f;
                    n += dpp_sum_u32((uint32_t)__builtin_popcount(f));
                } else if (SRC == SEL_LANES1) {
                    // thread t holds rows 8 t .. 8 t + 7: wholly packed or wholly raw
                    // (the packed part is a multiple of 64)
                    uint64_t d[8];
                    const uint64_t r0 = u * 512 + 8 * t;
                    uint32_t in = 0xff;
                    if (r0 < pt.n_compr) {
                        uint64_t g = u * 64 + t;
                        asm volatile("" : "+v"(g));   // keeps per-width offsets of g from being hoisted
                        dec_dispatch(c.g.bw, (const uint64_t *)c.data, 1, 0, g, d);
                    } else {
                        const uint64_t *y = (const uint64_t *)(c.data + pt.rest_off) + (r0 - pt.n_compr);
                        in = 0;
#pragma unroll
                        for (uint32_t m = 0; m < 8; m++) {
                            const bool ok = r0 + m < pt.n;
                            d[m] = ok ? gload(y + m) : 0ull;
                            in |= ok ? 1u << m : 0u;
                        }
                    }
                    uint32_t bits = 0;
#pragma unroll
                    for (uint32_t m = 0; m < 8; m++) {
                        const bool take = ((in >> m) & 1) && pred_eval(p, d[m]);
                        bits |= take ? 1u << m : 0u;
                        n += (uint32_t)__popcll(__ballot(take));
                    }
                    ((uint8_t *)rows)[t] = (uint8_t)bits;
                } else {
                    uint64_t d[8], mine = 0;
#pragma unroll
                    for (uint32_t r = 0; r < 8; r++) {
                        const uint64_t i = u * 512 + 64 * r + t;
                        d[r] = i < pt.n ? gload(x + i) : 0ull;
                    }
#pragma unroll
                    for (uint32_t r = 0; r < 8; r++) {
                        const uint64_t F = __ballot(u * 512 + 64 * r + t < pt.n && pred_eval(p, d[r]));
                        n += (uint32_t)__popcll(F);
                        if (t == r) mine = F;
                    }
                    if (t < 8) rows[t] = mine;
                }
            }
            if (t == 0) s_cnt[w] = n;
        }
        __syncthreads();
        uint64_t next = ~0ull;
        uint32_t mine = 0, total = 0;
        if (have) {
            next = readlane64(s_ticket, 0);
#pragma unroll
            for (uint32_t i = 0; i < SEL_WAVES; i++) {
                if (i == w) mine = total;
                total += __builtin_amdgcn_readfirstlane(s_cnt[i]);
            }
            if (w == 0) lb_publish(tiles, tile, total);
        }
        if (w == 0 && ptile != ~0ull) {
            uint64_t words[LB_SPAN];
            lb_request(tiles, (int64_t)ptile - 1, words);
            const uint64_t base = lb_exclusive(tiles, ptile, ptotal, words);
            if (t == 0) s_base = base;
        }
        __syncthreads();
        if (ptile != ~0ull) {
            uint64_t o = readlane64(s_base, 0) + pmine;
            const uint64_t u0 = ptile * tile_units + w * per_wave;
            // the wave's row words, one per lane
            uint64_t mine_w = (&s_rows[turn ^ 1][w][0][0])[t % (8 * SEL_UNITS)];
            if (SRC == SEL_LANES8) mine_w = flag_rows(mine_w);
#pragma unroll 4
            for (uint32_t r = 0; r < 8 * per_wave; r++) {
                const uint64_t F = readlane64(mine_w, r);
                if (F == 0) continue;
                if (__builtin_amdgcn_inverse_ballot_w64(F))
                    pos[o + lanes_below(F)] = u0 * 512 + 64 * r + t;
                o += (uint32_t)__popcll(F);
            }
            if (ptile == ntiles - 1 && threadIdx.x == 0) {
                const uint64_t all = s_base + ptotal;
                *d_cnt = all;
                if (om) {
                    om->count = all;
                    om->size_used = 8 * all;
                    om->size_compr = 0;
                    om->status = 0;
                    om->aux[0] = 8 * all;
                    for (int k = 1; k < 4; k++) om->aux[k] = 0;
                }
            }
        }
        if (!have) return;
        pmine = mine;
        ptotal = total;
        ptile = tile;
        tile = next;
    }
}

bool select_flags_ok(const ms_col *in)
{
    ms_colv v;
    if (colv_of(in, v) != MS_OK) return false;
    return (v.g.kind == MS_DYNAMIC_VBP || v.g.kind == MS_FOR) && fast_blocks(v);
}

// The count pass of the block-layout select and the scan of its unit
// counts (with the total at uoff[units]); no compaction.
int launch_select_flags(const ms_col *in, const ms_pred &p, sel_flags &sf, temps &sc)
{
    hipStream_t s = sc.s;
    const uint64_t nb = in->count_bound;
    ms_colv v;
    MS_TRY(colv_of(in, v));
    if (!((v.g.kind == MS_DYNAMIC_VBP || v.g.kind == MS_FOR) && fast_blocks(v)))
        return ms_fail(MS_ERR_INVALID, "select flags: layout without a block decoder");
    const uint64_t units = nb / 512 + 1;
    uint64_t *d_u = (uint64_t *)sc.get(64);
    uint64_t *cnt = (uint64_t *)sc.get(units * 8 + 64);
    uint64_t *off = (uint64_t *)sc.get(units * 8 + 64);
    uint64_t *flags = (uint64_t *)sc.get(units * 64 + 64);
    if (!d_u || !cnt || !off || !flags) return ms_fail(MS_ERR_NOMEM, "select scratch");
    auto k = v.g.kind == MS_FOR ? k_sel_count_blocks<true> : k_sel_count_blocks<false>;
    hipLaunchKernelGGL(k, dim3(stride_grid((const void *)k, nb / 2048 + 1)), dim3(WG), 0, s, v, p, make_bwtab(p), d_u,
                       cnt, flags);
    MS_HIP(hipGetLastError());
    MS_TRY(launch_exclusive_scan_n(cnt, off, d_u, 1, units + 1, sc));
    sf.flags = flags;
    sf.uoff = off;
    sf.d_units = d_u;
    sf.units_bound = units;
    return MS_OK;
}

int launch_select_positions(const ms_col *in, const ms_pred &p, uint64_t *d_pos, uint64_t *d_cnt, temps &sc,
                            ms_dev_meta *om)
{
    hipStream_t s = sc.s;
    const uint64_t nb = in->count_bound;
    ms_colv v;
    MS_TRY(colv_of(in, v));
    // few units per wave while that leaves CUs without a tile, many for few
    // tickets.  Calls one after the other, 1 / 2 / 4 units, us, half of the
    // rows selected:
    //   rows     static_vbp_f<12, 1>   dynamic_vbp_f       uncompr_f
    //   2^18     11.5 / 12.3 / 16.9    10.3 / 11.9 / 15.6  10.5 / 12.3 / 15.8
    //   2^20     12.2 / 13.3 / 17.6    12.3 / 12.6 / 15.5  12.4 / 13.2 / 16.5
    //   2^20.5   15.5 / 14.3 / 17.8    15.4 / 12.9 / 16.0  15.3 / 13.9 / 17.9
    //   2^21     18.1 / 14.6 / 18.2    18.5 / 14.6 / 16.7  18.6 / 15.2 / 19.0
    //   2^23     32.6 / 27.2 / 30.5    33.6 / 27.6 / 30.4  34.0 / 29.9 / 37.2
    //   2^23.5   39.8 / 32.6 / 32.3    41.1 / 33.1 / 32.2  42.7 / 39.1 / 39.2
    //   2^24     50.3 / 40.1 / 35.8    51.9 / 40.2 / 35.0  54.4 / 48.9 / 44.1
    // (4 are 10% better around 2^22 from the packed sources: one round of
    // tiles per resident workgroup.)
    const uint32_t per_wave = nb <= 1ull << 20 ? 1 : nb <= 1ull << 23 ? 2 : SEL_UNITS;
    const uint64_t tiles = nb / (512ull * SEL_WAVES * per_wave) + 1;
    uint64_t *state = (uint64_t *)sc.get((1 + tiles) * 8);
    if (!state) return ms_fail(MS_ERR_NOMEM, "select scratch");
    MS_TRY(launch_fill_u64(state, 1 + tiles, 0, s));
    const bool lanes8 = ((v.g.kind == MS_DYNAMIC_VBP || v.g.kind == MS_FOR) && fast_blocks(v)) ||
                        (v.g.kind == MS_STATIC_VBP && v.g.lanes == 8);
    auto k = lanes8                                             ? k_select_onepass<SEL_LANES8>
           : v.g.kind == MS_STATIC_VBP && v.g.lanes == 1        ? k_select_onepass<SEL_LANES1>
                                                                : k_select_onepass<SEL_RAW>;
    const uint64_t *x = nullptr;
    if (k == k_select_onepass<SEL_RAW>) {
        x = (const uint64_t *)in->data;
        if (in->g.kind != MS_UNCOMPR) {
            uint64_t *tmp = (uint64_t *)sc.get(nb * 8 + 64);
            if (!tmp) return ms_fail(MS_ERR_NOMEM, "select scratch");
            MS_TRY(launch_decompress(in, tmp, s));
            x = tmp;
        }
    }
    const uint32_t r = resident_grid((const void *)k, SEL_WAVES * 64);
    hipLaunchKernelGGL(k, dim3(grid_for(tiles, 1, r)), dim3(SEL_WAVES * 64), 0, s, v, x, p, state, d_pos, d_cnt, om,
                       per_wave);
    MS_HIP(hipGetLastError());
    return MS_OK;
}

// ------------------------------------------------------------------
// Exclusive scan of the first min(*d_n + extra, bound) values, sized from
// the device count: G workgroups each take one contiguous chunk (sum,
// then the chunk scan on the sum of the sums before it).  Arrays allocated for
// a host bound are scanned only as far as they are used; without a device
// count (d_n null) all `bound` values are scanned.  Counts are 64-bit
// throughout.
// ------------------------------------------------------------------
__device__ __forceinline__ void chunk_of(const uint64_t *d_n, uint64_t extra, uint64_t bound, uint64_t &lo,
                                         uint64_t &hi)
{
    uint64_t n = d_n ? *d_n + extra : bound;
    if (n > bound) n = bound;
    const uint64_t chunk = (n + gridDim.x - 1) / gridDim.x;
    lo = (uint64_t)blockIdx.x * chunk;
    hi = lo + chunk < n ? lo + chunk : n;
    if (lo > hi) lo = hi;
}

__device__ __forceinline__ uint64_t block_sum(uint64_t v)
{
    __shared__ uint64_t s_w[WAVES];
    v = wave_sum_u64(v);
    if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = v;
    __syncthreads();
    uint64_t t = 0;
#pragma unroll
    for (int w = 0; w < WAVES; w++) t += s_w[w];
    __syncthreads();
    return t;
}

// Exclusive scan over the workgroup; *total receives the sum.
__device__ __forceinline__ uint64_t block_exscan(uint64_t v, uint64_t *total)
{
    __shared__ uint64_t s_w[WAVES];
    const uint32_t t = threadIdx.x & 63;
    uint64_t incl = v;
#pragma unroll
    for (uint32_t o = 1; o < 64; o <<= 1) {
        const uint64_t y = __shfl_up(incl, o, MS_WAVE);
        if (t >= o) incl += y;
    }
    if (t == 63) s_w[threadIdx.x >> 6] = incl;
    __syncthreads();
    uint64_t before = 0, all = 0;
#pragma unroll
    for (uint32_t w = 0; w < WAVES; w++) {
        const uint64_t x = s_w[w];
        if (w < (threadIdx.x >> 6)) before += x;
        all += x;
    }
    __syncthreads();
    *total = all;
    return before + incl - v;
}

__global__ __launch_bounds__(WG) void k_scan_part(const uint64_t *in, const uint64_t *d_n, uint64_t extra,
                                                  uint64_t bound, uint64_t *part)
{
    uint64_t lo, hi;
    chunk_of(d_n, extra, bound, lo, hi);
    uint64_t acc = 0;
    for (uint64_t i = lo + threadIdx.x; i < hi; i += WG) acc += in[i];
    acc = block_sum(acc);
    if (threadIdx.x == 0) part[blockIdx.x] = acc;
}

__global__ __launch_bounds__(WG) void k_scan_apply(const uint64_t *in, uint64_t *out, const uint64_t *d_n,
                                                   uint64_t extra, uint64_t bound, const uint64_t *part)
{
    uint64_t lo, hi;
    chunk_of(d_n, extra, bound, lo, hi);
    // the chunk's offset: the sums of the chunks before it (at most 1024)
    uint64_t before = 0;
    for (uint32_t k = threadIdx.x; k < blockIdx.x; k += WG) before += part[k];
    uint64_t carry = block_sum(before);
    for (uint64_t base = lo; base < hi; base += WG) {
        const uint64_t i = base + threadIdx.x;
        const uint64_t v = i < hi ? in[i] : 0;
        uint64_t tot;
        const uint64_t ex = block_exscan(v, &tot);
        if (i < hi) out[i] = carry + ex;
        carry += tot;
    }
}

int launch_exclusive_scan_n(const uint64_t *d_in, uint64_t *d_out, const uint64_t *d_n, uint64_t extra,
                            uint64_t bound, temps &sc)
{
    if (bound == 0) return MS_OK;
    const uint32_t G = grid_for(bound, 4096, 1024);
    uint64_t *part = (uint64_t *)sc.get(G * 8 + 64);
    if (!part) return ms_fail(MS_ERR_NOMEM, "scan scratch");
    hipLaunchKernelGGL(k_scan_part, dim3(G), dim3(WG), 0, sc.s, d_in, d_n, extra, bound, part);
    hipLaunchKernelGGL(k_scan_apply, dim3(G), dim3(WG), 0, sc.s, d_in, d_out, d_n, extra, bound,
                       (const uint64_t *)part);
    MS_HIP(hipGetLastError());
    return MS_OK;
}

int launch_exclusive_scan(const uint64_t *d_in, uint64_t *d_out, uint64_t n, temps &sc)
{
    return launch_exclusive_scan_n(d_in, d_out, nullptr, 0, n, sc);
}

}  // namespace ms
