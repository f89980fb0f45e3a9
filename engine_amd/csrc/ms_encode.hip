// ms_encode.hip -- write side of the compression-aware path on gfx950.
//
// One emitter produces every compressed format the operators write:
//   * column-level morph (morph.h:157-197): one morph_batch call over the
//     compressed part, then the uncompressed rest behind the gap;
//   * write-iterator output (write_iterator.h:66-196, delta.h:369-490):
//     independent morph_batch calls of m_CountBuffer = round_up(bs, 2048)
//     values, each starting fresh pages, then done()'s remainder and rest.
// The innermost vertical-bit-packed blocks are the unit of work: a kernel
// finds each block's bit width (dynamic_vbp.h:122-158) and the bytes of
// page headers in front of it (dvbp meta bytes, for_f reference pages), a
// scan places the blocks, and a pack kernel assembles each block's
// interleaved words in LDS and writes payload, headers and the block index.
#include "ms_kernels.h"
#include "ms_lookback.hpp"

namespace ms {

static constexpr int WG = 256;

static inline uint32_t grid_for(uint64_t items, uint64_t per_wg, uint32_t cap = 8192)
{
    uint64_t g = (items + per_wg - 1) / per_wg;
    if (g < 1) g = 1;
    if (g > cap) g = cap;
    return (uint32_t)g;
}

struct emit_layout {
    uint32_t kind;       // MS_STATIC_VBP, MS_DYNAMIC_VBP, MS_DELTA, MS_FOR
    uint32_t leaf;       // innermost layout
    uint32_t bw;         // static leaf bit width (64 for an uncompressed leaf)
    uint32_t S;          // innermost lanes
    uint32_t dstep;      // delta step
    uint32_t E;          // for_f lanes (reference-value minimum)
    uint64_t B;          // innermost block (values)
    uint64_t P;          // dvbp leaf page (blocks)
    uint64_t L;          // outer block (delta/for) or B
    uint64_t FP;         // for_f page (blocks)
    uint64_t bpo;        // innermost blocks per outer block
    uint64_t K;          // values per morph_batch call (0: one call)
    uint64_t bs;         // outer m_BlockSize
    uint64_t gap;        // rest gap
    uint64_t cap;        // bytes of the output image
    uint64_t *status;    // the output's status word (MS_ERR_CAPACITY past cap)
    // Chunked mode (both null otherwise): every K values are one morph_batch
    // call over the values v[cmap[c] * K ...] (its delta predecessors start
    // at zero), written at cout[c] of the image.
    const uint32_t *cmap;
    const uint64_t *cout;
};

struct emit_plan {
    uint64_t m;          // values
    uint64_t m_c;        // values in the compressed part
    uint64_t nb;         // innermost blocks
    uint64_t nfb;        // outer blocks (for_f)
};

// a / d and a % d (d > 0) for the layout's block and page counts, which are
// mostly powers of two: a shift and a mask then, the division otherwise.
__device__ __forceinline__ uint64_t ldiv(uint64_t a, uint64_t d)
{
    return (d & (d - 1)) == 0 ? a >> __builtin_ctzll(d) : a / d;
}
__device__ __forceinline__ uint64_t lmod(uint64_t a, uint64_t d)
{
    return (d & (d - 1)) == 0 ? a & (d - 1) : a % d;
}

__device__ __forceinline__ emit_plan plan_of(const emit_layout &l, uint64_t m)
{
    emit_plan p;
    p.m = m;
    uint64_t mc;
    if (l.K == 0) mc = ldiv(m, l.bs) * l.bs;
    else {
        const uint64_t full = ldiv(m, l.K), rem = m - full * l.K;
        mc = full * l.K + ldiv(rem, l.bs) * l.bs;
    }
    p.m_c = mc;
    p.nb = ldiv(mc, l.B);
    p.nfb = ldiv(mc, l.L);
    return p;
}

// Records that a write would pass the end of the output image; the write
// is dropped (the host sizes outputs so that this does not happen).
__device__ __forceinline__ void emit_overflow(const emit_layout &l)
{
    atomicCAS((unsigned long long *)l.status, 0ull, (unsigned long long)MS_ERR_CAPACITY);
}

// Bytes of headers in front of innermost block b.
__device__ __forceinline__ uint64_t hdr_of(const emit_layout &l, uint64_t b)
{
    uint64_t h = 0;
    if (l.leaf == MS_DYNAMIC_VBP) {
        uint64_t q;
        if (l.kind == MS_DYNAMIC_VBP) q = l.K ? lmod(b, ldiv(l.K, l.B)) : b;
        else q = lmod(b, l.bpo);                  // each outer block is one inner call
        if (lmod(q, l.P) == 0) h += l.P;
    }
    if (l.kind == MS_FOR && lmod(b, l.bpo) == 0) {
        const uint64_t fb = ldiv(b, l.bpo);
        const uint64_t fq = l.K ? lmod(fb, ldiv(l.K, l.L)) : fb;
        if (lmod(fq, l.FP) == 0) h += 8 * l.FP;
    }
    return h;
}

// The values of the call holding value `first`: returns the array they are
// indexed in and sets `lo` to first's index in it (delta predecessors exist
// from index dstep of that array on).
__device__ __forceinline__ const uint64_t *chunk_src(const emit_layout &l, const uint64_t *v, uint64_t first,
                                                     uint64_t &lo)
{
    if (!l.cmap) { lo = first; return v; }
    const uint64_t c = first / l.K;
    lo = first - c * l.K;
    return v + (uint64_t)l.cmap[c] * l.K;
}

// Image offset of innermost block b's headers.
__device__ __forceinline__ uint64_t out_pos(const emit_layout &l, const uint64_t *start, uint64_t b)
{
    if (!l.cout) return start[b];
    const uint64_t bpc = ldiv(l.K, l.B), c = ldiv(b, bpc);
    return l.cout[c] + start[b] - start[c * bpc];
}

// xform over a value getter: get(gi) = value gi of the call's array.
template <class G>
__device__ __forceinline__ uint64_t xform_g(const emit_layout &l, const G &get, uint64_t gi, uint64_t ref)
{
    const uint64_t x = get(gi);
    if (l.kind == MS_DELTA) return x - (gi >= l.dstep ? get(gi - l.dstep) : 0ull);
    if (l.kind == MS_FOR) return x - ref;
    return x;
}

// ------------------------------------------------------------------
// Values straight from a select's flags (no materialised positions): the
// value of rank r is the row of the r-th selected row.
// ------------------------------------------------------------------
struct flag_src {
    sel_flags sf;
    const uint32_t *ustart;   // per innermost block b: the unit holding rank r0(b)
    uint32_t pred;            // delta predecessors a block reads (0 unless delta_f)
};

// First rank a block's kernels read: its predecessors included.
__device__ __forceinline__ uint64_t flag_r0(const emit_layout &l, const flag_src &fs, uint64_t b)
{
    const uint64_t first = b * l.B;
    return first >= fs.pred ? first - fs.pred : 0ull;
}

// One wave writes the rows of ranks [r0, r0 + cnt) to st(rank - r0, row),
// walking the units from u (a unit at or before the one holding rank r0)
// eight at a time.  Lane t takes rows 64 gl .. 64 gl + 63 of unit
// u + t / 8 (gl = t & 7): its flag word, whose bits flag_rows puts in row
// order.  Its first rank is the unit's offset plus the set bits of the
// unit's lower row words (a scan over the lane's group of 8); then it
// writes its set bits in order.
template <class St>
__device__ __forceinline__ void gather_ranks(const sel_flags &sf, uint64_t nunits, uint64_t u, uint64_t r0,
                                             uint64_t cnt, const St &st)
{
    const uint32_t t = threadIdx.x & 63, gl = t & 7;
    const uint64_t r1 = r0 + cnt;
    if (cnt == 0 || cnt >= (1ull << 31)) return;   // callers ask for at most a few thousand ranks
    for (; u < nunits; u += 8) {
        const uint64_t uu = u + (t >> 3);
        const uint64_t ue = u + 8 < nunits ? u + 8 : nunits;
        const uint64_t end_rank = gload(sf.uoff + ue);   // requested with the group's loads
        uint64_t rw = 0, rank = 0;
        if (uu < nunits) {
            rw = flag_rows(gload(sf.flags + 8 * uu + gl));
            rank = gload(sf.uoff + uu);
        }
        // exclusive scan of the row words' counts within the group of 8
        const uint32_t c = (uint32_t)__popcll(rw);
        uint32_t incl = c;
#pragma unroll
        for (uint32_t o = 1; o < 8; o <<= 1) {
            const uint32_t y = (uint32_t)__shfl_up((int)incl, o, 8);
            if (gl >= o) incl += y;
        }
        rank += incl - c;
        if (rank >= r1 || rank + c <= r0) rw = 0;
        // a lane with bits left has rank in (r0 - 64, r1): 32-bit from here
        int32_t rel = (int32_t)(int64_t)(rank - r0);
        const uint32_t n32 = (uint32_t)cnt;
        const uint64_t row0 = uu * 512 + 64 * gl;
        uint32_t x = (uint32_t)rw;
        while (x) {
            const uint32_t p = (uint32_t)__builtin_ctz(x);
            if ((uint32_t)rel < n32) st((uint64_t)rel, row0 + p);
            rel++;
            x &= x - 1;
        }
        x = (uint32_t)(rw >> 32);
        while (x) {
            const uint32_t p = (uint32_t)__builtin_ctz(x) + 32;
            if ((uint32_t)rel < n32) st((uint64_t)rel, row0 + p);
            rel++;
            x &= x - 1;
        }
        if (end_rank >= r1) break;
    }
}

// The select's split (thread 0): the selected rows below the scalar
// remainder's first row thr are counted from the unit offsets and thr's
// unit's flags.
__device__ __forceinline__ void select_split(const sel_flags &sf, const sel_split &sp, uint64_t nunits)
{
    const ms_dev_meta *in = sp.in_meta;
    const ms_geom &g = sp.in_g;
    const ms_parts pt = ms_parts_of(g, in->count, in->size_used, in->size_compr);
    const bool has_rest = g.kind == MS_UNCOMPR ? in->count != 0 : in->size_compr != in->size_used;
    const uint64_t r = has_rest ? pt.n_rest % sp.lanes : 0;
    const uint64_t thr = pt.n - r;
    const uint64_t total = sf.uoff[nunits];
    const uint64_t u = thr / 512, w = thr % 512;
    uint64_t na = u < nunits ? sf.uoff[u] : total;
    if (u < nunits && w) {
        for (uint32_t gl = 0; 64 * gl < w; gl++) {
            const uint64_t k = w - 64 * gl;   // rows of the word below thr
            na += __popcll(flag_rows(sf.flags[8 * u + gl]) & (k < 64 ? (1ull << k) - 1 : ~0ull));
        }
    }
    *sp.d_cnt = total;
    *sp.d_na = na;
    *sp.d_flag = r != 0;
}

// ustart[b] for every block whose first read rank r0(b) lies in unit u's
// ranks [uoff[u], uoff[u+1]); one thread per unit.  Thread 0 also makes
// the select's split.
__global__ __launch_bounds__(WG) void k_flag_starts(emit_layout l, flag_src fs, sel_split sp, uint64_t cap,
                                                    uint32_t *ustart, ms_dev_meta *om)
{
    const uint64_t nunits = *fs.sf.d_units;
    if (blockIdx.x == 0 && threadIdx.x == 0) select_split(fs.sf, sp, nunits);
    // the output's meta starts cleared: the first kernel of the emission
    if (blockIdx.x == 0 && threadIdx.x < sizeof(ms_dev_meta) / 8) ((uint64_t *)om)[threadIdx.x] = 0;
    for (uint64_t u = (uint64_t)blockIdx.x * WG + threadIdx.x; u < nunits; u += (uint64_t)gridDim.x * WG) {
        const uint64_t lo = fs.sf.uoff[u], hi = fs.sf.uoff[u + 1];
        if (lo == hi) continue;
        // r0(b) = max(b B - pred, 0): b = 0 starts at rank 0
        uint64_t b = (lo + fs.pred + l.B - 1) / l.B;
        if (lo == 0) {
            if (cap > 0) ustart[0] = (uint32_t)u;
            if (b == 0) b = 1;
        }
        for (; b < cap && b * l.B - fs.pred < hi; b++) ustart[b] = (uint32_t)u;
    }
}

// for.h:121-161 reference value of one outer block, one wave per block.
// FL: the values come from a select's flags (dynamic LDS: L words).
template <bool FL>
__global__ __launch_bounds__(64) void k_for_refs(emit_layout l, const uint64_t *v, flag_src fs, const uint64_t *d_m,
                                                 uint64_t *refs)
{
    extern __shared__ unsigned long long fvals[];
    const emit_plan pl = plan_of(l, *d_m);
    const uint32_t t = threadIdx.x;
    const uint64_t nunits = FL ? *fs.sf.d_units : 0;
    for (uint64_t fb = blockIdx.x; fb < pl.nfb; fb += gridDim.x) {
        uint64_t lo;
        const uint64_t *xg = nullptr;
        if (FL) {
            gather_ranks(fs.sf, nunits, fs.ustart[fb * l.L / l.B], fb * l.L, l.L,
                         [&](uint64_t i, uint64_t row) { fvals[i] = row; });
            __syncthreads();
        } else {
            xg = chunk_src(l, v, fb * l.L, lo) + lo;
        }
        const auto x = [&](uint64_t i) -> uint64_t { return FL ? (uint64_t)fvals[i] : xg[i]; };
        uint64_t r;
        if (l.E == 1) {
            r = ~0ull;
            for (uint64_t i = t; i < l.L; i += 64) r = x(i) < r ? x(i) : r;
            for (int o = 32; o >= 1; o >>= 1) {
                const uint64_t y = __shfl_xor(r, o, 64);
                r = y < r ? y : r;
            }
        } else {
            // lane j = i % E: signed minimum per lane, then unsigned over lanes
            int64_t sm = INT64_MAX;
            for (uint64_t i = t; i < l.L; i += 64) sm = (int64_t)x(i) < sm ? (int64_t)x(i) : sm;
            for (uint32_t o = 32; o >= l.E; o >>= 1) {
                const int64_t y = (int64_t)__shfl_xor((uint64_t)sm, o, 64);
                sm = y < sm ? y : sm;
            }
            r = (uint64_t)sm;
            for (uint32_t o = l.E >> 1; o >= 1; o >>= 1) {
                const uint64_t y = __shfl_xor(r, o, 64);
                r = y < r ? y : r;
            }
        }
        if (t == 0) refs[fb] = r == ~0ull ? r - 1 : r;
        if (FL) __syncthreads();
    }
}

// Bit width of innermost block b over a value getter (one wave; lane t).
template <class G>
__device__ __forceinline__ uint32_t block_bw(const emit_layout &l, const G &get, uint64_t lo, uint64_t ref,
                                             uint32_t t)
{
    uint64_t o = 1;
    for (uint64_t i = t; i < l.B; i += 64) o |= xform_g(l, get, lo + i, ref);
    o = wave_or_u64(o);
    return 64 - __clzll(o);
}

// Assembles the interleaved words of innermost block b (one wave, lane t)
// in lds (B words; the first B bw / 64 hold the block).  sync() orders the
// wave's LDS accesses (the workgroup barrier when the workgroup is this
// wave); the words are complete when it returns.
template <class G, class Sync>
__device__ __forceinline__ void assemble_block(const emit_layout &l, uint32_t bw, const G &get, uint64_t lo,
                                               uint64_t ref, unsigned long long *lds, uint32_t t, const Sync &sync)
{
    // Lane counts that divide the wave and blocks of whole waves of codes
    // let each thread own a run of consecutive codes of one lane.
    const uint32_t S = (uint32_t)l.S;
    const bool runs = S != 0 && S <= 64 && 64 % S == 0 && l.B % 64 == 0;
    const uint32_t j = runs ? t % S : 0, g = runs ? t / S : 0, C = (uint32_t)(l.B >> 6);
    const uint64_t words = l.B * bw / 64;
    for (uint64_t w = t; w < words; w += 64) lds[w] = 0;
    sync();
    // OR every code in, unmasked (vbp_routine_gen.py:101, 111)
    if (runs) {
        // Thread (j, g) owns codes g*C .. g*C+C-1 of lane j: consecutive
        // codes share words, so it ORs them in registers and issues one
        // LDS atomic per word it touches instead of one per code.
        const uint64_t base = lo + j;
        uint32_t k = g * C, bit = k * bw, cw = bit >> 6;
        uint64_t acc = 0;
        // A delta step of one lane width makes each code's predecessor
        // the thread's previous code: one extra load per run.
        const bool own_pred = l.kind == MS_DELTA && l.dstep == S;
        uint64_t prev = 0;
        if (own_pred) {
            const uint64_t g0 = base + (uint64_t)k * S;
            prev = g0 >= S ? get(g0 - S) : 0ull;
        }
        for (uint32_t c0 = 0; c0 < C; c0 += 8) {
            uint64_t x[8];
#pragma unroll
            for (uint32_t q = 0; q < 8; ++q) {
                const uint64_t gi = base + (uint64_t)(k + q) * S;
                x[q] = c0 + q < C ? (own_pred ? get(gi) : xform_g(l, get, gi, ref)) : 0ull;
            }
            if (own_pred) {
#pragma unroll
                for (uint32_t q = 0; q < 8; ++q) {
                    const uint64_t r = x[q];
                    x[q] = r - prev;
                    prev = r;
                }
            }
#pragma unroll
            for (uint32_t q = 0; q < 8; ++q) {
                if (c0 + q >= C) break;
                const uint32_t w = bit >> 6, sh = bit & 63;
                if (w != cw) {
                    atomicOr(&lds[cw * S + j], (unsigned long long)acc);
                    acc = 0;
                    cw = w;
                }
                acc |= x[q] << sh;
                if (sh + bw > 64) {
                    atomicOr(&lds[cw * S + j], (unsigned long long)acc);
                    cw = w + 1;
                    acc = x[q] >> (64 - sh);
                }
                bit += bw;
            }
            k += 8;
        }
        atomicOr(&lds[cw * S + j], (unsigned long long)acc);
    } else {
        for (uint64_t i = t; i < l.B; i += 64) {
            const uint64_t c = xform_g(l, get, lo + i, ref);
            const uint64_t j = i % l.S, k = i / l.S;
            const uint64_t bit = k * bw;
            const uint64_t w = bit >> 6;
            const uint32_t sh = (uint32_t)(bit & 63);
            atomicOr(&lds[w * l.S + j], (unsigned long long)(c << sh));
            if (sh + bw > 64) atomicOr(&lds[(w + 1) * l.S + j], (unsigned long long)(c >> (64 - sh)));
        }
    }
    sync();
}

// What follows block b's words at image offset off: the block index entry,
// the dvbp page meta and the for_f reference page.  Lanes t < NL of a group
// of NL lanes write them.
template <uint32_t NL = 64>
__device__ __forceinline__ void finish_block(const emit_layout &l, const emit_plan &pl, uint64_t b, uint32_t bw,
                                             uint64_t off, uint64_t ref, const uint64_t *refs, const uint64_t *start,
                                             uint8_t *out, uint64_t *index, uint64_t *refs_out, uint32_t t)
{
    const uint64_t fb = ldiv(b, l.bpo);
    if (t == 0) index[b] = (off << 8) | bw;
    // dynamic_vbp page meta (dynamic_vbp.h:216-255)
    if (l.leaf == MS_DYNAMIC_VBP) {
        uint64_t q, call_end;
        if (l.kind == MS_DYNAMIC_VBP) {
            if (l.K) {
                const uint64_t bpc = ldiv(l.K, l.B);
                q = lmod(b, bpc);
                call_end = b - q + bpc;
                if (call_end > pl.nb) call_end = pl.nb;
            } else {
                q = b;
                call_end = pl.nb;
            }
        } else {
            q = lmod(b, l.bpo);
            call_end = b - q + l.bpo;
        }
        const uint64_t qp = lmod(q, l.P);
        const uint64_t bpf = b - qp;                                      // first block of the page
        const uint64_t meta = out_pos(l, start, bpf) + hdr_of(l, bpf) - l.P; // meta bytes end the header
        if (t == 0) out[meta + qp] = (uint8_t)bw;
        if (b == bpf) {
            const uint64_t npage = call_end - bpf < l.P ? call_end - bpf : l.P;
            for (uint64_t x = npage + t; x < l.P; x += NL) out[meta + x] = (uint8_t)MS_VBP_BW_NOBLOCK;
        }
    }
    // for_f reference page (for.h:207-233)
    if (l.kind == MS_FOR && lmod(b, l.bpo) == 0) {
        if (t == 0) refs_out[fb] = ref;
        const uint64_t fpc = l.K ? ldiv(l.K, l.L) : 0;
        const uint64_t fq = l.K ? lmod(fb, fpc) : fb;
        if (lmod(fq, l.FP) == 0) {
            uint64_t fcall_end = l.K ? fb - lmod(fb, fpc) + fpc : pl.nfb;
            if (fcall_end > pl.nfb) fcall_end = pl.nfb;
            const uint64_t nfp = fcall_end - fb < l.FP ? fcall_end - fb : l.FP;
            uint64_t *rp = (uint64_t *)(out + out_pos(l, start, b));
            for (uint64_t x = t; x < l.FP; x += NL) rp[x] = x < nfp ? refs[fb + x] : (x == nfp ? ~0ull : 0ull);
        }
    }
}

// Packs innermost block b (one wave, lane t) at image offset off: its words
// are assembled in lds (B words) and written out, then finish_block.
template <class G, class Sync>
__device__ __forceinline__ void pack_block(const emit_layout &l, const emit_plan &pl, uint64_t b, uint32_t bw,
                                           uint64_t off, const G &get, uint64_t lo, uint64_t ref, const uint64_t *refs,
                                           const uint64_t *start, unsigned long long *lds, uint8_t *out,
                                           uint64_t *index, uint64_t *refs_out, uint32_t t, const Sync &sync)
{
    assemble_block(l, bw, get, lo, ref, lds, t, sync);
    const uint64_t words = l.B * bw / 64;
    uint64_t *dst = (uint64_t *)(out + off);
    for (uint64_t w = t; w < words; w += 64) dst[w] = lds[w];
    sync();
    finish_block(l, pl, b, bw, off, ref, refs, start, out, index, refs_out, t);
}

// Bit width and header+payload bytes of every innermost block.
// With d_nb the blocks past the column's own (*d_nb, written here) are left
// alone, for a scan sized by that count; without it they get size 0.
__global__ __launch_bounds__(64) void k_block_sizes(emit_layout l, const uint64_t *v, const uint64_t *d_m,
                                                    const uint64_t *refs, uint64_t nb_bound, uint64_t *sz,
                                                    uint32_t *bws, uint64_t *d_nb)
{
    const emit_plan pl = plan_of(l, *d_m);
    const uint32_t t = threadIdx.x;
    if (d_nb) {
        if (blockIdx.x == 0 && t == 0) *d_nb = pl.nb;
        if (nb_bound > pl.nb) nb_bound = pl.nb;
    }
    for (uint64_t b = blockIdx.x; b < nb_bound; b += gridDim.x) {
        if (b >= pl.nb) {
            if (t == 0) { sz[b] = 0; bws[b] = 0; }
            continue;
        }
        uint32_t bw = l.bw;
        if (l.leaf == MS_DYNAMIC_VBP) {
            const uint64_t ref = l.kind == MS_FOR ? refs[b / l.bpo] : 0;
            uint64_t lo;
            const uint64_t *src = chunk_src(l, v, b * l.B, lo);
            bw = block_bw(l, [&](uint64_t gi) { return src[gi]; }, lo, ref, t);
        }
        if (t == 0) {
            sz[b] = hdr_of(l, b) + l.B * bw / 8;
            bws[b] = bw;
        }
    }
}

// Packs one innermost block per wave.  Dynamic LDS: B 64-bit words.
__global__ __launch_bounds__(64) void k_pack_blocks(emit_layout l, const uint64_t *v, const uint64_t *d_m,
                                                    const uint64_t *refs, const uint64_t *start, const uint32_t *bws,
                                                    uint8_t *out, uint64_t *index, uint64_t *refs_out)
{
    extern __shared__ unsigned long long lds[];
    const emit_plan pl = plan_of(l, *d_m);
    const uint32_t t = threadIdx.x;
    for (uint64_t b = blockIdx.x; b < pl.nb; b += gridDim.x) {
        const uint32_t bw = bws[b];
        const uint64_t off = out_pos(l, start, b) + hdr_of(l, b);
        if (off + 8 * (l.B * bw / 64) > l.cap) {   // uniform per wave
            if (t == 0) emit_overflow(l);
            continue;
        }
        uint64_t lo;
        const uint64_t *src = chunk_src(l, v, b * l.B, lo);
        const uint64_t ref = l.kind == MS_FOR ? refs[b / l.bpo] : 0;
        pack_block(l, pl, b, bw, off, [&](uint64_t gi) { return src[gi]; }, lo, ref, refs, start, lds, out, index,
                   refs_out, t, [] { __syncthreads(); });
    }
}

// Sizes and packed words from a select's flags, one innermost block per
// wave (dynamic LDS: B packed words, then the B + pred gathered values).
// Block b's words go to stage + b B, its size to sz[b], its width to
// bws[b]; *d_nb receives the number of blocks (the scan's length).  The
// positions read by rank later go to pos: a delta tile's predecessors
// (gathered with the block the tile starts at) and, by workgroup 0 after
// its blocks, the tail behind the compressed part.
__global__ __launch_bounds__(64) void k_flag_stage(emit_layout l, flag_src fs, const uint64_t *d_m,
                                                   const uint64_t *refs, const uint64_t *d_total, uint64_t *d_nb,
                                                   uint64_t *sz, uint32_t *bws, uint64_t *stage, uint64_t *pos)
{
    extern __shared__ unsigned long long lds[];
    unsigned long long *fvals = lds + l.B;
    const emit_plan pl = plan_of(l, *d_m);
    const uint32_t t = threadIdx.x;
    const uint64_t nunits = *fs.sf.d_units;
    if (blockIdx.x == 0 && t == 0) *d_nb = pl.nb;
    for (uint64_t b = blockIdx.x; b < pl.nb; b += gridDim.x) {
        const uint64_t r0 = flag_r0(l, fs, b), lo = b * l.B;
        gather_ranks(fs.sf, nunits, fs.ustart[b], r0, lo + l.B - r0,
                     [&](uint64_t i, uint64_t row) { fvals[i] = row; });
        __syncthreads();
        if (fs.pred && lo > 0 && lo % MS_DELTA_TILE == 0)
            for (uint32_t i = t; i < fs.pred; i += 64) pos[r0 + i] = fvals[i];
        const uint64_t ref = l.kind == MS_FOR ? refs[b / l.bpo] : 0;
        const auto get = [&](uint64_t gi) -> uint64_t { return fvals[gi - r0]; };
        const uint32_t bw = block_bw(l, get, lo, ref, t);
        if (t == 0) {
            sz[b] = hdr_of(l, b) + l.B * bw / 8;
            bws[b] = bw;
        }
        assemble_block(l, bw, get, lo, ref, lds, t, [] { __syncthreads(); });
        const uint64_t words = l.B * bw / 64;
        uint64_t *dst = stage + b * l.B;
        for (uint64_t w = t; w < words; w += 64) dst[w] = lds[w];
        __syncthreads();
    }
    if (blockIdx.x == 0) {
        const uint64_t total = *d_total, r0 = pl.m_c;
        const uint64_t cnt = total > r0 ? total - r0 : 0;
        if (cnt) gather_ranks(fs.sf, nunits, fs.ustart[pl.nb], r0, cnt,
                              [&](uint64_t i, uint64_t row) { pos[r0 + i] = row; });
    }
}

// Moves each staged block to its offset in the image and writes what
// follows it (index entry, page meta, reference page).  A group of 16
// lanes takes a block, so a wave has four blocks' loads in flight; four
// waves per workgroup.
__global__ __launch_bounds__(256) void k_flag_place(emit_layout l, const uint64_t *d_m, const uint64_t *refs,
                                                    const uint64_t *start, const uint32_t *bws,
                                                    const uint64_t *stage, uint8_t *out, uint64_t *index,
                                                    uint64_t *refs_out)
{
    constexpr uint32_t NL = 16;
    const emit_plan pl = plan_of(l, *d_m);
    const uint32_t t = threadIdx.x % NL;
    const uint64_t step = (uint64_t)gridDim.x * (256 / NL);
    for (uint64_t b = (uint64_t)blockIdx.x * (256 / NL) + threadIdx.x / NL; b < pl.nb; b += step) {
        const uint64_t *src = stage + b * l.B;
        const uint32_t bw = bws[b];
        const uint64_t off = out_pos(l, start, b) + hdr_of(l, b);
        const uint64_t words = l.B * bw / 64;
        if (off + 8 * words > l.cap) {
            if (t == 0) emit_overflow(l);
            continue;
        }
        uint64_t *dst = (uint64_t *)(out + off);
        for (uint64_t w = t; w < words; w += NL) dst[w] = src[w];
        const uint64_t ref = l.kind == MS_FOR ? refs[ldiv(b, l.bpo)] : 0;
        finish_block<NL>(l, pl, b, bw, off, ref, refs, start, out, index, refs_out, t);
    }
}

// Static bit width: every output word straight from its codes.
__global__ __launch_bounds__(WG) void k_pack_static(emit_layout l, const uint64_t *v, const uint64_t *d_m,
                                                    uint8_t *out)
{
    const emit_plan pl = plan_of(l, *d_m);
    const uint64_t bw = l.bw, S = l.S;
    const uint64_t nwords = pl.m_c * bw / 64;
    if (nwords * 8 > l.cap) {
        if (blockIdx.x == 0 && threadIdx.x == 0) emit_overflow(l);
        return;
    }
    uint64_t *o = (uint64_t *)out;
    for (uint64_t W = (uint64_t)blockIdx.x * WG + threadIdx.x; W < nwords; W += (uint64_t)gridDim.x * WG) {
        const uint64_t j = W % S, w = W / S;
        const uint64_t b0 = 64 * w, b1 = 64 * w + 64;
        uint64_t k = (b0 + bw - 1) / bw;          // first code starting in this word
        uint64_t word = 0;
        if (k > 0) {
            const uint64_t kc = k - 1;            // code crossing in from the previous word
            if (kc * bw + bw > b0) word |= v[kc * S + j] >> (b0 - kc * bw);
        }
        for (; k * bw < b1; k++) word |= v[k * S + j] << (k * bw - b0);
        o[W] = word;
    }
}

// The end of an emission in one launch: the output's meta (block 0), the
// delta_f tile carries (carries non-null) and the raw rest behind the gap;
// every workgroup derives the gap's end itself.  start / bws are null for
// static_vbp_f.
// With d_flag (a select's split): values [*d_m, *d_total) are appended raw
// behind the output when *d_flag (select_compr.h:209-250).
__global__ __launch_bounds__(WG) void k_emit_tail(emit_layout l, const uint64_t *v, const uint64_t *d_m,
                                                  const uint64_t *start, const uint32_t *bws, ms_dev_meta *meta,
                                                  uint64_t *carries, uint8_t *out,
                                                  const uint64_t *d_total, const uint64_t *d_flag)
{
    const emit_plan pl = plan_of(l, *d_m);
    uint64_t C;
    if (l.kind == MS_STATIC_VBP) C = pl.m_c * l.bw / 8;
    else if (pl.nb == 0) C = 0;
    else C = start[pl.nb - 1] + hdr_of(l, pl.nb - 1) + l.B * bws[pl.nb - 1] / 8;
    const uint64_t R = ms_align64(C + l.gap);
    const uint64_t rest = pl.m - pl.m_c;
    const bool fits = R + 8 * rest <= l.cap;
    const uint64_t tid = (uint64_t)blockIdx.x * WG + threadIdx.x, nth = (uint64_t)gridDim.x * WG;
    const uint64_t app = rest ? R + 8 * rest : R;   // the write-iterator's append offset
    const bool appending = d_flag && *d_flag;
    const uint64_t total = appending ? *d_total : pl.m;
    const bool afits = !appending || app + 8 * (total - pl.m) <= l.cap;
    if (tid == 0) {
        if (!fits || !afits) emit_overflow(l);
        const bool app_done = appending && afits;
        meta->count = app_done ? total : pl.m;
        meta->size_compr = C;
        meta->size_used = app_done ? app + 8 * (total - pl.m) : rest ? R + 8 * rest : C;
        meta->aux[0] = app;
        meta->aux[1] = R;
    }
    if (appending && afits) {
        uint64_t *dst = (uint64_t *)(out + app);
        for (uint64_t i = pl.m + tid; i < total; i += nth) dst[i - pl.m] = v[i];
    }
    if (carries) {
        const uint64_t ntiles = (pl.m_c + MS_DELTA_TILE - 1) / MS_DELTA_TILE;
        for (uint64_t i = tid; i < ntiles * 8; i += nth) {
            const uint64_t tile = i / 8, j = i % 8;
            carries[i] = (tile == 0 || j >= l.dstep) ? 0ull : v[tile * MS_DELTA_TILE - l.dstep + j];
        }
    }
    if (fits) {
        uint64_t *dst = (uint64_t *)(out + R);
        for (uint64_t i = tid; i < rest; i += nth) dst[i] = v[pl.m_c + i];
    }
}

// The emit layout of an output column written as `chunk`-value calls.
static emit_layout out_layout(ms_col *out, uint64_t chunk)
{
    const ms_format_desc &f = out->f;
    const ms_geom &g = out->g;
    emit_layout l = {};
    l.kind = f.kind;
    l.leaf = g.leaf;
    l.bw = g.bw;
    l.S = g.lanes;
    l.dstep = g.dstep;
    l.B = g.inner_bs;
    l.P = g.leaf_page;
    l.bs = g.bs;
    l.gap = g.gap;
    l.K = chunk;
    l.cap = out->size_alloc;
    l.status = &out->meta->status;
    if (f.kind == MS_DELTA || f.kind == MS_FOR) {
        l.L = g.outer_block;
        l.FP = g.outer_page;
        l.bpo = g.outer_block / g.inner_bs;
        l.E = f.kind == MS_FOR ? (f.step ? f.step : g.lanes) : 1;
    } else {
        l.L = l.B;
        l.bpo = 1;
    }
    return l;
}

// ------------------------------------------------------------------
// Single-pass emission of 8-lane 512-value blocks (every DEFAULT_* cascade
// and dynamic_vbp_f<512, P, 8>): a block's offset depends on the widths of
// all blocks before it, so sizes and packing used to read the values twice
// (for_f three times: its references first).  Here a wave keeps 4 blocks
// (2048 values, one delta tile) in registers and a workgroup's 32 blocks
// are one tile of a look-back over the tiles' byte totals.  A tile is packed
// into LDS before its offset is known, and written out a tile later: its
// look-back runs when the workgroup's next tile has published its total, so
// a workgroup does not wait for every earlier tile's values to arrive.
// Bound by HBM (values read once, the image written once).  Measured, kernel
// time of all passes before and of this one: dynamic_vbp_f of 2^27 values
// 630 -> 277 us (4.9 TB/s), delta_f 547 -> 246 us, for_f of 10^8 values
// 703 -> 208 us; without the deferred look-back 319 / 290 / 251 us, with
// tiles of 16 blocks (4 waves) 342 / 303 / 239 us.
// ------------------------------------------------------------------
typedef unsigned long long op_u64x2 __attribute__((ext_vector_type(2)));
constexpr uint32_t OP_WAVES = 8;                 // waves per workgroup
constexpr uint32_t OP_WB = 4;                    // blocks per wave
constexpr uint32_t OP_TILE = OP_WAVES * OP_WB;   // blocks per tile
constexpr uint32_t OP_B = 512, OP_S = 8;
constexpr uint32_t OP_SLOT = 256;                // LDS words per block: codes of up to 32 bits

// Thread (g, j) holds codes 8 g .. 8 g + 7 of lane j (at most 32 bits each):
// 8 bw bits that start at byte g bw of the lane's stream.  They are ORed
// into the block's words (cleared here), two codes at a time and with one
// LDS atomic per word touched.
__device__ __forceinline__ void op_pack(uint32_t bw, const uint64_t (&c)[8], unsigned long long *lds, uint32_t t)
{
    const uint32_t byte0 = (t >> 3) * bw;
    for (uint32_t i = t; i < 4 * bw; i += 64) ((op_u64x2 *)lds)[i] = op_u64x2{0, 0};
    wave_lds_sync();
    unsigned long long *p = lds + (byte0 >> 3) * 8 + (t & 7);
    uint32_t sh = (byte0 & 7) * 8;
    uint64_t acc = 0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const uint64_t x = (uint64_t)(uint32_t)c[2 * q] | ((uint64_t)(uint32_t)c[2 * q + 1] << bw);
        acc |= x << sh;
        const uint32_t n = sh + 2 * bw;
        if (n >= 64) {
            atomicOr(p, (unsigned long long)acc);
            p += 8;
            acc = n > 64 ? x >> (64 - sh) : 0ull;        // n > 64 only with sh > 0
        }
        sh = n & 63;
    }
    if (sh) atomicOr(p, (unsigned long long)acc);
    wave_lds_sync();
}

// Words of the launch's look-back state: the ticket counter, a word per
// tile, then (a column-level dynamic_vbp_f) a page start per page.
static uint64_t op_tiles(uint64_t nb_bound) { return nb_bound / OP_TILE + 1; }

// The n blocks of 512 values at src into x (thread (g, j): codes 8 g .. of
// lane j); `before` = lane j's value in front of them (delta_f, g = 0).
template <uint32_t KIND>
__device__ __forceinline__ void op_load(const uint64_t *src, uint32_t n, bool first, uint32_t t,
                                        uint64_t (&x)[OP_WB][8], uint64_t &before)
{
    const uint64_t *p = src + (t >> 3) * 64 + (t & 7);
#pragma unroll
    for (uint32_t k = 0; k < OP_WB; k++) {
#pragma unroll
        for (uint32_t q = 0; q < 8; q++) x[k][q] = k < n ? gload(p + k * OP_B + q * 8) : 0ull;
    }
    before = KIND == MS_DELTA && n && !first && t < 8 ? gload(src - 8 + t) : 0ull;
}

__device__ __forceinline__ void op_copy(uint32_t bw, const unsigned long long *lds, uint8_t *dst, uint32_t t)
{
    // written once, more than the caches hold (283 -> 276 us for 2^27 values)
    for (uint32_t i = t; i < 4 * bw; i += 64)
        __builtin_nontemporal_store(((const op_u64x2 *)lds)[i], (op_u64x2 *)dst + i);
}

// A block of a wave that holds codes of more than 32 bits, which the LDS
// slots have no room for: its values are read again (they are warm in the
// caches) once its offset is known, two at a time so that this rare path
// does not set the kernel's register budget.
template <uint32_t KIND>
__device__ __forceinline__ void op_wide_block(const uint64_t *src, bool first, uint64_t ref, uint32_t bw,
                                              unsigned long long *lds, uint8_t *dst, uint32_t t)
{
    const uint32_t g = t >> 3, words = 8 * bw;
    for (uint32_t i = t; i < words; i += 64) lds[i] = 0;
    wave_lds_sync();
    const uint64_t *p = src + g * 64 + (t & 7);
    uint32_t bit = g * 8 * bw;
#pragma unroll 1
    for (uint32_t q = 0; q < 8; q += 2) {
        const bool start = KIND == MS_DELTA && first && g == 0 && q == 0;   // no value in front
        uint64_t a = gload(p + q * 8), b = gload(p + q * 8 + 8), before = 0;
        if (KIND == MS_DELTA && !start) before = gload(p + q * 8 - 8);
        if (KIND == MS_DELTA) {
            b -= a;
            a -= before;
        }
        if (KIND == MS_FOR) {
            a -= ref;
            b -= ref;
        }
#pragma unroll
        for (uint32_t h = 0; h < 2; h++) {
            const uint64_t c = h ? b : a;
            unsigned long long *w = lds + (bit >> 6) * 8 + (t & 7);
            const uint32_t sh = bit & 63;
            atomicOr(w, (unsigned long long)(c << sh));
            if (sh + bw > 64) atomicOr(w + 8, (unsigned long long)(c >> (64 - sh)));
            bit += bw;
        }
    }
    wave_lds_sync();
    op_copy(bw, lds, dst, t);
    wave_lds_sync();
}

// refs_out: for_f's references, delta_f's tile carries (a wave's 4 blocks
// are one tile).  The last tile writes the column's meta and the raw rest.
template <uint32_t KIND>
__global__ __launch_bounds__(OP_WAVES * 64, 4) void k_emit_onepass(emit_layout l, const uint64_t *v, const uint64_t *d_m,
                                                                 uint64_t *state, uint64_t tiles_bound,
                                                                 ms_dev_meta *meta, uint8_t *out, uint64_t *index,
                                                                 uint64_t *refs_out)
{
    __shared__ __align__(16) unsigned long long s_words[OP_WAVES][OP_WB * OP_SLOT];
    __shared__ uint64_t s_ref[4][OP_TILE], s_tile, s_base, s_page;   // s_ref: of the last tiles, in turn
    __shared__ uint32_t s_tot[OP_WAVES];
    const emit_plan pl = plan_of(l, *d_m);
    const uint32_t t = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t g = t >> 3;
    uint64_t *tiles = state + 1, *pages = tiles + tiles_bound;
    const uint64_t ntiles = pl.nb ? (pl.nb + OP_TILE - 1) / OP_TILE : 1;
    const bool paged = KIND == MS_DYNAMIC_VBP && l.K == 0;   // pages of many tiles
    const uint32_t bpo = (uint32_t)l.bpo;                     // 1, 2 or 4
    const uint32_t P = (uint32_t)l.P, FP = (uint32_t)l.FP, fpb = FP * bpo;
    const auto first_of = [&](uint64_t tile) -> uint64_t { return tile * OP_TILE + w * OP_WB; };
    const auto blocks_of = [&](uint64_t b0) -> uint32_t {    // blocks of a wave that starts at b0
        return b0 >= pl.nb ? 0u : pl.nb - b0 < OP_WB ? (uint32_t)(pl.nb - b0) : OP_WB;
    };
    if (blockIdx.x >= ntiles) return;   // as many workgroups as tiles take tickets
    if (threadIdx.x == 0) s_tile = lb_ticket(state);
    __syncthreads();
    uint64_t tile = readlane64(s_tile, 0);   // uniform: addresses and branches stay scalar
    __syncthreads();
    if (tile >= ntiles) return;
    uint64_t x[OP_WB][8], before;
    op_load<KIND>(v + first_of(tile) * OP_B, blocks_of(first_of(tile)), first_of(tile) == 0, t, x, before);
    // the packed tile that waits for its offset: its blocks' widths and
    // headers, the bytes of the waves before this one and of the tile
    uint64_t ptile = ~0ull;
    uint32_t pbw[OP_WB] = {0, 0, 0, 0}, phdr[OP_WB] = {0, 0, 0, 0}, pmine = 0, ptotal = 0;
    for (uint32_t turn = 0;; turn = (turn + 1) & 3) {
        const bool have = tile < ntiles;
        uint32_t bw[OP_WB] = {0, 0, 0, 0}, hdr[OP_WB] = {0, 0, 0, 0};
        if (have) {
            // the workgroup's next tile
            if (threadIdx.x == 0) s_tile = lb_ticket(state);
            const uint64_t b0 = first_of(tile);
            const uint32_t n = blocks_of(b0);
            if (KIND == MS_DELTA) {
                // the code before a thread's first one is lane t - 8's last
                // (of the previous block for g = 0)
                if (n && g == 0) refs_out[b0 / OP_WB * 8 + t] = before;
#pragma unroll
                for (uint32_t k = 0; k < OP_WB; k++) {
                    const uint64_t last = __shfl(x[k][7], (int)((t + 56) & 63), MS_WAVE);
                    const uint64_t prev = g ? last : before;
                    before = last;
#pragma unroll
                    for (uint32_t q = 7; q > 0; q--) x[k][q] -= x[k][q - 1];
                    x[k][0] -= prev;
                }
            }
            if (KIND == MS_FOR) {
                // signed minimum per lane, then unsigned over the lanes (for.h:121-161)
                int64_t sm[OP_WB];
#pragma unroll
                for (uint32_t k = 0; k < OP_WB; k++) {
                    sm[k] = (int64_t)x[k][0];
#pragma unroll
                    for (uint32_t q = 1; q < 8; q++) sm[k] = (int64_t)x[k][q] < sm[k] ? (int64_t)x[k][q] : sm[k];
                }
                if (bpo >= 2) {
                    sm[0] = sm[1] < sm[0] ? sm[1] : sm[0];
                    sm[2] = sm[3] < sm[2] ? sm[3] : sm[2];
                }
                if (bpo == 4) sm[0] = sm[2] < sm[0] ? sm[2] : sm[0];
                uint64_t ref = 0;
#pragma unroll
                for (uint32_t k = 0; k < OP_WB; k++) {
                    if ((k & (bpo - 1)) == 0) {
#pragma unroll
                        for (uint32_t o = 8; o < 64; o <<= 1) {
                            const int64_t y = (int64_t)__shfl_xor((uint64_t)sm[k], (int)o, MS_WAVE);
                            sm[k] = y < sm[k] ? y : sm[k];
                        }
                        uint64_t r = (uint64_t)sm[k];
#pragma unroll
                        for (uint32_t o = 1; o < 8; o <<= 1) {
                            const uint64_t y = __shfl_xor(r, (int)o, MS_WAVE);
                            r = y < r ? y : r;
                        }
                        ref = readlane64(r == ~0ull ? r - 1 : r, 0);
                        if (t == 0 && k < n) {
                            s_ref[turn][(w * OP_WB + k) / bpo] = ref;
                            refs_out[(b0 + k) / bpo] = ref;
                        }
                    }
#pragma unroll
                    for (uint32_t q = 0; q < 8; q++) x[k][q] -= ref;
                }
            }
            // header bytes in front of the wave's blocks: page meta at every
            // call of the inner layout, for_f's reference page (of at least
            // 8 references) at its page's first block
            const bool page0 = KIND == MS_DYNAMIC_VBP ? (paged ? lmod(b0, P) == 0 : true)
                             : KIND == MS_FOR         ? (l.K || (b0 & (fpb - 1)) == 0) : false;
            uint32_t bytes = 0;
#pragma unroll
            for (uint32_t k = 0; k < OP_WB; k++) {
                if (k >= n) continue;
                uint64_t o = 1;
#pragma unroll
                for (uint32_t q = 0; q < 8; q++) o |= x[k][q];
                bw[k] = dpp_max_u32(64 - __clzll(o));
                if (KIND == MS_DYNAMIC_VBP) hdr[k] = k == 0 && page0 ? P : 0;
                else hdr[k] = ((k & (bpo - 1)) == 0 ? P : 0) + (KIND == MS_FOR && k == 0 && page0 ? 8 * FP : 0);
                bytes += hdr[k] + OP_B / 8 * bw[k];
            }
            if (t == 0) s_tot[w] = bytes;
        }
        __syncthreads();
        uint64_t next = ~0ull;
        uint32_t mine = 0, total = 0;
        if (have) {
            next = readlane64(s_tile, 0);
#pragma unroll
            for (uint32_t i = 0; i < OP_WAVES; i++) {
                if (i == w) mine = total;
                total += __builtin_amdgcn_readfirstlane(s_tot[i]);
            }
            if (w == 0) lb_publish(tiles, tile, total);
        }
        if (w == 0 && ptile != ~0ull) {
            uint64_t words[LB_SPAN];
            lb_request(tiles, (int64_t)ptile - 1, words);
            const uint64_t base = lb_exclusive(tiles, ptile, ptotal, words);
            uint64_t page = 0;
            if (paged) {
                // the page's first tile publishes where the page starts; its
                // others (whose tickets are later) wait for that
                const uint64_t pg = ldiv(first_of(ptile), P);
                if (first_of(ptile) == pg * P) {
                    page = base;
                    if (t == 0) lb_store(pages + pg, base + 1);
                } else {
                    while ((page = lb_load(pages + pg)) == 0) __builtin_amdgcn_s_sleep(1);
                    page--;
                }
            }
            if (t == 0) {
                s_base = base;
                s_page = page;
            }
        }
        __syncthreads();
        if (ptile != ~0ull) {
            const uint64_t tbase = readlane64(s_base, 0), page = readlane64(s_page, 0);
            const uint64_t b0 = first_of(ptile);
            const uint32_t n = blocks_of(b0), pturn = (turn + 3) & 3;
            const bool wide = pbw[0] > 32 || pbw[1] > 32 || pbw[2] > 32 || pbw[3] > 32;
            const bool page0 = phdr[0] > P;
            uint64_t at = tbase + pmine;
#pragma unroll
            for (uint32_t k = 0; k < OP_WB; k++) {
                if (k >= n) break;
                const uint64_t b = b0 + k, off = at + phdr[k];
                at = off + OP_B / 8 * pbw[k];
                if (at > l.cap) {                       // uniform per wave
                    if (t == 0) emit_overflow(l);
                    continue;
                }
                if (wide) op_wide_block<KIND>(v + b * OP_B, b == 0,
                                              KIND == MS_FOR ? s_ref[pturn][(w * OP_WB + k) / bpo] : 0ull, pbw[k],
                                              s_words[w], out + off, t);
                else op_copy(pbw[k], s_words[w] + k * OP_SLOT, out + off, t);
                if (t == 0) index[b] = (off << 8) | pbw[k];
                if (paged) {
                    if (t == 0) out[page + lmod(b, P)] = (uint8_t)pbw[k];
                } else if (phdr[k]) {
                    // a call's page meta: its blocks are this wave's
                    const uint32_t nin = KIND == MS_DYNAMIC_VBP ? n : bpo;
                    uint64_t m = ~0ull;
#pragma unroll
                    for (uint32_t i = OP_WB; i-- > 0;)
                        if (i >= k && i - k < nin) m = (m << 8) | pbw[i];
                    uint64_t *mp = (uint64_t *)(out + off - P);
                    for (uint32_t i = t; i < P / 8; i += 64) mp[i] = i ? ~0ull : m;
                    if (KIND == MS_FOR && k == 0 && page0) {
                        // reference page (for.h:207-233): its blocks are this
                        // wave's (a write-iterator's call) or this tile's
                        const uint64_t left = pl.nfb - b / bpo;
                        const uint32_t nfp = l.K ? n / bpo : left < FP ? (uint32_t)left : FP;
                        uint64_t *rp = (uint64_t *)(out + off - phdr[k]);
                        for (uint32_t i = t; i < FP; i += 64)
                            rp[i] = i < nfp ? s_ref[pturn][w * OP_WB / bpo + i] : (i == nfp ? ~0ull : 0ull);
                    }
                }
            }
            if (ptile == ntiles - 1) {
                const uint64_t C = tbase + ptotal, R = ms_align64(C + l.gap), rest = pl.m - pl.m_c;
                const bool fits = R + 8 * rest <= l.cap;
                if (threadIdx.x == 0) {
                    if (!fits) emit_overflow(l);
                    meta->count = pl.m;
                    meta->size_compr = C;
                    meta->size_used = rest ? R + 8 * rest : C;
                    meta->aux[0] = rest ? R + 8 * rest : R;   // the write-iterator's append offset
                    meta->aux[1] = R;
                }
                if (fits)
                    for (uint64_t i = threadIdx.x; i < rest; i += OP_WAVES * 64)
                        ((uint64_t *)(out + R))[i] = v[pl.m_c + i];
                if (paged && pl.nb && C <= l.cap)             // blocks the last page lacks
                    for (uint64_t i = lmod(pl.nb - 1, P) + 1 + threadIdx.x; i < P; i += OP_WAVES * 64)
                        out[page + i] = (uint8_t)MS_VBP_BW_NOBLOCK;
            }
        }
        if (!have) return;
        wave_lds_sync();   // the packed words go where the written ones were
        if (bw[0] <= 32 && bw[1] <= 32 && bw[2] <= 32 && bw[3] <= 32) {
#pragma unroll
            for (uint32_t k = 0; k < OP_WB; k++)
                if (bw[k]) op_pack(bw[k], x[k], s_words[w] + k * OP_SLOT, t);
        }
#pragma unroll
        for (uint32_t k = 0; k < OP_WB; k++) {
            pbw[k] = bw[k];
            phdr[k] = hdr[k];
        }
        pmine = mine;
        ptotal = total;
        ptile = tile;
        tile = next;
        if (tile < ntiles)
            op_load<KIND>(v + first_of(tile) * OP_B, blocks_of(first_of(tile)), first_of(tile) == 0, t, x, before);
    }
}

// Clears an output's meta and a launch's look-back state.
__global__ __launch_bounds__(WG) void k_emit_init(uint64_t *meta, uint64_t *state, uint64_t words)
{
    if (blockIdx.x == 0 && threadIdx.x < 32) meta[threadIdx.x] = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * WG + threadIdx.x; i < words; i += (uint64_t)gridDim.x * WG) state[i] = 0;
}

// Layouts the single-pass emission takes: blocks of one wave's shape whose
// page meta lies within a wave (or, column-level dynamic_vbp_f, in pages of
// whole tiles) and whose reference pages lie within a tile.
static bool onepass_ok(const emit_layout &l)
{
    if (l.leaf != MS_DYNAMIC_VBP || l.S != OP_S || l.B != OP_B || l.P % 64 || l.P > (1u << 24) || l.FP > (1u << 24) || l.cmap || l.cout) return false;
    if (l.K != 0 && l.K != OP_WB * OP_B) return false;
    if (l.kind == MS_DYNAMIC_VBP) return true;
    if (l.bpo != 1 && l.bpo != 2 && l.bpo != 4) return false;
    if (l.kind == MS_DELTA) return l.dstep == OP_S;
    return l.kind == MS_FOR && l.E == OP_S && l.FP % 8 == 0 && (l.K != 0 || OP_TILE % (l.FP * l.bpo) == 0);
}

static int launch_emit_onepass(ms_col *out, const emit_layout &l, const uint64_t *d_v, const uint64_t *d_m,
                               uint64_t m_bound, temps &sc)
{
    hipStream_t s = sc.s;
    const uint64_t nb_bound = m_bound / l.B + 1, tiles = op_tiles(nb_bound);
    const uint64_t words = 1 + tiles + (l.kind == MS_DYNAMIC_VBP && l.K == 0 ? nb_bound / l.P + 1 : 0);
    if (out->index_cap < nb_bound - 1 || (l.kind == MS_FOR && out->refs_cap < m_bound / l.L) ||
        (l.kind == MS_DELTA && out->refs_cap < (m_bound / MS_DELTA_TILE + 1) * 8))
        return ms_fail(MS_ERR_CAPACITY, "emit: index capacity");
    uint64_t *state = (uint64_t *)sc.get(words * 8);
    if (!state) return ms_fail(MS_ERR_NOMEM, "emit scratch");
    hipLaunchKernelGGL(k_emit_init, dim3(grid_for(words, WG * 4ull, 256)), dim3(WG), 0, s, (uint64_t *)out->meta,
                       state, words);
    MS_HIP(hipGetLastError());
    auto k = l.kind == MS_DYNAMIC_VBP ? k_emit_onepass<MS_DYNAMIC_VBP>
           : l.kind == MS_DELTA       ? k_emit_onepass<MS_DELTA>
                                      : k_emit_onepass<MS_FOR>;
    const uint32_t resident = resident_grid((const void *)k, OP_WAVES * 64);
    hipLaunchKernelGGL(k, dim3(grid_for(tiles, 1, resident)), dim3(OP_WAVES * 64), 0, s, l, d_v, d_m, state, tiles,
                       out->meta, out->data, out->index, out->refs);
    MS_HIP(hipGetLastError());
    return MS_OK;
}

int launch_emit(ms_col *out, const uint64_t *d_v, const uint64_t *d_m, uint64_t m_bound, uint64_t chunk, temps &sc)
{
    hipStream_t s = sc.s;
    const ms_format_desc &f = out->f;
    const emit_layout l = out_layout(out, chunk);
    if (f.kind != MS_STATIC_VBP && l.B * 8 > 65536)
        return ms_fail(MS_ERR_INVALID, "emit: innermost blocks above 8192 values are not supported");
    if (onepass_ok(l)) return launch_emit_onepass(out, l, d_v, d_m, m_bound, sc);
    MS_TRY(launch_fill_u64((uint64_t *)out->meta, 32, 0, s));
    const uint64_t nb_bound = m_bound / l.B + 1;
    if (f.kind == MS_STATIC_VBP) {
        hipLaunchKernelGGL(k_pack_static, dim3(grid_for(m_bound * l.bw / 64 + 1, WG * 4ull)), dim3(WG), 0, s, l, d_v,
                           d_m, out->data);
        MS_HIP(hipGetLastError());
        hipLaunchKernelGGL(k_emit_tail, dim3(grid_for(l.bs + l.K + 1, WG, 64)), dim3(WG), 0, s, l, d_v, d_m,
                           (const uint64_t *)nullptr, (const uint32_t *)nullptr, out->meta,
                           (uint64_t *)nullptr, out->data, (const uint64_t *)nullptr, (const uint64_t *)nullptr);
    } else {
        uint64_t *sz = (uint64_t *)sc.get(nb_bound * 8 + 64);
        uint64_t *start = (uint64_t *)sc.get(nb_bound * 8 + 64);
        uint32_t *bws = (uint32_t *)sc.get(nb_bound * 4 + 64);
        uint64_t *refs = nullptr;
        if (!sz || !start || !bws) return ms_fail(MS_ERR_NOMEM, "emit scratch");
        if (f.kind == MS_FOR) {
            refs = (uint64_t *)sc.get((m_bound / l.L + 1) * 8 + 64);
            if (!refs) return ms_fail(MS_ERR_NOMEM, "emit scratch");
            hipLaunchKernelGGL(k_for_refs<false>, dim3(grid_for(m_bound / l.L + 1, 1, 65536)), dim3(64), 0, s, l, d_v,
                               flag_src{}, d_m, refs);
            MS_HIP(hipGetLastError());
        }
        uint64_t *d_nb = (uint64_t *)sc.get(64);
        if (!d_nb) return ms_fail(MS_ERR_NOMEM, "emit scratch");
        hipLaunchKernelGGL(k_block_sizes, dim3(grid_for(nb_bound, 1, 65536)), dim3(64), 0, s, l, d_v, d_m,
                           (const uint64_t *)refs, nb_bound, sz, bws, d_nb);
        MS_HIP(hipGetLastError());
        MS_TRY(launch_exclusive_scan_n(sz, start, d_nb, 0, nb_bound, sc));
        if (out->index_cap < nb_bound - 1 || (f.kind == MS_FOR && out->refs_cap < m_bound / l.L))
            return ms_fail(MS_ERR_CAPACITY, "emit: index capacity");
        hipLaunchKernelGGL(k_pack_blocks, dim3(grid_for(nb_bound, 1, 65536)), dim3(64), l.B * 8, s, l, d_v, d_m,
                           (const uint64_t *)refs, (const uint64_t *)start, (const uint32_t *)bws, out->data,
                           out->index, out->refs);
        MS_HIP(hipGetLastError());
        if (f.kind == MS_DELTA && out->refs_cap < (m_bound / MS_DELTA_TILE + 1) * 8)
            return ms_fail(MS_ERR_CAPACITY, "emit: delta carries capacity");
        const uint64_t tail = std::max<uint64_t>(l.bs + l.K + 1, m_bound / MS_DELTA_TILE * 8 + 8);
        hipLaunchKernelGGL(k_emit_tail, dim3(grid_for(tail, WG, 1024)), dim3(WG), 0, s, l, d_v, d_m,
                           (const uint64_t *)start, (const uint32_t *)bws, out->meta,
                           f.kind == MS_DELTA ? out->refs : (uint64_t *)nullptr, out->data, (const uint64_t *)nullptr,
                           (const uint64_t *)nullptr);
    }
    MS_HIP(hipGetLastError());
    return MS_OK;
}

// ------------------------------------------------------------------
// Emission straight from a select's flags.
// ------------------------------------------------------------------
bool emit_flags_ok(const ms_format_desc &f)
{
    if (f.kind != MS_DYNAMIC_VBP && f.kind != MS_DELTA && f.kind != MS_FOR) return false;
    const ms_geom g = ms_make_geom(f);
    if (g.leaf != MS_DYNAMIC_VBP || g.inner_bs == 0 || g.inner_bs > 2048 || 2048 % g.inner_bs) return false;
    if (f.kind == MS_DELTA && (g.dstep == 0 || g.dstep > 64 || g.dstep >= g.inner_bs)) return false;
    if (f.kind == MS_FOR && g.outer_block > 4096) return false;
    return true;
}

int launch_emit_flags(ms_col *out, const sel_flags &sf, const sel_split &sp, uint64_t *pos, uint64_t m_bound,
                      uint64_t chunk, temps &sc)
{
    const uint64_t *d_m = sp.d_na, *d_total = sp.d_cnt;
    hipStream_t s = sc.s;
    const ms_format_desc &f = out->f;
    if (!emit_flags_ok(f)) return ms_fail(MS_ERR_INVALID, "emit from flags: format kind %u", f.kind);
    const emit_layout l = out_layout(out, chunk);
    const uint64_t nb_bound = m_bound / l.B + 1;
    flag_src fs = {};
    fs.sf = sf;
    fs.pred = f.kind == MS_DELTA ? l.dstep : 0;
    // blocks whose first read rank exists: b B - pred < m_bound
    const uint64_t starts = (m_bound + fs.pred) / l.B + 2;
    uint32_t *ustart = (uint32_t *)sc.get(starts * 4 + 64);
    uint64_t *sz = (uint64_t *)sc.get(nb_bound * 8 + 64);
    uint64_t *start = (uint64_t *)sc.get(nb_bound * 8 + 64);
    uint32_t *bws = (uint32_t *)sc.get(nb_bound * 4 + 64);
    if (!ustart || !sz || !start || !bws) return ms_fail(MS_ERR_NOMEM, "emit scratch");
    if (sf.units_bound >= (1ull << 32)) return ms_fail(MS_ERR_CAPACITY, "emit from flags: %llu units",
                                                      (unsigned long long)sf.units_bound);
    fs.ustart = ustart;
    hipLaunchKernelGGL(k_flag_starts, dim3(grid_for(sf.units_bound, WG)), dim3(WG), 0, s, l, fs, sp, starts, ustart,
                       out->meta);
    MS_HIP(hipGetLastError());
    uint64_t *refs = nullptr;
    if (f.kind == MS_FOR) {
        refs = (uint64_t *)sc.get((m_bound / l.L + 1) * 8 + 64);
        if (!refs) return ms_fail(MS_ERR_NOMEM, "emit scratch");
        hipLaunchKernelGGL(k_for_refs<true>, dim3(grid_for(m_bound / l.L + 1, 1, 65536)), dim3(64), l.L * 8, s, l,
                           (const uint64_t *)nullptr, fs, d_m, refs);
        MS_HIP(hipGetLastError());
    }
    const uint32_t vals_lds = (uint32_t)((l.B + fs.pred) * 8);
    const uint32_t fl_grid = grid_for(nb_bound, 1, 65536);
    uint64_t *d_nb = (uint64_t *)sc.get(64);
    if (!d_nb) return ms_fail(MS_ERR_NOMEM, "emit scratch");
    // every block's words staged at a fixed slot of B words, so the packing
    // happens in the same pass as the sizes and placing them is a copy
    uint64_t *stage = (uint64_t *)sc.get(nb_bound * l.B * 8 + 64);
    if (!stage) return ms_fail(MS_ERR_NOMEM, "emit scratch");
    hipLaunchKernelGGL(k_flag_stage, dim3(fl_grid), dim3(64), l.B * 8 + vals_lds, s, l, fs, d_m,
                       (const uint64_t *)refs, d_total, d_nb, sz, bws, stage, pos);
    MS_HIP(hipGetLastError());
    MS_TRY(launch_exclusive_scan_n(sz, start, d_nb, 0, nb_bound, sc));
    if (out->index_cap < nb_bound - 1 || (f.kind == MS_FOR && out->refs_cap < m_bound / l.L))
        return ms_fail(MS_ERR_CAPACITY, "emit: index capacity");
    hipLaunchKernelGGL(k_flag_place, dim3(grid_for(nb_bound, 16, 16384)), dim3(256), 0, s, l, d_m,
                       (const uint64_t *)refs, (const uint64_t *)start, (const uint32_t *)bws,
                       (const uint64_t *)stage, out->data, out->index, out->refs);
    MS_HIP(hipGetLastError());
    if (f.kind == MS_DELTA && out->refs_cap < (m_bound / MS_DELTA_TILE + 1) * 8)
        return ms_fail(MS_ERR_CAPACITY, "emit: delta carries capacity");
    const uint64_t tail = std::max<uint64_t>(l.bs + l.K + 1, m_bound / MS_DELTA_TILE * 8 + 8);
    hipLaunchKernelGGL(k_emit_tail, dim3(grid_for(tail, WG, 1024)), dim3(WG), 0, s, l, (const uint64_t *)pos, d_m,
                       (const uint64_t *)start, (const uint32_t *)bws, out->meta,
                       f.kind == MS_DELTA ? out->refs : (uint64_t *)nullptr, out->data, d_total,
                       (const uint64_t *)sp.d_flag);
    MS_HIP(hipGetLastError());
    return MS_OK;
}

// ------------------------------------------------------------------
// Chunked emission: one morph_batch call per chunk of K values.
// ------------------------------------------------------------------
static emit_layout chunk_layout(const chunk_emit &ce)
{
    const ms_format_desc &f = ce.f;
    const ms_geom g = ms_make_geom(f);
    emit_layout l = {};
    l.kind = f.kind;
    l.leaf = g.leaf;
    l.bw = g.bw;
    l.S = g.lanes;
    l.dstep = g.dstep;
    l.B = g.inner_bs;
    l.P = g.leaf_page;
    l.bs = g.bs;
    l.K = ce.K;
    l.cap = ~0ull;
    if (f.kind == MS_DELTA || f.kind == MS_FOR) {
        l.L = g.outer_block;
        l.FP = g.outer_page;
        l.bpo = g.outer_block / g.inner_bs;
        l.E = f.kind == MS_FOR ? (f.step ? f.step : g.lanes) : 1;
    } else {
        l.L = l.B;
        l.bpo = 1;
    }
    l.cmap = ce.cmap;
    return l;
}

__global__ __launch_bounds__(WG) void k_chunk_bytes(const uint64_t *start, uint64_t bpc, uint64_t n, uint64_t *csz)
{
    for (uint64_t c = (uint64_t)blockIdx.x * WG + threadIdx.x; c < n; c += (uint64_t)gridDim.x * WG)
        csz[c] = start[(c + 1) * bpc] - start[c * bpc];
}

int launch_chunk_sizes(chunk_emit &ce, uint64_t *d_csz, temps &sc)
{
    hipStream_t s = sc.s;
    const emit_layout l = chunk_layout(ce);
    const ms_geom g = ms_make_geom(ce.f);
    if (g.leaf != MS_DYNAMIC_VBP || (ce.f.kind != MS_DYNAMIC_VBP && ce.f.kind != MS_DELTA && ce.f.kind != MS_FOR))
        return ms_fail(MS_ERR_INVALID, "chunked emission: dynamic_vbp_f or a cascade over it");
    if (ce.K == 0 || ce.K % l.L || ce.K % l.B || l.B * 8 > 65536)
        return ms_fail(MS_ERR_INVALID, "chunked emission: chunk of %llu values", (unsigned long long)ce.K);
    const uint64_t m = ce.nchunks * ce.K;
    ce.nb = m / l.B;
    ce.d_m = (uint64_t *)sc.get(64);
    ce.sz = (uint64_t *)sc.get((ce.nb + 1) * 8 + 64);
    ce.start = (uint64_t *)sc.get((ce.nb + 1) * 8 + 64);
    ce.bws = (uint32_t *)sc.get((ce.nb + 1) * 4 + 64);
    ce.refs = nullptr;
    if (!ce.d_m || !ce.sz || !ce.start || !ce.bws) return ms_fail(MS_ERR_NOMEM, "chunked emission scratch");
    MS_TRY(launch_fill_u64(ce.d_m, 1, m, s));
    if (ce.nchunks == 0) return MS_OK;
    if (ce.f.kind == MS_FOR) {
        ce.refs = (uint64_t *)sc.get((m / l.L + 1) * 8 + 64);
        if (!ce.refs) return ms_fail(MS_ERR_NOMEM, "chunked emission scratch");
        hipLaunchKernelGGL(k_for_refs<false>, dim3(grid_for(m / l.L, 1, 65536)), dim3(64), 0, s, l, ce.v, flag_src{},
                           ce.d_m, ce.refs);
        MS_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(k_block_sizes, dim3(grid_for(ce.nb + 1, 1, 65536)), dim3(64), 0, s, l, ce.v, ce.d_m,
                       (const uint64_t *)ce.refs, ce.nb + 1, ce.sz, ce.bws, (uint64_t *)nullptr);
    MS_HIP(hipGetLastError());
    MS_TRY(launch_exclusive_scan(ce.sz, ce.start, ce.nb + 1, sc));
    if (d_csz) {
        hipLaunchKernelGGL(k_chunk_bytes, dim3(grid_for(ce.nchunks, WG)), dim3(WG), 0, s, (const uint64_t *)ce.start,
                           ce.K / l.B, ce.nchunks, d_csz);
        MS_HIP(hipGetLastError());
    }
    return MS_OK;
}

int launch_chunk_pack(const chunk_emit &ce, const uint64_t *d_cout, uint8_t *out, uint64_t cap, uint64_t *status,
                      uint64_t *index_out, uint64_t *refs_out, hipStream_t s)
{
    if (ce.nchunks == 0) return MS_OK;
    emit_layout l = chunk_layout(ce);
    l.cout = d_cout;
    l.cap = cap;
    l.status = status;
    hipLaunchKernelGGL(k_pack_blocks, dim3(grid_for(ce.nb, 1, 65536)), dim3(64), l.B * 8, s, l, ce.v,
                       (const uint64_t *)ce.d_m, (const uint64_t *)ce.refs, (const uint64_t *)ce.start,
                       (const uint32_t *)ce.bws, out, index_out, refs_out);
    MS_HIP(hipGetLastError());
    return MS_OK;
}

// ------------------------------------------------------------------
// rle_f (rle.h:95-147): maximal runs, the values read once.  A wave takes
// 2048 values (16 rows of 128), a workgroup's 8 waves are one tile.  A run
// belongs to the wave holding its first value (its head).  A wave compacts
// its heads (value, place) into LDS while the tile's number of heads goes
// through the look-back, and the pairs are written a tile later, as in
// k_emit_onepass: a run's length is the distance to the next head, which
// only a tile's last run leaves to k_rle_close.  A wave of more heads than
// its LDS slots (runs shorter than 8 values on average) reads its values
// again for its pairs.
// Bound by HBM.  Measured for 2^26 values in runs of 64 on average, all
// passes before (a count and a write pass, a value per lane and load) and
// now: 459 -> 140 us (4.0 TB/s; 114 us without the look-back).
// ------------------------------------------------------------------
constexpr uint32_t RLE_WAVES = 8, RLE_ROWS = 16;
constexpr uint32_t RLE_WV = RLE_ROWS * 128;             // values per wave
constexpr uint32_t RLE_TILE = RLE_WAVES * RLE_WV;       // values per tile
constexpr uint32_t RLE_SLOT = 256;                      // heads per wave kept in LDS

// The n values at src, two consecutive ones per lane and row; `before` =
// the value in front of them.
__device__ __forceinline__ void rle_load(const uint64_t *src, uint32_t n, bool first, uint32_t t,
                                         op_u64x2 (&x)[RLE_ROWS], uint64_t &before)
{
    if (n == RLE_WV) {
#pragma unroll
        for (uint32_t r = 0; r < RLE_ROWS; r++) x[r] = gload((const op_u64x2 *)(src + 128 * r + 2 * t));
    } else {
#pragma unroll
        for (uint32_t r = 0; r < RLE_ROWS; r++) {
            const uint32_t i = 128 * r + 2 * t;
            x[r] = op_u64x2{0, 0};
            if (i + 1 < n) x[r] = gload((const op_u64x2 *)(src + i));
            else if (i < n) x[r].x = gload(src + i);
        }
    }
    before = first || !n ? 0ull : gload(src - 1);
}

// The pairs of a wave whose heads the LDS slots have no room for, from its
// n values at index i0; r = its first run.  A head writes its value and the
// length of the run before it; the wave's last run is left to the caller,
// its first value's index is returned.
__device__ __forceinline__ uint64_t rle_dense(const uint64_t *v, uint64_t i0, uint32_t n, uint64_t r, uint32_t t,
                                              uint64_t *out_w)
{
    uint64_t last = ~0ull;
#pragma unroll 1
    for (uint32_t o = 0; o < n; o += 64) {
        const uint64_t i = i0 + o + t;
        const bool in = o + t < n;
        const uint64_t x = in ? gload(v + i) : 0ull;
        const uint64_t y = in && i ? gload(v + i - 1) : 0ull;
        const bool head = in && (i == 0 || x != y);
        const uint64_t b = __ballot(head);
        if (head) {
            const uint64_t below = b & ((1ull << t) - 1ull);
            const uint64_t k = r + __popcll(below);
            out_w[2 * k] = x;
            if (below) out_w[2 * (k - 1) + 1] = i - (i0 + o + 63 - __clzll(below));
            else if (last != ~0ull) out_w[2 * (k - 1) + 1] = i - last;
        }
        if (b) last = i0 + o + 63 - __clzll(b);
        r += __popcll(b);
    }
    return last;
}

// cnt / first / roff: every tile's heads, its first head's index (~0:
// none) and its first run, for k_rle_close.
__global__ __launch_bounds__(RLE_WAVES * 64, 4) void k_rle_onepass(const uint64_t *v, const uint64_t *d_m,
                                                                   uint64_t *state, uint64_t *cnt, uint64_t *first,
                                                                   uint64_t *roff, uint64_t *out_w)
{
    __shared__ uint64_t s_val[2][RLE_WAVES][RLE_SLOT], s_tile, s_base;
    __shared__ uint16_t s_at[2][RLE_WAVES][RLE_SLOT];
    __shared__ uint32_t s_cnt[RLE_WAVES], s_first[4][RLE_WAVES];   // s_first: of the last tiles, in turn
    const uint64_t m = *d_m;
    const uint64_t ntiles = (m + RLE_TILE - 1) / RLE_TILE;
    const uint32_t t = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint64_t *tiles = state + 1;
    const auto first_of = [&](uint64_t tile) -> uint64_t { return tile * RLE_TILE + w * RLE_WV; };
    const auto values_of = [&](uint64_t i0) -> uint32_t {
        return i0 >= m ? 0u : m - i0 < RLE_WV ? (uint32_t)(m - i0) : RLE_WV;
    };
    if (blockIdx.x >= ntiles) return;   // as many workgroups as tiles take tickets
    if (threadIdx.x == 0) s_tile = lb_ticket(state);
    __syncthreads();
    uint64_t tile = readlane64(s_tile, 0);
    __syncthreads();
    if (tile >= ntiles) return;
    op_u64x2 x[RLE_ROWS];
    uint64_t before;
    rle_load(v + first_of(tile), values_of(first_of(tile)), first_of(tile) == 0, t, x, before);
    uint64_t ptile = ~0ull;                       // the tile that waits for its first run
    uint32_t pheads = 0, pmine = 0, ptotal = 0;   // its heads in this wave, in the waves before, in all
    for (uint32_t turn = 0;; turn = (turn + 1) & 3) {
        const bool have = tile < ntiles;
        uint32_t heads = 0;
        if (have) {
            if (threadIdx.x == 0) s_tile = lb_ticket(state);
            const uint64_t i0 = first_of(tile);
            const uint32_t n = values_of(i0);
            uint64_t *sv = s_val[turn & 1][w];
            uint16_t *sa = s_at[turn & 1][w];
            uint64_t carry = readlane64(before, 0);
#pragma unroll
            for (uint32_t r = 0; r < RLE_ROWS; r++) {
                const uint32_t i = 128 * r + 2 * t;
                const uint64_t a = x[r].x, b = x[r].y;
                // the value before a: lane t - 1's second (wave_shr:1)
                const uint32_t plo = (uint32_t)__builtin_amdgcn_update_dpp((int)(uint32_t)carry, (int)(uint32_t)b,
                                                                           0x138, 0xf, 0xf, false);
                const uint32_t phi = (uint32_t)__builtin_amdgcn_update_dpp((int)(uint32_t)(carry >> 32),
                                                                           (int)(uint32_t)(b >> 32), 0x138, 0xf, 0xf,
                                                                           false);
                const uint64_t p = ((uint64_t)phi << 32) | plo;
                carry = readlane64(b, 63);
                const bool ha = i < n && (a != p || i0 + i == 0), hb = i + 1 < n && b != a;
                const uint64_t Ha = __ballot(ha), Hb = __ballot(hb);
                if ((Ha | Hb) == 0) continue;
                const uint32_t ra = heads + lanes_below(Ha) + lanes_below(Hb), rb = ra + (ha ? 1u : 0u);
                if (ha && ra < RLE_SLOT) {
                    sv[ra] = a;
                    sa[ra] = (uint16_t)i;
                }
                if (hb && rb < RLE_SLOT) {
                    sv[rb] = b;
                    sa[rb] = (uint16_t)(i + 1);
                }
                heads += (uint32_t)__popcll(Ha) + (uint32_t)__popcll(Hb);
            }
            wave_lds_sync();
            if (t == 0) {
                s_cnt[w] = heads;
                s_first[turn][w] = heads ? w * RLE_WV + sa[0] : ~0u;
            }
        }
        __syncthreads();
        uint64_t next = ~0ull;
        uint32_t mine = 0, total = 0;
        if (have) {
            next = readlane64(s_tile, 0);
#pragma unroll
            for (uint32_t i = 0; i < RLE_WAVES; i++) {
                if (i == w) mine = total;
                total += __builtin_amdgcn_readfirstlane(s_cnt[i]);
            }
            if (w == 0) lb_publish(tiles, tile, total);
        }
        uint64_t words[LB_SPAN];
        const bool waits = w == 0 && ptile != ~0ull;
        if (waits) lb_request(tiles, (int64_t)ptile - 1, words);
        __builtin_amdgcn_sched_barrier(0);   // the words' loads stay in front of the values'
        if (next < ntiles)
            rle_load(v + first_of(next), values_of(first_of(next)), false, t, x, before);
        __builtin_amdgcn_sched_barrier(0);
        if (waits) {
            const uint64_t base = lb_exclusive(tiles, ptile, ptotal, words);
            if (t == 0) s_base = base;
        }
        __syncthreads();
        if (ptile != ~0ull) {
            const uint64_t tbase = readlane64(s_base, 0), i0 = first_of(ptile);
            const uint32_t pturn = (turn + 3) & 3;
            const uint64_t r0 = tbase + pmine;
            // the next head behind this wave's values, in the tile's other waves
            uint32_t nf = ~0u, tf = ~0u;
#pragma unroll
            for (uint32_t i = RLE_WAVES; i-- > 0;) {
                const uint32_t f = __builtin_amdgcn_readfirstlane(s_first[pturn][i]);
                tf = f < tf ? f : tf;
                if (i > w) nf = f < nf ? f : nf;
            }
            const uint64_t after = ptile * RLE_TILE + nf;
            if (pheads > RLE_SLOT) {
                const uint64_t last = rle_dense(v, i0, values_of(i0), r0, t, out_w);
                if (t == 0) out_w[2 * (r0 + pheads - 1) + 1] = nf == ~0u ? last : after - last;
            } else {
                const uint64_t *sv = s_val[pturn & 1][w];
                const uint16_t *sa = s_at[pturn & 1][w];
                for (uint32_t k = t; k < pheads; k += 64) {
                    op_u64x2 pr;
                    pr.x = sv[k];
                    if (k + 1 < pheads) pr.y = sa[k + 1] - sa[k];
                    else pr.y = nf == ~0u ? i0 + sa[k] : after - (i0 + sa[k]);
                    ((op_u64x2 *)out_w)[r0 + k] = pr;
                }
            }
            if (threadIdx.x == 0) {
                cnt[ptile] = ptotal;
                first[ptile] = tf == ~0u ? ~0ull : ptile * RLE_TILE + tf;
                roff[ptile] = tbase;
            }
        }
        if (!have) return;
        pheads = heads;
        pmine = mine;
        ptotal = total;
        ptile = tile;
        tile = next;
    }
}

// The length of every tile's last run, whose first value's index
// k_rle_onepass left in its place: up to the next tile's head (a wave per
// tile looks 64 tiles ahead at a time); then the column's meta.
__global__ __launch_bounds__(WG) void k_rle_close(const uint64_t *d_m, const uint64_t *cnt, const uint64_t *first,
                                                  const uint64_t *roff, uint64_t *out_w, ms_dev_meta *meta)
{
    const uint64_t m = *d_m;
    const uint64_t nt = (m + RLE_TILE - 1) / RLE_TILE;
    const uint32_t t = threadIdx.x & 63;
    const uint64_t step = (uint64_t)gridDim.x * (WG / 64);
    for (uint64_t c = (uint64_t)blockIdx.x * (WG / 64) + (threadIdx.x >> 6); c < nt; c += step) {
        const uint64_t n = cnt[c];
        if (!n) continue;
        uint64_t next = m;
        for (uint64_t d = c + 1; d < nt; d += 64) {
            const uint64_t f = d + t < nt ? first[d + t] : ~0ull;
            const uint64_t b = __ballot(f != ~0ull);
            if (b) {
                next = __shfl(f, __builtin_ctzll(b), MS_WAVE);
                break;
            }
        }
        if (t == 0) {
            const uint64_t r = roff[c] + n - 1;
            out_w[2 * r + 1] = next - out_w[2 * r + 1];
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        const uint64_t runs = nt ? roff[nt - 1] + cnt[nt - 1] : 0;
        meta->count = m;
        meta->size_used = meta->size_compr = 16 * runs;
    }
}

int launch_rle_compress(ms_col *out, const uint64_t *d_v, const uint64_t *d_m, uint64_t m_bound, temps &sc)
{
    hipStream_t s = sc.s;
    if ((uintptr_t)d_v % 16) return ms_fail(MS_ERR_INVALID, "rle: values not aligned to 16 bytes");
    const uint64_t tiles = m_bound / RLE_TILE + 1;
    uint64_t *state = (uint64_t *)sc.get((1 + 4 * tiles) * 8);
    if (!state) return ms_fail(MS_ERR_NOMEM, "rle scratch");
    uint64_t *cnt = state + 1 + tiles, *first = cnt + tiles, *roff = first + tiles;
    hipLaunchKernelGGL(k_emit_init, dim3(grid_for(1 + tiles, WG * 4ull, 256)), dim3(WG), 0, s, (uint64_t *)out->meta,
                       state, 1 + tiles);
    MS_HIP(hipGetLastError());
    const uint32_t resident = resident_grid((const void *)k_rle_onepass, RLE_WAVES * 64);
    hipLaunchKernelGGL(k_rle_onepass, dim3(grid_for(tiles, 1, resident)), dim3(RLE_WAVES * 64), 0, s, d_v, d_m, state,
                       cnt, first, roff, (uint64_t *)out->data);
    MS_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_rle_close, dim3(grid_for(tiles, WG / 64)), dim3(WG), 0, s, d_m, (const uint64_t *)cnt,
                       (const uint64_t *)first, (const uint64_t *)roff, (uint64_t *)out->data, out->meta);
    MS_HIP(hipGetLastError());
    return MS_OK;
}

}  // namespace ms
