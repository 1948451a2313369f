// Specialised implicit-GEMM forward / dX convolution for the (k, stride, pad)
// pairs rustnn uses: 3x3/s1/p1, 3x3/s2/p1, 1x1/s2/p0 (and 1x1/s1/p0).
//
// Persistent workgroups walk a list of work items -- (tile of output
// positions, group of MB blocks of 32 output channels) -- and, per item, the
// source channels in chunks of CH.  Producer waves stage each (item, chunk)
// into one of two LDS buffers -- the zero-padded source window (x for
// forward, dY for dX) and the chunk's weights -- while the compute waves
// multiply the previous one; M = output channels, N = output positions (32
// per group), K = (channel, tap):
//   * 3x3: on the bf16 matrix cores, each float in three exact parts
//     (mfma_split.h); the producers load through registers and split;
//   * 1x1 (bound by memory): v_mfma_f32_32x32x2f32; the producers DMA
//     (buffer_load ... lds) the window as [channel quad][position][4] and the
//     weights in fragment order [mb][quad][tap][lane][4], one ds_read_b128
//     per 4 k-steps, lane half h carrying channel h*CH/2 + 4q + i.
//
// For dX with stride s the workgroup computes all s*s parity classes of its
// block positions from the same dY window, each tap feeding exactly one class
// accumulator (gather-form col2im: no atomics, every dX element written once).
//
// 3x3 at batch 128, packed weights, fp32 pipe -> here (us, forward / dX):
// 32 -> 32 @32x32 29.8 / 28.4 -> 23.4 / 22.9; 64 -> 64 @16x16 28.3 / 28.0 ->
// 20.3 / 20.5; 128 -> 128 @8x8 28.4 / 28.5 -> 23.6 / 23.3; 96 -> 96 @16x16
// 69.1 / 68.9 -> 37.5 / 37.7; stride 2 64 -> 128 @16x16 18.7 / 29.6 -> 20.4 /
// 24.0.  Without loads and splitting 17-21 us are left of the stride-1 ones:
// the ramp, LDS reads and MFMAs.  Errors against 64 bits 2-3 times smaller
// (32 -> 32 2.1e-7 / 3.0e-7 -> 0.9e-7 / 1.1e-7).
//
// Reference: conv.rs forward_image (168-203), dx_image (205-246) and the
// Conv2d batch drivers (nn.rs:166-250).
#include "conv_common.h"
#include "mfma_split.h"

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>

namespace {

constexpr int FAST_NW = 4;  // waves per workgroup

// 1x1: window DMA rows of 16 positions that one wave stages per channel quad:
// row u of wave w covers window positions (w + 4u)*16 .. +16.
constexpr int WIN_ROWS = 4;

struct FastArgs {
    const float *src;  // [N][CS][HS][WS]
    const float *w;    // [cout][cin][k][k]
    const float *wp;   // the same weights packed in slab order (conv_pack), or null
    int wpbytes;       // bytes of wp
    float *dst;        // [N][CD][HD][WD]
    int N, CS, HS, WS;
    int CD, HD, WD;
    int GA, GB;        // output block grid per image
    int TR, tiles_a, ntiles, ngroups;
    int CH, nchunks;   // source channels per stage (multiple of 8; 3x3: 8)
    int sm, sc;        // weight strides of output row m and source channel ch
    int wbytes;        // bytes of W
    int dymin, dxmin;  // smallest tap offsets (window origin)
    int lrow, lcol;    // window rows / columns per output row / column step
    int plane;         // window positions (multiple of 64) per channel quad or bf16 part
    int ppw;           // plane / 64: window rows per quad and wave, or 64-position groups
    int xwords;        // LDS words of the window: CH * plane (3x3: 3 parts of 8 bf16: 12 * plane)
    int stage;         // LDS words of one stage: window, then weight slabs
    TileGeo geo;       // window geometry in positions (chs unused)
    // 3x3: the two taps of each k step (one per lane half; -1 none) and their
    // window-position offsets
    int ptap[10], poff[10];
    uint32_t m_imgs, m_tiwp;  // FastDiv multipliers of geo.imgs and geo.TIWP
    int npart;         // store-pass statistics: partials per channel (= ntiles)
    ConvStats stats;   // store-pass statistics (forward with EPI = 1)
};

// Wave-uniform description of the stage being staged by DMA.
struct StageDMA {
    __amdgpu_buffer_rsrc_t rs;  // source images n0 .. n0 + IMGS
    float *buf;                 // stage buffer
    int c0, grp;                // first source channel, output-channel group
    int ebase;                  // element offset of window row 0 in image n0 (may be < 0)
    int ylo, yhi;               // window rows inside the source image
    int nimg;                   // images of the tile inside the batch
    int mlim;                   // output rows of the group inside [0, CD)
};

template <int K, int S, int P, bool DX, int SL>
__device__ __forceinline__ StageDMA stage_dma(const FastArgs &g, int item, int chunk,
                                              float *buf) {
    using T = ConvTaps<K, S, P, DX>;
    StageDMA d;
    const int tile = item % g.ntiles;
    d.grp = item / g.ntiles;
    const int n0 = (tile / g.tiles_a) * g.geo.IMGS;
    const int y0 = (tile % g.tiles_a) * g.TR * T::IS + g.dymin;
    const int rowstep = g.geo.rowstep;
    const long long img_elems = (long long)g.CS * g.HS * g.WS;
    d.rs = make_rsrc(g.src + (long long)n0 * img_elems,
                     (uint32_t)(min(g.N - n0, g.geo.IMGS) * img_elems * 4));
    d.buf = buf;
    d.c0 = chunk * g.CH;
    d.ebase = y0 * g.WS;
    d.ylo = y0 >= 0 ? 0 : (-y0 + rowstep - 1) / rowstep;
    d.yhi = min(g.geo.TIH, (g.HS - y0 + rowstep - 1) / rowstep);
    if (d.yhi < d.ylo) d.yhi = d.ylo;
    d.nimg = min(g.N - n0, g.geo.IMGS);
    d.mlim = g.CD - d.grp * SL * 32;
    return d;
}

// Per-lane constants of the DMA rows (computed once per workgroup).
struct LaneDMA {
    int toff[WIN_ROWS];   // window row u: element offset in the tile, channel lane&3
    int tmeta[WIN_ROWS];  // window row ty | img << 8 (ty = 255: no source element)
    int wl;               // weight row: (lane/4)*sm + (lane%4)*sc
    // Per work item: byte offset of window row u for channel lane&3 of
    // channel 0, or an offset >= 2^31 (beyond any buffer) when the row has
    // no source data.  A stage adds its channel's byte offset.
    uint32_t roff[WIN_ROWS];
};

__device__ __forceinline__ void lane_dma_init(const FastArgs &g, LaneDMA &L, int wave, int lane) {
    const TileGeo &t = g.geo;
    const int i = lane & 3;
#pragma unroll
    for (int u = 0; u < WIN_ROWS; u++) {
        const int pos = (wave + FAST_NW * u) * 16 + (lane >> 2);
        const uint32_t mi = g.m_imgs, mt = g.m_tiwp;  // FastDiv magic multipliers
        const int img = (int)(mi ? __umulhi((uint32_t)pos, mi) : (uint32_t)pos);
        const int rem = pos - img * t.imgs;
        const int ty = (int)(mt ? __umulhi((uint32_t)rem, mt) : (uint32_t)rem);
        const int col = rem - ty * t.TIWP;
        const int tx = t.deint ? (col < t.HALF ? 2 * col : 2 * (col - t.HALF) + 1) : col;
        const int x = g.dxmin + tx * t.colstep;
        const bool ok = u < g.ppw && img < t.IMGS && ty < t.TIH && tx < t.TIW && x >= 0 &&
                        x < g.WS;
        L.toff[u] = ((img * g.CS + i) * g.HS + ty * t.rowstep) * g.WS + x;
        L.tmeta[u] = ok ? (ty | (img << 8)) : 255;
    }
    L.wl = (lane >> 2) * g.sm + i * g.sc;
}

// 1x1 weight rows (mb, q) of stage d gathered from W in [cout][cin] order:
// 64-word row `wave` of each slab, lane l = wave*16 + lane/4.
template <int SL>
__device__ __forceinline__ void issue_w_gather(const FastArgs &g, const StageDMA &d,
                                               const LaneDMA &L, __amdgpu_buffer_rsrc_t rs_w,
                                               int q, int wave, int lane) {
    const int CP = g.CH >> 1, cq = g.CH >> 3;
#pragma unroll
    for (int mb = 0; mb < SL; mb++) {
        const int mrel = mb * 32 + (wave & 1) * 16;
        const int cbase = d.c0 + (wave >> 1) * CP + 4 * q;
        const bool ok = (lane >> 2) < d.mlim - mrel && (lane & 3) < g.CS - cbase;
        const int e = L.wl + (d.grp * SL * 32 + mrel) * g.sm + cbase * g.sc;
        const uint32_t off = max((uint32_t)e * 4u, ok ? 0u : DMA_OOB);
        float *dst = d.buf + g.xwords + (mb * cq + q) * 256 + wave * 64;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_w, (lds_ptr_t)dst, 4, off, 0, 0, 0);
    }
}

// The per-item window row offsets (LaneDMA::roff) of stage d's work item.
__device__ __forceinline__ void item_rows(const FastArgs &g, const StageDMA &d, LaneDMA &L) {
#pragma unroll
    for (int u = 0; u < WIN_ROWS; u++) {
        const int ty = L.tmeta[u] & 255, img = L.tmeta[u] >> 8;
        const bool rowok = (unsigned)(ty - d.ylo) < (unsigned)(d.yhi - d.ylo) && img < d.nimg;
        L.roff[u] = rowok ? (uint32_t)(L.toff[u] + d.ebase) * 4u : 0x80000000u;
    }
}

// ---------------------------------------------------------------------------
// 3x3 convolutions: products on the bf16 matrix cores (mfma_split.h).  A stage
// is 8 source channels; a k step of 16 is those 8 channels under two taps of
// one parity class, one tap per lane half (nine taps: the tenth half step
// meets zero weights).  The producers load the window and the weights into
// registers, split each float into its three bf16 parts and store the parts
// in operand order -- window [part][position][8 channels], weights [mb][tap
// pair][part][lane][8 channels] -- so that the compute waves only read
// operands (one ds_read_b128 each) and multiply, and a value is split once
// and not once per tap.
template <int S, int P, bool DX>
struct ConvPairs {
    using T = ConvTaps<3, S, P, DX>;
    static constexpr int N = 5;
    int t[2 * N] = {}, cls[N] = {};
    constexpr ConvPairs() {
        int n = 0;
        for (int c = 0; c < T::NCLS; c++) {
            int k = 0;
            for (int i = 0; i < 9; i++)
                if (T::cls(i) == c) {
                    if (k % 2 == 0) {
                        cls[n] = c;
                        t[2 * n] = i;
                        t[2 * n + 1] = -1;
                        n++;
                    } else {
                        t[2 * n - 1] = i;
                    }
                    k++;
                }
        }
    }
};

// s_waitcnt lgkmcnt(0) alone, and a barrier that waits for this wave's LDS
// accesses only (loads into registers stay in flight across it).
__device__ __forceinline__ void wait_lds() { __builtin_amdgcn_s_waitcnt(0xC07F); }
__device__ __forceinline__ void lds_barrier() {
    asm volatile("" ::: "memory");
    wait_lds();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

constexpr int SPLIT_U = 3;  // 64-position window groups per producer wave

// A producer wave's share of a stage: window groups dw, dw + 4, .. and weight
// tasks (mb, tap pair), dealt from the wave after the last window group.
template <int SL, int U, bool PK>
struct SplitStage {
    static constexpr int TW = (5 * SL + FAST_NW - 1) / FAST_NW;
    int toff[U], tmeta[U];  // as LaneDMA's, for channel 0
    uint32_t roff[U];       // byte offset for the work item, >= 2^31: none
    uint32_t woff[TW];      // byte offset of weight task u at chunk 0
    // Two stages in flight.  Every load is issued, past the end with an offset
    // out of range, so that the wait for one stage leaves the next in flight.
    float v[2][U][8], wv[2][TW][8];

    __device__ __forceinline__ static int wtask(const FastArgs &g, int u, int dw) {
        return ((dw - g.ppw) & (FAST_NW - 1)) + FAST_NW * u;
    }

    __device__ __forceinline__ void init(const FastArgs &g, int dw, int lane) {
        const TileGeo &t = g.geo;
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int pos = (dw + FAST_NW * u) * 64 + lane;
            const uint32_t mi = g.m_imgs, mt = g.m_tiwp;
            const int img = (int)(mi ? __umulhi((uint32_t)pos, mi) : (uint32_t)pos);
            const int rem = pos - img * t.imgs;
            const int ty = (int)(mt ? __umulhi((uint32_t)rem, mt) : (uint32_t)rem);
            const int col = rem - ty * t.TIWP;
            const int tx = t.deint ? (col < t.HALF ? 2 * col : 2 * (col - t.HALF) + 1) : col;
            const int x = g.dxmin + tx * t.colstep;
            const bool ok = pos < g.plane && img < t.IMGS && ty < t.TIH && tx < t.TIW && x >= 0 &&
                            x < g.WS;
            toff[u] = (img * g.CS * g.HS + ty * t.rowstep) * g.WS + x;
            tmeta[u] = ok ? (ty | (img << 8)) : 255;
        }
    }

    __device__ __forceinline__ void item(const FastArgs &g, const StageDMA &d, int dw, int lane) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int ty = tmeta[u] & 255, img = tmeta[u] >> 8;
            const bool ok = (unsigned)(ty - d.ylo) < (unsigned)(d.yhi - d.ylo) && img < d.nimg;
            roff[u] = ok ? (uint32_t)(toff[u] + d.ebase) * 4u : 0x80000000u;
        }
#pragma unroll
        for (int u = 0; u < TW; u++) {
            const int t = wtask(g, u, dw), mb = t / 5, pair = t - 5 * mb;
            const int blk = d.grp * SL + mb, m = blk * 32 + (lane & 31);
            if (t >= 5 * SL) {
                woff[u] = DMA_OOB;
            } else if (PK) {
                woff[u] = (uint32_t)(blk * g.nchunks * 2560 + pair * 512 + lane * 8) * 4u;
            } else {
                const int tap = lane < 32 ? g.ptap[2 * pair] : g.ptap[2 * pair + 1];
                woff[u] = tap >= 0 && m < g.CD ? (uint32_t)(m * g.sm + tap) * 4u : DMA_OOB;
            }
        }
    }

    // Loads the share of the item's `chunk` into register set B.
    template <int B>
    __device__ __forceinline__ void load(const FastArgs &g, const StageDMA &d, int chunk,
                                         __amdgpu_buffer_rsrc_t rs_w) {
        const uint32_t hsws4 = (uint32_t)(g.HS * g.WS) * 4u;
        const int c0 = chunk * 8;
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const bool live = c0 + c < g.CS;
            const uint32_t so = live ? (uint32_t)(c0 + c) * hsws4 : 0u;
#pragma unroll
            for (int u = 0; u < U; u++)
                v[B][u][c] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                    d.rs, live ? roff[u] : 0x80000000u, so, 0));
            if constexpr (!PK) {
                const uint32_t sw = live ? (uint32_t)((c0 + c) * g.sc) * 4u : 0u;
#pragma unroll
                for (int u = 0; u < TW; u++)
                    wv[B][u][c] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                        rs_w, live ? woff[u] : DMA_OOB, sw, 0));
            }
        }
        if constexpr (PK) {
            const uint32_t so = (uint32_t)chunk * 10240u;
#pragma unroll
            for (int u = 0; u < TW; u++)
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const u32x4 a =
                        __builtin_amdgcn_raw_buffer_load_b128(rs_w, woff[u] + 16 * q, so, 0);
#pragma unroll
                    for (int i = 0; i < 4; i++) wv[B][u][4 * q + i] = __uint_as_float(a[i]);
                }
        }
    }

    // Splits register set B into the stage buffer.
    template <int B>
    __device__ __forceinline__ void store(const FastArgs &g, float *buf, int dw, int lane) const {
        u32x4 *x = reinterpret_cast<u32x4 *>(buf), *w = reinterpret_cast<u32x4 *>(buf + g.xwords);
#pragma unroll
        for (int u = 0; u < U; u++)
            if (dw + FAST_NW * u < g.ppw) {
                const Bf3 p = bf3_split(v[B][u]);
                u32x4 *q = x + (dw + FAST_NW * u) * 64 + lane;
                q[0] = p.hi;
                q[g.plane] = p.mid;
                q[2 * g.plane] = p.lo;
                __builtin_amdgcn_sched_barrier(0);  // one group's parts live at a time
            }
#pragma unroll
        for (int u = 0; u < TW; u++) {
            const int t = wtask(g, u, dw);
            if (t < 5 * SL) {
                const Bf3 p = bf3_split_near(wv[B][u]);
                u32x4 *q = w + t * 192 + lane;
                q[0] = p.hi;
                q[64] = p.mid;
                q[128] = p.lo;
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
};

// A stage on the compute waves: vb the lane's window position of each
// 32-position group, po the offset of each pair's tap in its lane half.
template <int S, int P, bool DX, int NPW, int MB, int WM>
__device__ __forceinline__ void compute_split(
    const FastArgs &g, const float *__restrict__ buf, const int (&vb)[NPW], const int (&po)[5],
    f32x16 (&acc)[ConvTaps<3, S, P, DX>::NCLS][MB][NPW][2], int wave, int lane) {
    constexpr ConvPairs<S, P, DX> CP;
    constexpr int WP = FAST_NW / WM;
    const u32x4 *xs = reinterpret_cast<const u32x4 *>(buf);
    const u32x4 *ws = reinterpret_cast<const u32x4 *>(buf + g.xwords) + wave / WP * MB * 960 + lane;
    Bf3 a[MB], b[NPW];
    auto fetch = [&](int i, Bf3 (&fa)[MB], Bf3 (&fb)[NPW]) {
#pragma unroll
        for (int mb = 0; mb < MB; mb++) {
            const u32x4 *q = ws + (mb * 5 + i) * 192;
            fa[mb] = Bf3{q[0], q[64], q[128]};
        }
#pragma unroll
        for (int j = 0; j < NPW; j++) {
            const u32x4 *q = xs + vb[j] + po[i];
            fb[j] = Bf3{q[0], q[g.plane], q[2 * g.plane]};
        }
    };
    // With one block a wave there are registers to read the next pair while
    // this one is multiplied; with more, the MFMAs of a pair outlast the reads.
    constexpr bool AHEAD = NPW * MB == 1;
    if constexpr (AHEAD) fetch(0, a, b);
    static_for<0, 5>([&](auto pc) {
        constexpr int i = decltype(pc)::value, c = CP.cls[i];
        Bf3 na[MB], nb[NPW];
        if constexpr (!AHEAD)
            fetch(i, a, b);
        else if constexpr (i + 1 < 5)
            fetch(i + 1, na, nb);
        if constexpr (AHEAD) __builtin_amdgcn_sched_barrier(0);
        bf3_products([&](auto pick, auto kind) {
            constexpr int A = decltype(kind)::value;
#pragma unroll
            for (int mb = 0; mb < MB; mb++)
#pragma unroll
                for (int j = 0; j < NPW; j++)
                    acc[c][mb][j][A] = pick(a[mb], b[j], acc[c][mb][j][A]);
        });
        if constexpr (AHEAD && i + 1 < 5) {
#pragma unroll
            for (int mb = 0; mb < MB; mb++) a[mb] = na[mb];
#pragma unroll
            for (int j = 0; j < NPW; j++) b[j] = nb[j];
        }
    });
}

// The item's sums with fp32 MFMAs from global memory: for values that are not
// finite in the split (see bf3_nonfinite).
template <int S, int P, bool DX, int NPW, int MB, int WM>
__device__ __forceinline__ void compute_slow(
    const FastArgs &g, f32x16 (&acc)[ConvTaps<3, S, P, DX>::NCLS][MB][NPW][2], int wave, int lane,
    int grp, int a0, int n0) {
    using T = ConvTaps<3, S, P, DX>;
    constexpr int WP = FAST_NW / WM, SL = WM * MB;
    const int h = lane >> 5, l32 = lane & 31, tpix = g.TR * g.GB;
#pragma unroll
    for (int j = 0; j < NPW; j++) {
        const int p = ((wave % WP) * NPW + j) * 32 + l32;
        const int img = p / tpix, rem = p - img * tpix, r = rem / g.GB, cb = rem - r * g.GB;
        const int n = n0 + img, a = a0 + r;
        const bool live = p < g.geo.IMGS * tpix && n < g.N && a < g.GA;
#pragma unroll
        for (int mb = 0; mb < MB; mb++) {
            const int m = (grp * SL + (wave / WP) * MB + mb) * 32 + l32;
#pragma unroll
            for (int c = 0; c < T::NCLS; c++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc[c][mb][j][0][v] = 0.f;
#pragma unroll
            for (int c = 0; c < T::NCLS; c++)
#pragma unroll 1
                for (int t = 0; t < 9; t++) {
                    if (T::cls(t) != c) continue;
                    const int sy = a * T::IS + T::dy(t), sx = cb * T::IS + T::dx(t);
                    const bool in = live && sy >= 0 && sy < g.HS && sx >= 0 && sx < g.WS;
                    const float *xp = g.src + (((long long)n * g.CS + h) * g.HS + sy) * g.WS + sx;
                    const float *wp = g.w + (long long)m * g.sm + (long long)h * g.sc + t;
#pragma unroll 1
                    for (int k = h; k < g.CS + h; k += 2) {
                        const float b = in && k < g.CS ? *xp : 0.f;
                        const float wt = m < g.CD && k < g.CS ? *wp : 0.f;
                        acc[c][mb][j][0] =
                            __builtin_amdgcn_mfma_f32_32x32x2f32(wt, b, acc[c][mb][j][0], 0, 0, 0);
                        xp += 2ll * g.HS * g.WS;
                        wp += 2ll * g.sc;
                    }
                }
        }
    }
}

// One 1x1 stage of the GEMM on the MFMA waves: channel quads of the window `xs`
// and the weight slabs of the current buffer, the operands of the next quad
// read from LDS while the MFMAs of the current one run.
template <int NCLS, int NPW, int MB, int WM, int NACC>
__device__ __forceinline__ void compute_stage(const FastArgs &g, const float *__restrict__ xs,
                                              const int (&vb)[NPW],
                                              f32x16 (&acc)[NCLS][MB][NPW][NACC], int wave,
                                              int lane) {
    const int CQ = g.CH >> 3;
    const int wslab = CQ * 256;
    const float *ws = xs + g.xwords + lane * 4;
    constexpr int WP = FAST_NW / WM;  // waves along positions
    const float *wsw = ws + (wave / WP) * MB * wslab;  // this wave's m-blocks

    auto fetch = [&](int q, float4 *fa, float4 *fb) {
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
            fa[mb] = *reinterpret_cast<const float4 *>(wsw + mb * wslab + q * 256);
        const float *xq = xs + q * g.plane * 4;
#pragma unroll
        for (int j = 0; j < NPW; j++) fb[j] = *reinterpret_cast<const float4 *>(xq + vb[j]);
    };
    float4 ca[MB], cb[NPW];
    fetch(0, ca, cb);
    for (int q = 0; q < CQ; q++) {
        float4 na[MB], nb[NPW];
        if (q + 1 < CQ) fetch(q + 1, na, nb);
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int mb = 0; mb < MB; mb++)
#pragma unroll
                for (int j = 0; j < NPW; j++)
                    acc[0][mb][j][i % NACC] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                        ca[mb][i], cb[j][i], acc[0][mb][j][i % NACC], 0, 0, 0);
#pragma unroll
        for (int mb = 0; mb < MB; mb++) ca[mb] = na[mb];
#pragma unroll
        for (int j = 0; j < NPW; j++) cb[j] = nb[j];
    }
}

// All DMA of 1x1 stage `chunk` of the work item described by d (its window
// rows in L.roff) into `buf`, issued by producer wave `dw`: the window rows
// u = dw, dw + 4, ... of every channel quad, then the weights -- contiguous
// 1 KiB slabs of the packed copy, 16 bytes a lane, or gathered from W.
template <int SL>
__device__ __forceinline__ void issue_stage(const FastArgs &g, StageDMA d, float *buf, int chunk,
                                            const LaneDMA &L, __amdgpu_buffer_rsrc_t rs_w, int dw,
                                            int lane) {
    const int cq = g.CH >> 3;
    d.buf = buf;
    d.c0 = chunk * g.CH;
    const uint32_t hsws4 = (uint32_t)(g.HS * g.WS) * 4u;
    for (int hq = 0; hq < 2 * cq; hq++) {
        const int cb = d.c0 + 4 * hq;
        const uint32_t cbytes = (uint32_t)cb * hsws4;
        // lanes whose channel cb + lane%4 is beyond the source get no data
        const uint32_t chbad = g.CS - cb >= 4 ? 0u : ((lane & 3) >= g.CS - cb ? 0x80000000u : 0u);
        float *row0 = buf + (hq * g.plane + dw * 16) * 4;
#pragma unroll
        for (int u = 0; u < WIN_ROWS; u++)
            if (u < g.ppw)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    d.rs, (lds_ptr_t)(row0 + FAST_NW * u * 64), 4, (L.roff[u] + cbytes) | chbad, 0,
                    0, 0);
    }
    if (g.wp) {
        const __amdgpu_buffer_rsrc_t rs_p = make_rsrc(g.wp, (uint32_t)g.wpbytes);
        for (int k = dw; k < SL * cq; k += FAST_NW) {
            const int mb = k / cq, r = k - mb * cq;
            const uint32_t src =
                (uint32_t)(((d.grp * SL + mb) * g.nchunks + chunk) * cq + r) * 1024u;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_p, (lds_ptr_t)(buf + g.xwords + k * 256),
                                                     16, src + (uint32_t)lane * 16u, 0, 0, 0);
        }
    } else {
        for (int q = 0; q < cq; q++) issue_w_gather<SL>(g, d, L, rs_w, q, dw, lane);
    }
}

// Sums 4 values per lane over the 32 lanes of each half-wave: offsets 16 and
// 8 each keep half of the values, offsets 4, 2, 1 add the rest; lane l ends
// with the total of value 2*b4 + b3 (b = bits of l), the 8 lanes that share
// those bits holding the same total.  The order is fixed.
__device__ __forceinline__ double half_reduce4(const double (&x)[4], int l32) {
    const bool b4 = l32 & 16, b3 = l32 & 8;
    double a2[2];
#pragma unroll
    for (int i = 0; i < 2; i++)
        a2[i] = (b4 ? x[i + 2] : x[i]) + __shfl_xor(b4 ? x[i] : x[i + 2], 16, 64);
    double a1 = (b3 ? a2[1] : a2[0]) + __shfl_xor(b3 ? a2[0] : a2[1], 8, 64);
    a1 = a1 + __shfl_xor(a1, 4, 64);
    a1 = a1 + __shfl_xor(a1, 2, 64);
    return a1 + __shfl_xor(a1, 1, 64);
}

// The forward's store pass with the batch statistics' sums (see ConvStats):
// the same stores as the plain pass, with the accumulator registers taken 4
// at a time so that only 4 (sum y, sum y^2) pairs are live; each wave's
// totals over the item's positions, reduced over its lanes, are left in red
// (LDS) for the workgroup's fixed-order sum over its waves.
template <int K, int S, int P, int NPW, int MB, int WM, int NACC>
__device__ __forceinline__ void store_stats(
    const FastArgs &g, const f32x16 (&acc)[1][MB][NPW][NACC], int wave, int lane, int grp,
    int a0, int n0, double *__restrict__ red) {
    constexpr int VG = 4, WP = FAST_NW / WM, SL = WM * MB;
    const int h = lane >> 5, l32 = lane & 31;
    const int tpix = g.TR * g.GB, npix = g.geo.IMGS * tpix;
    const long long cst = (long long)g.HD * g.WD;
    static_for<0, 16 / VG>([&](auto gc) {
        constexpr int vbase = decltype(gc)::value * VG;
        double es[MB][2][VG];
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
#pragma unroll
            for (int u = 0; u < VG; u++) es[mb][0][u] = es[mb][1][u] = 0.0;
#pragma unroll
        for (int j = 0; j < NPW; j++) {
            const int p = ((wave % WP) * NPW + j) * 32 + l32;
            const int img = p / tpix, rem = p - img * tpix, r = rem / g.GB, cb = rem - r * g.GB;
            const int n = n0 + img, a = a0 + r;
            if (p >= npix || n >= g.N || a >= g.GA) continue;
            const long long o = ((long long)n * g.CD * g.HD + a) * g.WD + cb;
#pragma unroll
            for (int mb = 0; mb < MB; mb++) {
                f32x16 v16 = acc[0][mb][j][0];
                if constexpr (K == 1 && NACC == 2) v16 += acc[0][mb][j][1];
                static_for<0, VG>([&](auto uc) {
                    constexpr int u = decltype(uc)::value, v = vbase + u;
                    const int m = (grp * SL + (wave / WP) * MB + mb) * 32 + 8 * (v >> 2) + 4 * h +
                                  (v & 3);
                    if (m >= g.CD) return;
                    const float y = v16[v];
                    g.dst[o + m * cst] = y;
                    es[mb][0][u] += (double)y;
                    es[mb][1][u] += (double)y * (double)y;
                });
            }
        }
        // this wave's totals into red[wave % WP][channel of the group][kind]
        const int v = vbase + ((l32 >> 4) & 1) * 2 + ((l32 >> 3) & 1);
#pragma unroll
        for (int mb = 0; mb < MB; mb++) {
            const double t0 = half_reduce4(es[mb][0], l32), t1 = half_reduce4(es[mb][1], l32);
            const int cl = ((wave / WP) * MB + mb) * 32 + 8 * (v >> 2) + 4 * h + (v & 3);
            if ((l32 & 7) == 0) {
                red[((wave % WP) * 32 * SL + cl) * 2] = t0;
                red[((wave % WP) * 32 * SL + cl) * 2 + 1] = t1;
            }
        }
    });
}

// Waves 0..3 compute: WP = 4 / WM along positions (NPW groups of 32 each)
// times WM along output channels (MB blocks of 32 each).  Waves 4..7 only
// move data: producer wave 4 + w issues the DMA rows that the row tables
// assign to wave w, a whole stage at a time, so that the memory pipeline's
// back-pressure stalls a producer and never the MFMA issue of a compute
// wave.  One barrier per stage: when it completes, stage s has landed (each
// producer waited for its own DMA) and stage s - 1's buffer is free.
// EPI = 1: the forward's store pass also takes the batch statistics
// (store_stats, ConvStats), with one more barrier per work item that the
// producers match.
// 3x3 only: U window groups per producer wave, PK packed weights.
template <int K, int S, int P, bool DX, int NPW, int MB, int WM, int EPI, int U, bool PK>
__global__ __launch_bounds__(64 * FAST_NW * 2)
__attribute__((amdgpu_waves_per_eu((K == 3 ? S == 1 : EPI) ? 4 : 1))) void conv_fast_kernel(FastArgs g) {
    using T = ConvTaps<K, S, P, DX>;
    constexpr int NCLS = T::NCLS;
    // 1x1: a wave with a single output block alternates two accumulators so
    // that consecutive MFMAs do not depend on each other.  3x3: the products
    // of leading parts in one, the smaller ones in the other.
    constexpr int NACC = K == 3 || NCLS * NPW * MB == 1 ? 2 : 1;
    constexpr int WP = FAST_NW / WM, SL = WM * MB;
    extern __shared__ float smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_index();
    const int h = lane >> 5, l32 = lane & 31;
    const int CQ = g.CH >> 3;
    const int tpix = g.TR * g.GB, npix = g.geo.IMGS * tpix;
    const int nitems = g.ntiles * g.ngroups;
    if ((int)blockIdx.x >= nitems) return;

    if (wave >= FAST_NW) {
        // producer
        const int dw = wave - FAST_NW;
        if constexpr (K == 3) {
            const __amdgpu_buffer_rsrc_t rs_w =
                make_rsrc(PK ? g.wp : g.w, (uint32_t)(PK ? g.wpbytes : g.wbytes));
            SplitStage<SL, U, PK> L;
            L.init(g, dw, lane);
            // the cursor of the next stage to load; it stays on the last one
            int item = blockIdx.x, chunk = 0;
            StageDMA d = stage_dma<K, S, P, DX, SL>(g, item, 0, smem);
            L.item(g, d, dw, lane);
            auto next = [&]() {
                if (chunk + 1 < g.nchunks) {
                    chunk++;
                } else if (item + (int)gridDim.x < nitems) {
                    item += gridDim.x;
                    chunk = 0;
                    d = stage_dma<K, S, P, DX, SL>(g, item, 0, smem);
                    L.item(g, d, dw, lane);
                }
            };
            const int nst = (nitems - 1 - (int)blockIdx.x) / (int)gridDim.x * g.nchunks + g.nchunks;
            L.template load<0>(g, d, 0, rs_w);
            next();
            L.template load<1>(g, d, chunk, rs_w);
            int sc = 0;  // the stored stage's chunk
            auto stage = [&](auto bc) {
                constexpr int B = decltype(bc)::value;
                // buffer B: every wave is past the stage before last
                L.template store<B>(g, smem + B * g.stage, dw, lane);
                next();
                L.template load<B>(g, d, chunk, rs_w);
                lds_barrier();
                if (++sc == g.nchunks) {
                    sc = 0;
                    if constexpr (EPI != 0) lds_barrier();  // the compute waves' store-pass sums
                }
            };
            for (int s = 0; s < nst; s += 2) {
                stage(std::integral_constant<int, 0>{});
                if (s + 1 < nst) stage(std::integral_constant<int, 1>{});
            }
            return;
        } else {
        const __amdgpu_buffer_rsrc_t rs_w = make_rsrc(g.w, (uint32_t)g.wbytes);
        LaneDMA L;
        lane_dma_init(g, L, dw, lane);
        StageDMA d = stage_dma<K, S, P, DX, SL>(g, blockIdx.x, 0, smem);
        item_rows(g, d, L);
        issue_stage<SL>(g, d, smem, 0, L, rs_w, dw, lane);
        int s = 0;
        for (int item = blockIdx.x; item < nitems; item += gridDim.x) {
            for (int chunk = 0; chunk < g.nchunks; chunk++, s++) {
                dma_wait_barrier();
                float *nbuf = smem + ((s + 1) & 1) * g.stage;
                if (chunk + 1 < g.nchunks) {
                    issue_stage<SL>(g, d, nbuf, chunk + 1, L, rs_w, dw, lane);
                } else if (item + (int)gridDim.x < nitems) {
                    d = stage_dma<K, S, P, DX, SL>(g, item + gridDim.x, 0, nbuf);
                    item_rows(g, d, L);
                    issue_stage<SL>(g, d, nbuf, 0, L, rs_w, dw, lane);
                }
            }
            if constexpr (EPI != 0) __syncthreads();  // the compute waves' store-pass sums
        }
        return;
        }
    }

    // LDS word offset of this lane's channel half and window position for
    // each 32-position group (tile-relative: the same for every work item);
    // 3x3: the window position alone.
    int vb[NPW];
#pragma unroll
    for (int j = 0; j < NPW; j++) {
        int p = ((wave % WP) * NPW + j) * 32 + l32;
        if (p >= npix) p = 0;
        const int img = p / tpix, rem = p - img * tpix, r = rem / g.GB, c = rem - r * g.GB;
        const int pos = img * g.geo.imgs + r * g.lrow * g.geo.TIWP + c * g.lcol;
        vb[j] = K == 3 ? pos : (h * CQ * g.plane + pos) * 4;
    }
    int po[5];
    if constexpr (K == 3)
#pragma unroll
        for (int i = 0; i < 5; i++) po[i] = h ? g.poff[2 * i + 1] : g.poff[2 * i];

    f32x16 acc[NCLS][MB][NPW][NACC];
    int s = 0;
    for (int item = blockIdx.x; item < nitems; item += gridDim.x) {
#pragma unroll
        for (int c = 0; c < NCLS; c++)
#pragma unroll
            for (int mb = 0; mb < MB; mb++)
#pragma unroll
                for (int j = 0; j < NPW; j++)
#pragma unroll
                    for (int a = 0; a < NACC; a++)
#pragma unroll
                        for (int v = 0; v < 16; v++) acc[c][mb][j][a][v] = 0.f;
        for (int chunk = 0; chunk < g.nchunks; chunk++, s++) {
            // Stage s has landed and every wave is done with stage s-1, whose
            // buffer the producers fill with stage s+1 while stage s is computed.
            if constexpr (K == 3) {
                lds_barrier();
                compute_split<S, P, DX, NPW, MB, WM>(g, smem + (s & 1) * g.stage, vb, po, acc,
                                                     wave, lane);
                continue;
            } else {
            dma_wait_barrier();
            compute_stage<NCLS, NPW, MB, WM, NACC>(g, smem + (s & 1) * g.stage, vb, acc, wave, lane);
            }
        }
        // acc row 8*(v/4) + 4*h + v%4 = output channel in the block, column = position.
        const int tile = item % g.ntiles, grp = item / g.ntiles;
        const int a0 = (tile % g.tiles_a) * g.TR, n0 = (tile / g.tiles_a) * g.geo.IMGS;
        if constexpr (K == 3) {
            bool bad = false;
#pragma unroll
            for (int c = 0; c < NCLS; c++)
#pragma unroll
                for (int mb = 0; mb < MB; mb++)
#pragma unroll
                    for (int j = 0; j < NPW; j++) {
                        acc[c][mb][j][0] = (acc[c][mb][j][0] + acc[c][mb][j][1]) * BF3_DOWN;
#pragma unroll
                        for (int v = 0; v < 16; v++)
                            bad = bad || bf3_nonfinite(acc[c][mb][j][0][v]);
                    }
            if (__any(bad)) compute_slow<S, P, DX, NPW, MB, WM>(g, acc, wave, lane, grp, a0, n0);
        }
        if constexpr (EPI != 0) {
            // Store pass with the statistics' sums; then the WP position
            // waves' totals of each channel, summed in wave order, make partial
            // `tile` of the channel.  The barrier pairs with the producers'
            // one after the item.
            constexpr int NCH = 32 * SL;
            double *red = reinterpret_cast<double *>(smem + 2 * g.stage);
            store_stats<K, S, P, NPW, MB, WM, NACC>(g, acc, wave, lane, grp, a0, n0, red);
            if constexpr (K == 3)
                lds_barrier();
            else
                __syncthreads();
            for (int t = tid; t < 2 * NCH; t += 64 * FAST_NW) {
                const int cl = t >> 1, m = grp * NCH + cl;
                if (m >= g.CD) continue;
                double tot = red[t];
                for (int w = 1; w < WP; w++) tot += red[w * 2 * NCH + t];
                g.stats.part[((long long)m * g.npart + tile) * 2 + (t & 1)] = tot;
            }
            continue;
        }
#pragma unroll
        for (int j = 0; j < NPW; j++) {
            const int p = ((wave % WP) * NPW + j) * 32 + l32;
            if (p >= npix) continue;
            const int img = p / tpix, rem = p - img * tpix, r = rem / g.GB, cb = rem - r * g.GB;
            const int n = n0 + img, a = a0 + r;
            if (n >= g.N || a >= g.GA) continue;
            const long long cst = (long long)g.HD * g.WD;
            if constexpr (NCLS == 4) {
                // stride-2 dX: the two column classes of a row are adjacent in
                // dX, so one 8-byte store writes both (each line written once)
#pragma unroll
                for (int py = 0; py < 2; py++) {
                    const int y = 2 * a + py, x = 2 * cb;
                    if (y >= g.HD || x >= g.WD) continue;
                    float *dp = g.dst + ((long long)n * g.CD * g.HD + y) * g.WD + x;
                    const bool pair = (g.WD & 1) == 0;  // x + 1 < WD and 8-byte aligned
#pragma unroll
                    for (int mb = 0; mb < MB; mb++) {
                        f32x16 v0 = acc[2 * py][mb][j][0], v1 = acc[2 * py + 1][mb][j][0];
                        if constexpr (K == 1 && NACC == 2) {
                            v0 += acc[2 * py][mb][j][1];
                            v1 += acc[2 * py + 1][mb][j][1];
                        }
#pragma unroll
                        for (int v = 0; v < 16; v++) {
                            const int m = (grp * SL + (wave / WP) * MB + mb) * 32 + 8 * (v >> 2) + 4 * h + (v & 3);
                            if (m >= g.CD) continue;
                            if (pair) {
                                *reinterpret_cast<float2 *>(dp + m * cst) = float2{v0[v], v1[v]};
                            } else {
                                dp[m * cst] = v0[v];
                                if (x + 1 < g.WD) dp[m * cst + 1] = v1[v];
                            }
                        }
                    }
                }
            } else {
#pragma unroll
                for (int c = 0; c < NCLS; c++) {
                    const int y = a * T::OS + (DX ? c / S : 0), x = cb * T::OS + (DX ? c % S : 0);
                    if (y >= g.HD || x >= g.WD) continue;
                    float *dp = g.dst + ((long long)n * g.CD * g.HD + y) * g.WD + x;
#pragma unroll
                    for (int mb = 0; mb < MB; mb++) {
                        f32x16 v16 = acc[c][mb][j][0];
                        if constexpr (K == 1 && NACC == 2) v16 += acc[c][mb][j][1];
#pragma unroll
                        for (int v = 0; v < 16; v++) {
                            const int m = (grp * SL + (wave / WP) * MB + mb) * 32 + 8 * (v >> 2) + 4 * h + (v & 3);
                            if (m < g.CD) dp[m * cst] = v16[v];
                        }
                    }
                }
            }
        }
    }
}

struct FastPlan {
    int TR, IMGS, CH, NPW, MB, WM;
    int wpc;  // cap on resident workgroups per CU (0 = occupancy limit)
    size_t lds;
};

// Window geometry of a plan; returns the LDS bytes (two stage buffers), or
// 0 when the window does not fit the producers' registers.
template <int K, int S, int P, bool DX>
static size_t plan_geometry(const FastPlan &p, int GB, FastArgs &a) {
    using T = ConvTaps<K, S, P, DX>;
    int dymin = 1 << 20, dymax = -(1 << 20), dxmin = 1 << 20, dxmax = -(1 << 20);
    for (int t = 0; t < T::KK; t++) {
        dymin = std::min(dymin, T::dy(t));
        dymax = std::max(dymax, T::dy(t));
        dxmin = std::min(dxmin, T::dx(t));
        dxmax = std::max(dxmax, T::dx(t));
    }
    const int IS = T::IS;
    const int step = (T::KK == 1) ? IS : 1;  // 1x1: only every IS-th source row/column
    TileGeo &t = a.geo;
    t.IMGS = p.IMGS;
    t.rowstep = step;
    t.colstep = step;
    a.lrow = IS / step;
    t.TIH = (p.TR - 1) * a.lrow + (dymax - dymin) + 1;
    t.TIW = (GB - 1) * (IS / step) + (dxmax - dxmin) + 1;
    t.deint = (IS / step) == 2;
    t.HALF = (t.TIW + 1) / 2;
    t.TIWP = t.deint ? 2 * t.HALF : t.TIW;
    a.lcol = t.deint ? 1 : IS / step;
    t.imgs = t.TIH * t.TIWP;
    t.chs = 0;
    tilegeo_finish(t);
    a.plane = (p.IMGS * t.imgs + 63) / 64 * 64;
    a.ppw = a.plane / 64;
    if (a.ppw > (K == 3 ? SPLIT_U * FAST_NW : WIN_ROWS) || t.TIH > 254 || p.IMGS > 255)
        return 0;
    a.dymin = dymin;
    a.dxmin = dxmin;
    a.m_imgs = t.fd_imgstr.m;
    a.m_tiwp = t.fd_tiwp.m;
    if constexpr (K == 3) {
        constexpr ConvPairs<S, P, DX> cp;
        for (int i = 0; i < 10; i++) {
            const int tap = cp.t[i] >= 0 ? cp.t[i] : cp.t[i & ~1];
            const int dyp = T::dy(tap) - dymin, dxp = T::dx(tap) - dxmin;
            a.ptap[i] = cp.t[i];
            a.poff[i] = dyp * t.TIWP + (t.deint ? (dxp & 1) * t.HALF + (dxp >> 1) : dxp);
        }
        a.xwords = 12 * a.plane;
        a.stage = a.xwords + p.WM * p.MB * 5 * 3 * 256;
    } else {
        a.xwords = p.CH * a.plane;
        a.stage = a.xwords + p.WM * p.MB * p.CH * T::KK * 32;
    }
    return (size_t)2 * a.stage * 4;
}

template <int K, int S, int P, bool DX>
static bool plan_ok(FastPlan &p, int CS, int GA, int GB, FastArgs &a) {
    using T = ConvTaps<K, S, P, DX>;
    const int CSe = std::max(8, (CS + 7) & ~7);
    p.CH = K == 3 ? 8 : std::min(p.CH, std::min(32, CSe));
    p.TR = std::min(p.TR, GA);
    if (p.TR <= 0 || p.IMGS <= 0 || p.CH < 8 || p.CH % 8) return false;
    if (p.WM <= 0) p.WM = 1;
    const int nwm = p.NPW * 100 + p.MB * 10 + p.WM;
    const bool shape_ok = nwm == 111 || (nwm == 211 && T::NCLS == 1 && !(K == 3 && T::IS == 2)) ||
                          ((nwm == 112 || nwm == 212) && K == 3 && T::IS == 2);
    if (!shape_ok || p.IMGS * p.TR * GB > (FAST_NW / p.WM) * p.NPW * 32) return false;
    p.lds = plan_geometry<K, S, P, DX>(p, GB, a);
    return p.lds > 0 && p.lds <= 160 * 1024;
}

// Tile choice.  RNN_CONV_PLAN="TR,IMGS,CH,NPW,MB[,WM[,WPC]]" overrides
// (tuning sweeps).  Otherwise rules fitted to measured sweeps on MI355X:
// chunks of 8 channels (3x3) or 32 (1x1); stride-1 3x3 takes 256 positions in
// two 32-position groups per wave where that leaves two items a CU (32 -> 32
// @32x32, 512 items: 23.4 us), else 128 positions (64 -> 64 @16x16, 256 or 512
// items: 23.5 / 20.3; 48 -> 80 @23x29, 37 images: 25.2 / 21.2; one 32x32 image
// 13.9 / 9.5), but always 256 for a row of more than 128, which fits no other
// tile (one 160x160 image 32 -> 32: 16.2 us, 57.1 on the generic kernel); 1x1
// forward takes 256 positions when an image has as many;
// strided 3x3 forward splits the waves two ways along output channels, so that
// every wave has a 32x32 block at 64 positions, two at 128 where that leaves a
// CU one item (us, fp32 pipe / 64 / 128: 32 -> 64 @32x32, 256 items, 18.9 / 22.1
// / 19.9; 48 -> 96 @32x32 47.2 / 49.2 / 40.0; 128 -> 256 @16x16 60.0 / 61.9 /
// 48.8; 64 -> 128 @16x16, 128 items, 18.6 / 20.7 / 28.3); 32 positions where 64
// leave half of the CUs without one (32 images 32 -> 64 @32x32 11.8 / 13.5 /
// 11.1 at 32, one image 11.4 / 12.9 / 10.4).  A plan that does not fit falls
// back to shrinking the tile.
template <int K, int S, int P, bool DX>
static bool choose_plan(int CS, int CD, int GA, int GB, size_t n, size_t cus, FastPlan &best,
                        FastArgs &a) {
    using T = ConvTaps<K, S, P, DX>;
    if (const char *env = getenv("RNN_CONV_PLAN")) {
        FastPlan p{};
        const int got = sscanf(env, "%d,%d,%d,%d,%d,%d,%d", &p.TR, &p.IMGS, &p.CH, &p.NPW, &p.MB,
                               &p.WM, &p.wpc);
        if (got >= 5 && plan_ok<K, S, P, DX>(p, CS, GA, GB, a)) {
            best = p;
            return true;
        }
    }
    if (GB > 256) return false;
    const int ch = T::KK == 1 ? 32 : 8;
    const bool strided = T::KK == 9 && T::IS == 2;
    FastPlan r{};
    r.CH = ch;
    r.NPW = 1;
    r.MB = 1;
    r.WM = 1;
    int npos = 128;
    if (T::KK == 9 && T::NCLS == 1 && T::IS == 1) {
        const size_t tiles = n * (size_t)((GA + std::max(1, 256 / GB) - 1) / std::max(1, 256 / GB));
        if (GB > 128 || (GA * GB >= 256 && tiles * ((CD + 31) / 32) >= 2 * cus)) {
            r.NPW = 2;
            npos = 256;
        }
    } else if (strided) {
        npos = 64;
        if (CD > 32) {
            r.WM = 2;
            auto tile = [&](int np, FastPlan &q) -> size_t {  // sets it; work items
                q.TR = GA * GB <= np ? GA : std::max(1, np / GB);
                q.IMGS = GA * GB <= np ? std::max(1, np / (GA * GB)) : 1;
                return (n + q.IMGS - 1) / q.IMGS * ((GA + q.TR - 1) / q.TR) * ((CD + 63) / 64);
            };
            FastPlan q = r;
            q.NPW = 2;
            if (tile(128, q) >= cus && plan_ok<K, S, P, DX>(q, CS, GA, GB, a)) {
                best = q;
                return true;
            }
            if (2 * tile(64, q) <= cus) npos = 32;
        }
    } else if (T::KK == 1 && T::NCLS == 1 && GA * GB >= 256) {
        r.NPW = 2;
        npos = 256;
    }
    if (GA * GB <= npos) {
        r.TR = GA;
        r.IMGS = std::max(1, npos / (GA * GB));
    } else {
        r.TR = std::max(1, npos / GB);
        r.IMGS = 1;
    }
    for (;;) {
        FastPlan q = r;
        if (plan_ok<K, S, P, DX>(q, CS, GA, GB, a)) {
            best = q;
            return true;
        }
        if (r.IMGS > 1)
            r.IMGS /= 2;
        else if (r.TR > 1)
            r.TR = (r.TR + 1) / 2;
        else if (r.CH > 8)
            r.CH /= 2;
        else if (r.WM > 1)
            r.WM = 1;
        else
            return false;
    }
}

// LDS after the two stage buffers for the store-pass sums: per position wave,
// channel of the group and kind, one double.
static size_t epi_lds(const FastPlan &p) {
    return (size_t)(FAST_NW / p.WM) * 32 * p.WM * p.MB * 2 * sizeof(double);
}


// Operand roles, geometry and tile plan of a (k, stride, pad) forward / dX
// convolution; false when no plan fits.
template <int K, int S, int P, bool DX>
static bool setup(const rnn_conv_spec *sp, size_t n, size_t cus, FastArgs &a, FastPlan &p) {
    using T = ConvTaps<K, S, P, DX>;
    std::memset(&a, 0, sizeof(a));
    const int cin = sp->cin, cout = sp->cout;
    if (!DX) {
        a.CS = cin;
        a.HS = sp->h;
        a.WS = sp->w;
        a.CD = cout;
        a.HD = sp->oh;
        a.WD = sp->ow;
        a.GA = sp->oh;
        a.GB = sp->ow;
        a.sm = cin * T::KK;  // W[m = cout][ch = cin][tap]
        a.sc = T::KK;
    } else {
        a.CS = cout;
        a.HS = sp->oh;
        a.WS = sp->ow;
        a.CD = cin;
        a.HD = sp->h;
        a.WD = sp->w;
        a.GA = (sp->h + S - 1) / S;
        a.GB = (sp->w + S - 1) / S;
        a.sm = T::KK;  // W^T: m = cin, ch = cout
        a.sc = cin * T::KK;
    }
    if (!choose_plan<K, S, P, DX>(a.CS, a.CD, a.GA, a.GB, n, cus, p, a)) return false;
    if (getenv("RNN_CONV_DEBUG"))
        fprintf(stderr, "conv k%d s%d p%d %s %dx%d->%d: plan %d,%d,%d,%d,%d,%d lds %zu\n", K, S, P,
                DX ? "dx" : "fwd", a.CS, a.GA, a.CD, p.TR, p.IMGS, p.CH, p.NPW, p.MB, p.WM, p.lds);
    a.TR = p.TR;
    a.tiles_a = (a.GA + p.TR - 1) / p.TR;
    a.CH = p.CH;
    a.nchunks = (a.CS + p.CH - 1) / p.CH;
    return true;
}

template <int K, int S, int P, bool DX>
static PackGeo pack_geo(const FastArgs &a) {
    PackGeo pg;
    pg.CS = a.CS;
    pg.CD = a.CD;
    pg.KK = ConvTaps<K, S, P, DX>::KK;
    pg.CH = a.CH;
    pg.nchunks = a.nchunks;
    pg.nmblk = (a.CD + 31) / 32;
    pg.sm = a.sm;
    pg.sc = a.sc;
    pg.ptap = 0;
    for (int i = 0; i < 10; i++) pg.ptap |= (uint64_t)(a.ptap[i] & 15) << 4 * i;
    return pg;
}

// A kernel as a type, so that launch's static state is one of its own.
template <void (*F)(FastArgs)>
using Kern = std::integral_constant<void (*)(FastArgs), F>;

template <int K, int S, int P, bool DX>
static int launch(rnn_ctx *ctx, const rnn_conv_spec *sp, int n, const float *src, const float *w,
                  const float *wp, float *dst, const ConvStats *cs) {
    using T = ConvTaps<K, S, P, DX>;
    FastArgs a;
    FastPlan p;
    if (!setup<K, S, P, DX>(sp, (size_t)n, (size_t)ctx->num_cus, a, p))
        return RNN_E_UNSUPPORTED;  // no LDS tiling for the grid
    a.src = src;
    a.w = w;
    a.dst = dst;
    a.N = n;
    const long long wbytes = (long long)sp->cout * sp->cin * T::KK * 4;
    const long long pbytes = (long long)pack_geo<K, S, P, DX>(a).floats() * 4;
    if ((long long)p.IMGS * a.CS * a.HS * a.WS * 4 >= 0x7FFFFFF0ll || wbytes >= 0x7FFFFFF0ll ||
        pbytes >= 0x7FFFFFF0ll)
        return RNN_E_UNSUPPORTED;  // tile source or weights beyond 2 GiB
    a.wbytes = (int)wbytes;
    a.wp = wp;
    a.wpbytes = (int)pbytes;
    const int nmblk = (a.CD + 31) / 32;
    a.ntiles = a.tiles_a * ((n + p.IMGS - 1) / p.IMGS);
    a.ngroups = (nmblk + p.MB * p.WM - 1) / (p.MB * p.WM);
    const long long nitems = (long long)a.ntiles * a.ngroups;
    if (nitems > 0x7fffffffll) return RNN_E_UNSUPPORTED;
    const bool stats = cs != nullptr;
    if (stats) {
        if (DX || !cs->part)
            return rnn_fail(ctx, RNN_E_INVALID, "conv: store-pass statistics need a forward");
        a.stats = *cs;
        a.npart = a.ntiles;
        p.lds += epi_lds(p);
        if (p.lds > 160 * 1024) return RNN_E_UNSUPPORTED;  // no LDS for the store-pass sums
    }
    // Persistent grid: as many workgroups as fit on the chip at once.
    auto run = [&](auto kc) -> int {
        constexpr auto kern = decltype(kc)::value;
        // once an instance, not a host call a launch
        static const hipError_t attr = hipFuncSetAttribute(
            (const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        (void)attr;
        int occ = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kern, 64 * FAST_NW * 2, p.lds) !=
                hipSuccess ||
            occ < 1)
            occ = 1;
        if (p.wpc > 0) occ = std::min(occ, p.wpc);
        const long long grid = std::min<long long>(nitems, (long long)ctx->num_cus * occ);
        hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(64 * FAST_NW * 2), p.lds, ctx->stream,
                           a);
        RNN_LAUNCHED(ctx);
        return RNN_OK;
    };
    auto pick = [&](auto ec) -> int {
        constexpr int E = decltype(ec)::value;
        if constexpr (K == 3) {
            auto split = [&](auto nc, auto mc) -> int {  // groups per wave, blocks of channels
                constexpr int N = decltype(nc)::value, M = decltype(mc)::value;
                const int u = (a.ppw + FAST_NW - 1) / FAST_NW;
                if (wp)
                    return u == 1   ? run(Kern<conv_fast_kernel<K, S, P, DX, N, 1, M, E, 1, true>>{})
                           : u == 2 ? run(Kern<conv_fast_kernel<K, S, P, DX, N, 1, M, E, 2, true>>{})
                                    : run(Kern<conv_fast_kernel<K, S, P, DX, N, 1, M, E, 3, true>>{});
                return u == 1   ? run(Kern<conv_fast_kernel<K, S, P, DX, N, 1, M, E, 1, false>>{})
                       : u == 2 ? run(Kern<conv_fast_kernel<K, S, P, DX, N, 1, M, E, 2, false>>{})
                                : run(Kern<conv_fast_kernel<K, S, P, DX, N, 1, M, E, 3, false>>{});
            };
            using one = std::integral_constant<int, 1>;
            using two = std::integral_constant<int, 2>;
            if constexpr (T::IS == 2) {
                if (p.WM == 2) return p.NPW == 2 ? split(two{}, two{}) : split(one{}, two{});
            } else if constexpr (T::NCLS == 1) {
                if (p.NPW == 2) return split(two{}, one{});
            }
            return split(one{}, one{});
        } else {
            if constexpr (T::NCLS == 1)
                if (p.NPW == 2) return run(Kern<conv_fast_kernel<K, S, P, DX, 2, 1, 1, E, 1, false>>{});
            return run(Kern<conv_fast_kernel<K, S, P, DX, 1, 1, 1, E, 1, false>>{});
        }
    };
    if constexpr (!DX)
        if (stats) return pick(std::integral_constant<int, 1>{});
    return pick(std::integral_constant<int, 0>{});
}

template <int K, int S, int P>
static int parts_of(const rnn_ctx *ctx, const rnn_conv_spec *sp, size_t n) {
    FastArgs a;
    FastPlan p;
    if (!setup<K, S, P, false>(sp, n, (size_t)ctx->num_cus, a, p)) return -1;
    if (p.lds + epi_lds(p) > 160 * 1024) return -1;
    const long long np = (long long)a.tiles_a * (((long long)n + p.IMGS - 1) / p.IMGS);
    return np > 0x3fffffffll ? -1 : (int)np;
}


// Packs W for the forward (dx = 0) or dX (dx = 1) kernel in the order in which
// the kernel stages it (PackGeo: 1x1 [m-block][chunk][quad][lane][4], 3x3
// [m-block][chunk][tap pair][lane][8]), zero-filled beyond the channels, so that
// a stage's weights are one contiguous read.
__global__ __launch_bounds__(256) void conv_pack_kernel(const float *__restrict__ w, PackGeo g,
                                                        float *wp) {
    for (int r = blockIdx.x; r < g.slabs(); r += gridDim.x)
        wp[(size_t)r * 256 + threadIdx.x] = g.value(w, r, threadIdx.x);
}

// Several packs in one launch: block b serves the segment whose block range
// holds it, one 256-float slab at a time.
__global__ __launch_bounds__(256) void conv_pack_multi_kernel(const float *__restrict__ src,
                                                              const PackSeg *__restrict__ segs,
                                                              int nseg, float *dst) {
    int lo = 0, hi = nseg - 1;
    while (lo < hi) {  // last segment with blk0 <= blockIdx.x
        const int mid = (lo + hi + 1) >> 1;
        if (segs[mid].blk0 <= blockIdx.x)
            lo = mid;
        else
            hi = mid - 1;
    }
    const PackSeg sg = segs[lo];
    const float *w = src + sg.src;
    float *wp = dst + sg.dst;
    for (int r = blockIdx.x - sg.blk0; r < sg.geo.slabs(); r += sg.nblk)
        wp[(size_t)r * 256 + threadIdx.x] = sg.geo.value(w, r, threadIdx.x);
}

template <int K, int S, int P, bool DX>
static int geo_of(const rnn_conv_spec *sp, PackGeo *pg) {
    FastArgs a;
    FastPlan p;
    // (the packed layout does not depend on the batch: 3x3 plans share CH)
    if (!setup<K, S, P, DX>(sp, 1, 1, a, p)) return RNN_E_UNSUPPORTED;
    *pg = pack_geo<K, S, P, DX>(a);
    return RNN_OK;
}

}  // namespace

// Forward (dx = 0) or dX (dx = 1) through the specialised kernels; returns
// RNN_E_UNSUPPORTED (without recording an error) when (k, stride, pad) has no
// specialisation or the shape no tile, so the caller can take the generic
// per-class path.  wp:
// the weights packed by rnn_conv_pack for this direction, or null.
int rnn_conv_fast(rnn_ctx *ctx, int dx, const rnn_conv_spec *sp, size_t n, const float *src,
                  const float *w, const float *wp, float *dst, const ConvStats *stats) {
    if (getenv("RNN_CONV_GENERIC")) return RNN_E_UNSUPPORTED;
    const int k = sp->k, s = sp->stride, p = sp->pad;
    const int ni = (int)n;
#define RNN_CONV_CASE(K_, S_, P_)                                                               \
    if (k == K_ && s == S_ && p == P_)                                                          \
        return dx ? launch<K_, S_, P_, true>(ctx, sp, ni, src, w, wp, dst, stats)               \
                  : launch<K_, S_, P_, false>(ctx, sp, ni, src, w, wp, dst, stats);
    RNN_CONV_CASE(3, 1, 1)
    RNN_CONV_CASE(3, 2, 1)
    RNN_CONV_CASE(1, 2, 0)
    RNN_CONV_CASE(1, 1, 0)
#undef RNN_CONV_CASE
    return RNN_E_UNSUPPORTED;
}

int rnn_conv_fast_parts(const rnn_ctx *ctx, const rnn_conv_spec *sp, size_t n) {
    if (getenv("RNN_CONV_GENERIC") || n == 0 || n > 0x7fffffff) return -1;
    const int k = sp->k, s = sp->stride, p = sp->pad;
#define RNN_CONV_CASE(K_, S_, P_) \
    if (k == K_ && s == S_ && p == P_) return parts_of<K_, S_, P_>(ctx, sp, n);
    RNN_CONV_CASE(3, 1, 1)
    RNN_CONV_CASE(3, 2, 1)
    RNN_CONV_CASE(1, 2, 0)
    RNN_CONV_CASE(1, 1, 0)
#undef RNN_CONV_CASE
    return -1;
}

template <int K, int S, int P, bool DX>
static int plan_of(const rnn_conv_spec *sp, size_t n, size_t cus, int *plan) {
    FastArgs a;
    FastPlan p;
    if (!setup<K, S, P, DX>(sp, n, cus, a, p)) return RNN_E_UNSUPPORTED;
    const int v[6] = {p.TR, p.IMGS, p.CH, p.NPW, p.WM, a.plane};
    std::copy(v, v + 6, plan);
    return RNN_OK;
}

extern "C" int rnn_dbg_conv_plan(const rnn_conv_spec *sp, int dx, size_t n, size_t cus, int *plan) {
    if (!sp || !plan) return RNN_E_NULL;
    const int k = sp->k, s = sp->stride, p = sp->pad;
#define RNN_CONV_CASE(K_, S_, P_)                                        \
    if (k == K_ && s == S_ && p == P_)                                   \
        return dx ? plan_of<K_, S_, P_, true>(sp, n, cus, plan)          \
                  : plan_of<K_, S_, P_, false>(sp, n, cus, plan);
    RNN_CONV_CASE(3, 1, 1)
    RNN_CONV_CASE(3, 2, 1)
    RNN_CONV_CASE(1, 2, 0)
    RNN_CONV_CASE(1, 1, 0)
#undef RNN_CONV_CASE
    return RNN_E_UNSUPPORTED;
}

int rnn_conv_pack_geo(const rnn_conv_spec *sp, int dx, PackGeo *pg) {
    if (getenv("RNN_CONV_GENERIC")) return RNN_E_UNSUPPORTED;
    const int k = sp->k, s = sp->stride, p = sp->pad;
#define RNN_CONV_CASE(K_, S_, P_)                                                               \
    if (k == K_ && s == S_ && p == P_)                                                          \
        return dx ? geo_of<K_, S_, P_, true>(sp, pg) : geo_of<K_, S_, P_, false>(sp, pg);
    RNN_CONV_CASE(3, 1, 1)
    RNN_CONV_CASE(3, 2, 1)
    RNN_CONV_CASE(1, 2, 0)
    RNN_CONV_CASE(1, 1, 0)
#undef RNN_CONV_CASE
    return RNN_E_UNSUPPORTED;
}

int rnn_conv_pack(rnn_ctx *ctx, const rnn_conv_spec *sp, int dx, const float *w, float *wp) {
    PackGeo pg;
    const int rc = rnn_conv_pack_geo(sp, dx, &pg);
    if (rc) return rc;
    const unsigned grid = (unsigned)std::min(pg.slabs(), 4096);
    conv_pack_kernel<<<grid, 256, 0, ctx->stream>>>(w, pg, wp);
    RNN_LAUNCHED(ctx);
    return RNN_OK;
}

int rnn_conv_pack_multi_launch(rnn_ctx *ctx, const PackSeg *segs, int nseg, int nblocks,
                               const float *src, float *dst) {
    if (nseg <= 0) return RNN_OK;
    conv_pack_multi_kernel<<<nblocks, 256, 0, ctx->stream>>>(src, segs, nseg, dst);
    RNN_LAUNCHED(ctx);
    return RNN_OK;
}

// Packed copies of several convolutions' weights in one device block: the
// data (each copy a whole number of 256-float slabs), then the segment table
// that conv_pack_multi_kernel walks.  Sources are addressed from the lowest
// W pointer, so a segment's source offset is its W's distance from it.
struct rnn_conv_packs {
    void *mem = nullptr;
    PackSeg *segs = nullptr;
    int nseg = 0, nblk = 0;
    const float *src = nullptr;
    float *data = nullptr;
    std::vector<const float *> wp[2];
};

int rnn_conv_packs_create(rnn_ctx *ctx, size_t count, const rnn_conv_spec *specs, const float **w,
                          rnn_conv_packs **out) {
    if (!ctx || !out) return RNN_E_NULL;
    *out = nullptr;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    if (count == 0 || !specs || !w) return rnn_fail(ctx, RNN_E_NULL, "conv_packs: no convolutions");
    uintptr_t lo = UINTPTR_MAX;
    for (size_t i = 0; i < count; i++) {
        if (!w[i]) return rnn_fail(ctx, RNN_E_NULL, "conv_packs: null weights %zu", i);
        if ((uintptr_t)w[i] & 3) return rnn_fail(ctx, RNN_E_INVALID, "conv_packs: unaligned W");
        lo = std::min(lo, (uintptr_t)w[i]);
    }
    std::vector<PackSeg> segs;
    std::vector<std::pair<size_t, int>> who;  // (conv, direction) of each segment
    size_t floats = 0;
    uint32_t blk = 0;
    for (size_t i = 0; i < count; i++) {
        for (int dx = 0; dx < 2; dx++) {
            PackSeg sg;
            if (rnn_conv_pack_geo(&specs[i], dx, &sg.geo) != RNN_OK) continue;
            sg.src = ((uintptr_t)w[i] - lo) / sizeof(float);
            sg.dst = floats;
            sg.blk0 = blk;
            sg.nblk = (uint32_t)std::min(sg.geo.slabs(), 512);
            blk += sg.nblk;
            floats += sg.geo.floats();
            segs.push_back(sg);
            who.push_back({i, dx});
        }
    }
    if (blk > 0x7fffffffu) return rnn_fail(ctx, RNN_E_UNSUPPORTED, "conv_packs: too many slabs");
    auto *p = new (std::nothrow) rnn_conv_packs();
    if (!p) return rnn_fail(ctx, RNN_E_NOMEM, "conv_packs: host allocation");
    p->wp[0].assign(count, nullptr);
    p->wp[1].assign(count, nullptr);
    p->src = (const float *)lo;
    p->nseg = (int)segs.size();
    p->nblk = (int)blk;
    if (!segs.empty()) {
        const size_t dbytes = floats * sizeof(float), tbytes = segs.size() * sizeof(PackSeg);
        hipError_t e = hipMalloc(&p->mem, dbytes + tbytes);
        if (e != hipSuccess) {
            delete p;
            return rnn_fail(ctx, RNN_E_NOMEM, "conv_packs hipMalloc(%zu): %s", dbytes + tbytes,
                            hipGetErrorString(e));
        }
        p->data = (float *)p->mem;
        p->segs = (PackSeg *)((char *)p->mem + dbytes);
        e = hipMemcpy(p->segs, segs.data(), tbytes, hipMemcpyHostToDevice);
        if (e != hipSuccess) {
            (void)hipFree(p->mem);
            delete p;
            return rnn_fail(ctx, RNN_E_HIP, "conv_packs table upload: %s", hipGetErrorString(e));
        }
        for (size_t k = 0; k < segs.size(); k++)
            p->wp[who[k].second][who[k].first] = p->data + segs[k].dst;
    }
    const int rc = rnn_conv_pack_multi_launch(ctx, p->segs, p->nseg, p->nblk, p->src, p->data);
    if (rc) {
        rnn_conv_packs_destroy(p);
        return rc;
    }
    *out = p;
    return RNN_OK;
}

int rnn_conv_packs_update(rnn_ctx *ctx, rnn_conv_packs *p) {
    if (!ctx || !p) return RNN_E_NULL;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    return rnn_conv_pack_multi_launch(ctx, p->segs, p->nseg, p->nblk, p->src, p->data);
}

const float *rnn_conv_packs_get(const rnn_conv_packs *p, size_t i, int dx) {
    if (!p || (dx != 0 && dx != 1) || i >= p->wp[0].size()) return nullptr;
    return p->wp[dx][i];
}

void rnn_conv_packs_destroy(rnn_conv_packs *p) {
    if (!p) return;
    if (p->mem) (void)hipFree(p->mem);
    delete p;
}
