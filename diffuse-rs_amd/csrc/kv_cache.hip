// kv_cache.hip -- the inter-step KV cache in HBM (StepCache,
// src/model/cache.rs:25-115), bf16, position-indexed.
//
// Layout per (layer, batch slot), for n_head_kv heads and capacity `cap`
// positions (a multiple of 64), HD = the head-dim tile (64/128/256/512):
//   K  : [n_head_kv][cap][HD]              row = sequence position
//   V^T: [n_head_kv][cap/32][HD][32]       V transposed per 32-key tile: a
//                                          tile's d-row holds its 32 positions
// The attention kernel stages both as 16-byte loads; V^T is exactly the
// operand orientation the P.V MFMA needs, so the transpose is paid once per
// stored row instead of once per attention tile, and a key tile of either is
// one contiguous block (whole cache lines for the DMA).
//
// store:  StepCache::store (cache.rs:62-71) -- f32 rows -> bf16 at their
//         positions, optionally after per-head RMSNorm of K (norm_heads,
//         ops.rs:384-389, applied before the store in forward.rs:300-302).
//         A layer kept at hi/lo precision also gets the lo halves,
//         bf16(x - bf16(x)), of K and V in planes laid out like K and V^T.
//         One launch of one of three kernels (pick_store): one workgroup
//         per (kv head, 32 rows, K or V) or per (kv head, whole 32-key tile),
//         whole-line loads; or one per (64-row block, 64-wide head-dim chunk,
//         kv head), K converted in registers, V transposed through LDS, which
//         takes padded head dims and unaligned rows too.
// gather: StepCache::gather (cache.rs:73-82) -- bf16 back to f32 rows (hi +
//         lo where the layer keeps the lo halves).
#include <algorithm>

#include "dr_internal.hpp"

#include <math.h>

namespace dr {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint16_t f2bf(float x) {
    return __builtin_bit_cast(uint16_t, static_cast<__bf16>(x));
}
__device__ __forceinline__ float bf2f(uint16_t h) {
    return __uint_as_float(static_cast<uint32_t>(h) << 16);
}

// RoPE's rotation of one pair (ops.rs:447-448), without fused multiply-adds
// as Rust evaluates it.
__device__ __forceinline__ float rope_lo(float a, float b, float sn, float cs) {
#pragma clang fp contract(off)
    return a * cs - b * sn;
}
__device__ __forceinline__ float rope_hi(float a, float b, float sn, float cs) {
#pragma clang fp contract(off)
    return a * sn + b * cs;
}

constexpr int SR = 64;   // rows per store workgroup: one 128-byte line of a V^T row
constexpr int SD = 64;   // head-dim entries per store workgroup: one 128-byte line of a K row
constexpr int SPT = 16;  // consecutive values per thread (4 threads per row, 256 threads)

// One workgroup per (64-row block, 64-wide head-dim chunk, kv head), so that
// every 128-byte line of K and of V^T it writes is written whole by it.  All
// loads of the block (16 K and 16 V floats per thread) are issued before any
// store.  K: optional per-head RMSNorm, whose sum of squares covers the whole
// row (the other chunks' values are loaded for it), then bf16 at the row's
// position.  V: bf16 into an LDS tile transposed to [d][row]; each thread then
// writes 16 positions of one d-row of V^T (16-byte stores when the positions
// are contiguous and aligned).
template <int HD>
__global__ __launch_bounds__(256) void kv_store_kernel(const StoreArgs a) {
    constexpr int NDC = HD / SD;
    constexpr int V4 = SPT / 4;
    __shared__ __align__(16) uint16_t tile[SD][SR + 8];
    __shared__ __align__(16) uint16_t tile_lo[SD][SR + 8];  // V's lo half, when kept

    // Workgroup -> (kv head g, chunk dc, row block).  The hardware deals
    // workgroups round-robin over the 8 XCDs (XCD = blockIdx & 7); each XCD in
    // [xcd_lo, xcd_lo + xcd_n) takes a contiguous run of per_xcd logical ids,
    // so kv head g is written through the L2 of the XCD on which the attention
    // launch reads it (it deals heads to XCDs in the same contiguous way).
    const int x = blockIdx.x & 7;
    if (x < a.xcd_lo || x >= a.xcd_lo + a.xcd_n) return;
    const int lid = (x - a.xcd_lo) * a.per_xcd + (int)(blockIdx.x >> 3);
    if (lid >= a.n_head_kv * NDC * a.n_rb) return;
    const int hc = lid / a.n_rb;
    const int g = hc / NDC, dc = hc - g * NDC;
    const int r0 = (lid - hc * a.n_rb) * SR;
    const int tid = threadIdx.x, rl = tid >> 2, part = tid & 3;
    const int r = r0 + rl;
    const bool ok = r < a.n;
    const int d0 = dc * SD + part * SPT;  // first head-dim entry of this thread
    const size_t row = (size_t)(ok ? r : 0) * a.rstride + (size_t)g * a.hd;
    f32x4 xk[V4], xv[V4];
    if (ok && a.vec) {
#pragma unroll
        for (int i = 0; i < V4; ++i) {
            xk[i] = *reinterpret_cast<const f32x4*>(a.k + row + d0 + 4 * i);
            xv[i] = *reinterpret_cast<const f32x4*>(a.v + row + d0 + 4 * i);
        }
    } else {
#pragma unroll
        for (int i = 0; i < V4; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int d = d0 + 4 * i + e;
                const bool in = ok && d < a.hd;
                xk[i][e] = in ? a.k[row + d] : 0.0f;
                xv[i][e] = in ? a.v[row + d] : 0.0f;
            }
    }
    // The K-norm gains of this thread's dims and, with RoPE, of their
    // partners (d +- rot/2), requested with the rows: read where they are
    // used, after the row's norm, they cost a dependent round trip.
    f32x4 kw[V4], kwp[V4];
    if (a.kn_w) {
        const int hr = a.rot / 2;
#pragma unroll
        for (int i = 0; i < V4; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int d = d0 + 4 * i + e;
                kw[i][e] = d < a.hd ? a.kn_w[d] : 0.0f;
                kwp[i][e] = (a.rope && d < a.rot) ? a.kn_w[d < hr ? d + hr : d - hr] : 0.0f;
            }
    }
    const int pos = ok ? (a.pos0 >= 0 ? a.pos0 + r : (a.pos ? a.pos[r] : r)) : 0;
    // RoPE's (sin, cos) pairs of this thread's 16 dims, requested with the
    // rows: when rot/2 is a multiple of 16 they lie on one side of it, 32
    // contiguous floats of the position's table row
    const int rhalf = a.rot / 2;
    const bool tab_vec = a.rope && rhalf % SPT == 0 && d0 < a.rot;
    f32x4 tv[SPT / 2];
    if (tab_vec && ok) {
        const int j0 = d0 < rhalf ? d0 : d0 - rhalf;
        const f32x4* t = reinterpret_cast<const f32x4*>(a.rope + ((size_t)pos * rhalf + j0) * 2);
#pragma unroll
        for (int i = 0; i < SPT / 2; ++i) tv[i] = t[i];
    }

    // The Q/K/V epilogue's K and V part (forward.rs:291-310), when asked:
    // add_bias (ops.rs:373-382), then K's RMSNorm with the gain / V's
    // without one (Gemma, ops.rs:116-124), then RoPE on K (ops.rs:433-452).
    const float* kb = a.kb ? a.kb + (size_t)g * a.hd : nullptr;
    const float* vb = a.vb ? a.vb + (size_t)g * a.hd : nullptr;
    if (kb || vb) {
#pragma unroll
        for (int i = 0; i < V4; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int d = d0 + 4 * i + e;
                if (d < a.hd) {
                    if (kb) xk[i][e] += kb[d];
                    if (vb) xv[i][e] += vb[d];
                }
            }
    }
    // The row's other 64-wide chunks at this thread's 16 entries (bias
    // added), read once: the norms sum over the whole row, and with RoPE a
    // dim's partner (d +- rot/2) lies in one of them when rot/2 is a multiple
    // of 64.
    const bool need_ko = a.kn_w || a.rope;
    f32x4 ko[NDC][V4], vo[NDC][V4];
    auto load_other = [&](f32x4 (&xo)[NDC][V4], const float* src, const float* bias)
        __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < NDC; ++c) {
            if (c == dc) continue;
            const int e0 = c * SD + part * SPT;
            if (ok && a.vec) {
#pragma unroll
                for (int i = 0; i < V4; ++i) {
                    xo[c][i] = *reinterpret_cast<const f32x4*>(src + row + e0 + 4 * i);
                    if (bias) xo[c][i] += *reinterpret_cast<const f32x4*>(bias + e0 + 4 * i);
                }
            } else {
#pragma unroll
                for (int i = 0; i < V4; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int d = e0 + 4 * i + e;
                        float v = (ok && d < a.hd) ? src[row + d] : 0.0f;
                        if (bias && d < a.hd) v += bias[d];
                        xo[c][i][e] = v;
                    }
            }
        }
    };
    if (need_ko) load_other(ko, a.k, kb);
    if (a.v_norm) load_other(vo, a.v, vb);
    // rms_norm_inplace (ops.rs:106-114) / rms_norm_noscale: f32 squares
    // summed in f64 over the whole row
    auto row_scale = [&](const f32x4 (&x)[V4], const f32x4 (&xo)[NDC][V4], float eps)
        __attribute__((always_inline)) {
        double ss = 0.0;
#pragma unroll
        for (int c = 0; c < NDC; ++c)
#pragma unroll
            for (int i = 0; i < V4; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float xv = c == dc ? x[i][e] : xo[c][i][e];
                    const float sq = xv * xv;
                    ss += (double)sq;
                }
        ss += __shfl_xor(ss, 1);
        ss += __shfl_xor(ss, 2);
        return 1.0f / (float)sqrt(ss / (double)a.hd + (double)eps);
    };
    float ksc = 1.0f;
    if (a.kn_w) {
        ksc = row_scale(xk, ko, a.kn_eps);
#pragma unroll
        for (int i = 0; i < V4; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int d = d0 + 4 * i + e;
                if (d < a.hd) xk[i][e] = xk[i][e] * ksc * kw[i][e];
            }
    }
    if (a.v_norm) {
        const float vsc = row_scale(xv, vo, a.kn_eps);
#pragma unroll
        for (int i = 0; i < V4; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) xv[i][e] *= vsc;
    }
    if (a.rope && ok) {
        // the partner's value with the same bias and norm, then the pair
        // rotates (rotate_rows, ops.rs:433-452)
        const int half = a.rot / 2;
        const float* tab = a.rope + (size_t)pos * half * 2;
        const bool chunked = half % SD == 0;  // partner = same entry of chunk dc +- half/SD
        // (the thread's 16 dims lie on one side of half, so one chunk)
        const int pc = chunked ? (d0 < half ? dc + half / SD : dc - half / SD) : 0;
        f32x4 yk[V4];
#pragma unroll
        for (int i = 0; i < V4; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int d = d0 + 4 * i + e;
                yk[i][e] = xk[i][e];
                if (d >= a.rot) continue;
                const int pd = d < half ? d + half : d - half;
                float xp;
                if (chunked) {
                    xp = 0.0f;
#pragma unroll
                    for (int c = 0; c < NDC; ++c)
                        if (c == pc) xp = ko[c][i][e];  // pc != dc
                } else {
                    xp = a.k[row + pd];
                    if (kb) xp += kb[pd];
                }
                if (a.kn_w) xp = xp * ksc * kwp[i][e];
                const int j = d < half ? d : pd;
                float2 t;
                if (tab_vec) {
                    const int k4 = 4 * i + e;  // pair k4 of the 16: floats 2*k4, 2*k4+1
                    t = make_float2(tv[k4 / 2][2 * (k4 % 2)], tv[k4 / 2][2 * (k4 % 2) + 1]);
                } else {
                    t = *reinterpret_cast<const float2*>(tab + 2 * j);
                }
                yk[i][e] = d < half ? rope_lo(xk[i][e], xp, t.x, t.y) : rope_hi(xp, xk[i][e], t.x, t.y);
            }
#pragma unroll
        for (int i = 0; i < V4; ++i) xk[i] = yk[i];
    }
    if (ok) {
        uint16_t* dst = a.kc + ((size_t)g * a.cap + pos) * HD + d0;
#pragma unroll
        for (int i = 0; i < V4; i += 2) {
            u32x4 w;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                w[2 * j] = (uint32_t)f2bf(xk[i + j][0]) | ((uint32_t)f2bf(xk[i + j][1]) << 16);
                w[2 * j + 1] = (uint32_t)f2bf(xk[i + j][2]) | ((uint32_t)f2bf(xk[i + j][3]) << 16);
            }
            *reinterpret_cast<u32x4*>(dst + 4 * i) = w;
        }
        if (a.klo) {
            // the lo half: bf16 of what bf16 rounding dropped
            uint16_t* dlo = a.klo + ((size_t)g * a.cap + pos) * HD + d0;
#pragma unroll
            for (int i = 0; i < V4; i += 2) {
                u32x4 w;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    uint16_t lo[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) lo[e] = f2bf(xk[i + j][e] - bf2f(f2bf(xk[i + j][e])));
                    w[2 * j] = (uint32_t)lo[0] | ((uint32_t)lo[1] << 16);
                    w[2 * j + 1] = (uint32_t)lo[2] | ((uint32_t)lo[3] << 16);
                }
                *reinterpret_cast<u32x4*>(dlo + 4 * i) = w;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < V4; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) tile[part * SPT + 4 * i + e][rl] = f2bf(xv[i][e]);
    if (a.vlo) {
#pragma unroll
        for (int i = 0; i < V4; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                tile_lo[part * SPT + 4 * i + e][rl] = f2bf(xv[i][e] - bf2f(f2bf(xv[i][e])));
    }
    // (a pass without pos0: the position of row tid % 64 of the block, for
    // the V^T stores below, requested before the barrier)
    const bool known = a.pos0 >= 0 || a.pos == nullptr;
    const int my_row = r0 + (tid & 63);
    const int my_pos = (!known && my_row < a.n) ? a.pos[my_row] : 0;
    __syncthreads();

    if (!known) {
        // Positions from a list: the 64 lanes of a wave take the block's 64
        // rows of one d-row, so each store instruction's 2-byte writes fall
        // into the few 32-key tiles that the sorted positions span and merge
        // into a few segment writes.  (Lanes over 16 d-rows x 4 row groups
        // made 64 separate writes per instruction: 12.9 against 4.1 us for
        // C2's 256 rows.)
        if (my_row >= a.n) return;
        const size_t pofs = (size_t)(my_pos / VT_KEYS) * (HD * VT_KEYS) + my_pos % VT_KEYS;
        const size_t vbase = (size_t)g * HD * a.cap + (size_t)(dc * SD) * VT_KEYS + pofs;
        const int rr = tid & 63;
#pragma unroll
        for (int k = 0; k < SD / 4; ++k) {
            const int d = (tid >> 6) + 4 * k;
            a.vtc[vbase + (size_t)d * VT_KEYS] = tile[d][rr];
        }
        if (a.vlo) {
#pragma unroll
            for (int k = 0; k < SD / 4; ++k) {
                const int d = (tid >> 6) + 4 * k;
                a.vlo[vbase + (size_t)d * VT_KEYS] = tile_lo[d][rr];
            }
        }
        return;
    }

    // V^T: thread -> (d-row dl, positions p0 + [0,16)).
    const int dl = tid >> 2, p0 = (tid & 3) * SPT;
    const int rfirst = r0 + p0;
    if (rfirst >= a.n) return;
    const int cnt = min(SPT, a.n - rfirst);
    const int dv = dc * SD + dl;  // this thread's d-row
    // V^T element (g, dv, p): tile p / VT_KEYS, offset p % VT_KEYS in its d-row
    const size_t vrow = (size_t)g * HD * a.cap + (size_t)dv * VT_KEYS;
    auto vt_in = [&](uint16_t* plane, int p) __attribute__((always_inline)) {
        return plane + vrow + (size_t)(p / VT_KEYS) * (HD * VT_KEYS) + p % VT_KEYS;
    };
    auto vt_at = [&](int p) __attribute__((always_inline)) { return vt_in(a.vtc, p); };
    // (contiguous rows, pos0 >= 0: positions without a load)
    const int pbase = a.pos0 >= 0 ? a.pos0 : 0;
    const int q0 = pbase + rfirst;
    const bool contiguous = cnt == SPT && (q0 & 7) == 0;
    const uint16_t* t = &tile[dl][p0];
    if (contiguous) {
        // 8 positions from a multiple of 8 never cross a 32-key tile
#pragma unroll
        for (int h = 0; h < SPT / 8; ++h)
            *reinterpret_cast<u32x4*>(vt_at(q0 + 8 * h)) = *reinterpret_cast<const u32x4*>(t + 8 * h);
    } else {
        for (int e = 0; e < cnt; ++e) *vt_at(q0 + e) = t[e];
    }
    if (a.vlo) {
        // the same positions of the lo plane (V^T's layout)
        const uint16_t* tl = &tile_lo[dl][p0];
        if (contiguous) {
#pragma unroll
            for (int h = 0; h < SPT / 8; ++h)
                *reinterpret_cast<u32x4*>(vt_in(a.vlo, q0 + 8 * h)) = *reinterpret_cast<const u32x4*>(tl + 8 * h);
        } else {
            for (int e = 0; e < cnt; ++e) *vt_in(a.vlo, q0 + e) = tl[e];
        }
    }
}

// The store of rows that fill whole 32-key V^T tiles at contiguous positions
// (pos0 and n multiples of 32), head dim == HD (64, 128 or 256), without lo
// halves: the canvas rows of every denoise step.  One workgroup per (kv
// head, tile); thread (rg, dc), rg fastest, holds the 4 dims 4 dc .. 4 dc + 3
// of the tile's rows RPG rg .. RPG rg + RPG - 1.
// - Loads: per instruction the wave reads whole 128-byte lines (hd 128: 8
//   rows x 128 B), against 64-byte pieces at a 64-byte lane stride in
//   kv_store_kernel.
// - The K / V biases, the K norm and Gemma's V norm of the epilogue, as in
//   kv_store_kernel: a row's f32 squares summed in f64, over the 4 dims of
//   each thread, then across the lanes of the row in the wave (shuffles),
//   then across the 4 waves in wave order (LDS).  RoPE on K (rotate_rows,
//   ops.rs:433-452; rot a multiple of 8, so a thread's 4 dims lie on one side
//   of rot / 2) reads the partner dim d +- rot / 2 of the normed row from LDS
//   and the (sin, cos) pairs of the row's position, loaded with the rows.
// - K: bf16 of the 4 dims, 8 bytes per row.
// - V^T: at step e the thread writes the RPG keys of its rows in d-row
//   4 dc + e of the tile; the NRG lanes of one dc together write that
//   d-row's 64 bytes whole, so no LDS transpose and no barrier is needed.
// Same values as kv_store_kernel: bf16 (round to nearest even) of each f32.
// EPI: the epilogue (biases, norms, RoPE) is compiled in; the plain build
// keeps it out, since its conditional updates of the loaded rows made the K
// stores wait for every load.
template <int HD, bool EPI>
__global__ __launch_bounds__(256) void kv_store_tiles_kernel(const StoreArgs a) {
    constexpr int CPR = HD / 4;     // 4-dim pieces per row
    constexpr int NRG = 256 / CPR;  // row groups
    constexpr int RPG = VT_KEYS / NRG;  // rows per row group
    static_assert(NRG * RPG == VT_KEYS && RPG >= 2 && RPG <= 8, "tile geometry");

    const int x = blockIdx.x & 7;  // (XCD placement as kv_store_kernel)
    if (x < a.xcd_lo || x >= a.xcd_lo + a.xcd_n) return;
    const int lid = (x - a.xcd_lo) * a.per_xcd + (int)(blockIdx.x >> 3);
    const int ntl = a.n / VT_KEYS;
    if (lid >= a.n_head_kv * ntl) return;
    const int g = lid / ntl, tb = lid - g * ntl;
    const int tid = threadIdx.x;
    const int rg = tid % NRG, dc = tid / NRG;
    const int r0 = tb * VT_KEYS + rg * RPG;  // first row of this thread
    const size_t rstride = (size_t)a.rstride;
    const size_t src = (size_t)r0 * rstride + (size_t)g * HD + 4 * dc;
    f32x4 xk[RPG], xv[RPG];
#pragma unroll
    for (int j = 0; j < RPG; ++j) {
        xk[j] = *reinterpret_cast<const f32x4*>(a.k + src + j * rstride);
        xv[j] = *reinterpret_cast<const f32x4*>(a.v + src + j * rstride);
    }
    if constexpr (EPI) {
        const int half = a.rot / 2;
        const int d0 = 4 * dc;
        const bool rot_me = a.rope && d0 < a.rot;
        f32x4 tab[RPG][2];  // (sin, cos) of pairs jj .. jj + 3 at each row's position
        if (rot_me) {
            const int jj = d0 < half ? d0 : d0 - half;
            const int pp = (a.pos0 >= 0 ? a.pos0 : 0) + r0;
#pragma unroll
            for (int j = 0; j < RPG; ++j) {
                const float* t = a.rope + ((size_t)(pp + j) * half + jj) * 2;
                tab[j][0] = *reinterpret_cast<const f32x4*>(t);
                tab[j][1] = *reinterpret_cast<const f32x4*>(t + 4);
            }
        }
        f32x4 kw4 = {}, kb4 = {}, vb4 = {};
        if (a.kn_w) kw4 = *reinterpret_cast<const f32x4*>(a.kn_w + 4 * dc);
        if (a.kb) kb4 = *reinterpret_cast<const f32x4*>(a.kb + (size_t)g * HD + 4 * dc);
        if (a.vb) vb4 = *reinterpret_cast<const f32x4*>(a.vb + (size_t)g * HD + 4 * dc);
        // (each bias only where given: adding a zero would turn -0.0 into +0.0)
        if (a.kb) {
#pragma unroll
            for (int j = 0; j < RPG; ++j) xk[j] += kb4;
        }
        if (a.vb) {
#pragma unroll
            for (int j = 0; j < RPG; ++j) xv[j] += vb4;
        }
        if (a.kn_w || a.v_norm) {
            // rms_norm_inplace (ops.rs:106-114) / rms_norm_noscale: sum of the
            // row's f32 squares in f64; the row's lanes in this wave are lanes
            // rg + NRG i, the other CPR / (64 / NRG) - 1 shares are in the
            // other waves
            __shared__ double s_ss[2][4][VT_KEYS];  // [K, V][wave][row of the tile]
            const int wave = tid >> 6;
            auto row_ss = [&](const f32x4 (&x)[RPG], double (&ss)[RPG]) __attribute__((always_inline)) {
#pragma unroll
                for (int j = 0; j < RPG; ++j) {
                    double t = 0.0;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float sq = x[j][e] * x[j][e];
                        t += (double)sq;
                    }
#pragma unroll
                    for (int off = NRG; off < 64; off <<= 1) t += __shfl_xor(t, off);
                    ss[j] = t;
                }
            };
            double ssk[RPG], ssv[RPG];
            if (a.kn_w) row_ss(xk, ssk);
            if (a.v_norm) row_ss(xv, ssv);
            if ((tid & 63) < NRG) {
#pragma unroll
                for (int j = 0; j < RPG; ++j) {
                    if (a.kn_w) s_ss[0][wave][rg * RPG + j] = ssk[j];
                    if (a.v_norm) s_ss[1][wave][rg * RPG + j] = ssv[j];
                }
            }
            __syncthreads();
            auto scale_of = [&](int kv, int j) __attribute__((always_inline)) {
                const double t = ((s_ss[kv][0][rg * RPG + j] + s_ss[kv][1][rg * RPG + j]) + s_ss[kv][2][rg * RPG + j]) +
                                 s_ss[kv][3][rg * RPG + j];
                return 1.0f / (float)sqrt(t / (double)HD + (double)a.kn_eps);
            };
#pragma unroll
            for (int j = 0; j < RPG; ++j) {
                if (a.kn_w) {
                    const float sc = scale_of(0, j);
#pragma unroll
                    for (int e = 0; e < 4; ++e) xk[j][e] = xk[j][e] * sc * kw4[e];
                }
                if (a.v_norm) {
                    const float sc = scale_of(1, j);
#pragma unroll
                    for (int e = 0; e < 4; ++e) xv[j][e] *= sc;
                }
            }
        }
        if (a.rope) {
            __shared__ __align__(16) float s_k[VT_KEYS][HD + 4];  // the tile's normed K rows
#pragma unroll
            for (int j = 0; j < RPG; ++j) *reinterpret_cast<f32x4*>(&s_k[rg * RPG + j][d0]) = xk[j];
            __syncthreads();
            if (rot_me) {
                const int pd0 = d0 < half ? d0 + half : d0 - half;
#pragma unroll
                for (int j = 0; j < RPG; ++j) {
                    const f32x4 xp = *reinterpret_cast<const f32x4*>(&s_k[rg * RPG + j][pd0]);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float sn = tab[j][e >> 1][2 * (e & 1)], cs = tab[j][e >> 1][2 * (e & 1) + 1];
                        xk[j][e] = d0 < half ? rope_lo(xk[j][e], xp[e], sn, cs) : rope_hi(xp[e], xk[j][e], sn, cs);
                    }
                }
            }
        }
    }
    const int p0 = a.pos0 >= 0 ? a.pos0 : 0;  // (host: pos0 >= 0, or no position list)
    uint16_t* kdst = a.kc + ((size_t)g * a.cap + p0 + r0) * HD + 4 * dc;
#pragma unroll
    for (int j = 0; j < RPG; ++j) {
        uint32_t w0 = (uint32_t)f2bf(xk[j][0]) | ((uint32_t)f2bf(xk[j][1]) << 16);
        uint32_t w1 = (uint32_t)f2bf(xk[j][2]) | ((uint32_t)f2bf(xk[j][3]) << 16);
        *reinterpret_cast<uint2*>(kdst + (size_t)j * HD) = make_uint2(w0, w1);
    }
    uint16_t* vdst = a.vtc + (size_t)g * HD * a.cap + (size_t)(p0 / VT_KEYS + tb) * (HD * VT_KEYS) +
                     (size_t)(4 * dc) * VT_KEYS + rg * RPG;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        uint32_t w[RPG / 2];
#pragma unroll
        for (int j = 0; j < RPG / 2; ++j)
            w[j] = (uint32_t)f2bf(xv[2 * j][e]) | ((uint32_t)f2bf(xv[2 * j + 1][e]) << 16);
        uint16_t* row = vdst + e * VT_KEYS;
        if constexpr (RPG == 2) {
            *reinterpret_cast<uint32_t*>(row) = w[0];
        } else if constexpr (RPG == 4) {
            *reinterpret_cast<uint2*>(row) = make_uint2(w[0], w[1]);
        } else {
            *reinterpret_cast<u32x4*>(row) = u32x4{w[0], w[1], w[2], w[3]};
        }
    }
}

// The store of rows at contiguous positions or at a sorted position list, head
// dim == HD: the rows of a denoise step, the prompt, a first pass (pick_store
// tells which of them).  One workgroup per (kv head, 32-key tile that the rows
// touch, K or V); rows need not fill the first and the last tile.  K and V
// take a workgroup each, so a step's few tiles give twice the workgroups, each
// with half the loads to wait for.
// Thread (rg, dc), rg fastest, holds keys 4 rg .. 4 rg + 3 of the tile at
// dims 4 dc .. + 3 and HD / 2 + 4 dc .. + 3.
// - Loads: an instruction reads 8 rows x 128 bytes, whole lines.
// - K: with a full rotary a dim and its partner d + HD / 2 are in one thread
//   (a partial rotary takes the partner from LDS).  bf16 of 4 dims, 8 bytes
//   per row and half.
// - V^T: the thread writes its 4 keys of a d-row as 8 bytes, so the 8 lanes
//   of one dc write that d-row's 64 bytes whole, without a transpose in LDS.
//   A row group that is only partly stored (the ends of the run) writes its
//   keys one by one.
// - Norms: f32 squares summed in f64, over the thread's dims, the row's lanes
//   of the wave (shuffles) and the waves in order (LDS).
// HBM-bound where it is large, latency-bound in a step.  Against the general
// kernel (64-row blocks, every thread loading the whole row again for the
// norms) and the tile kernel: see the figures at pick_store.
// EPI: biases, norms and RoPE are compiled in (the plain build keeps them
// out: its stores then wait for their own loads only).  HILO: the lo planes
// are written too.  LIST: the rows go to the positions of a sorted list
// (split_active's rows), 32 rows of the list per workgroup; V is turned in
// LDS, so that a store instruction's 2-byte writes are 32 rows of two d-rows
// and fall into the few 32-key tiles that sorted positions span.
template <int HD, bool EPI, bool HILO, bool LIST>
__global__ __launch_bounds__(HD) void kv_store_run_kernel(const StoreArgs a) {
    constexpr int RPG = 4, NRG = VT_KEYS / RPG;  // rows per thread, row groups
    constexpr int NWV = HD / 64;                 // waves
    const int x = blockIdx.x & 7;  // (XCD placement as kv_store_kernel)
    if (x < a.xcd_lo || x >= a.xcd_lo + a.xcd_n) return;
    const int lid = (x - a.xcd_lo) * a.per_xcd + (int)(blockIdx.x >> 3);
    if (lid >= a.n_head_kv * a.n_rb * 2) return;
    const int g = lid / (2 * a.n_rb), rest = lid - g * 2 * a.n_rb;
    const bool is_v = rest & 1;
    const int kt = LIST ? 0 : a.pos0 / VT_KEYS + (rest >> 1);  // key tile
    const int tid = threadIdx.x, rg = tid % NRG, dc = tid / NRG;
    const int p0 = kt * VT_KEYS + rg * RPG;  // first position of this thread
    // its first row (rows outside [0, n) are not stored)
    const int r0 = LIST ? (rest >> 1) * VT_KEYS + rg * RPG : p0 - a.pos0;
    int lp[RPG];  // LIST: the rows' positions
    if constexpr (LIST) {
#pragma unroll
        for (int j = 0; j < RPG; ++j) lp[j] = a.pos[min(r0 + j, a.n - 1)];
    }
    const float* src = (is_v ? a.v : a.k) + (size_t)g * HD + 4 * dc;
    f32x4 xa[RPG], xb[RPG];  // dims 4 dc .., dims HD / 2 + 4 dc ..
#pragma unroll
    for (int j = 0; j < RPG; ++j) {
        const float* row = src + (size_t)min(max(r0 + j, 0), a.n - 1) * a.rstride;
        xa[j] = *reinterpret_cast<const f32x4*>(row);
        xb[j] = *reinterpret_cast<const f32x4*>(row + HD / 2);
    }
    if constexpr (EPI) {
        const int half = a.rot / 2;
        const bool rope = a.rope && !is_v;
        // (sin, cos) of pairs jj .. jj + 3 at each row's position, for each
        // of the thread's two pieces; a full rotary's two pieces share theirs
        f32x4 ta[RPG][2], tb[RPG][2];
        const int da = 4 * dc, db = HD / 2 + 4 * dc;
        auto table = [&](f32x4 (&t)[RPG][2], int d0) __attribute__((always_inline)) {
            const int jj = d0 < half ? d0 : d0 - half;
#pragma unroll
            for (int j = 0; j < RPG; ++j) {
                const int pos = LIST ? lp[j] : a.pos0 + min(max(r0 + j, 0), a.n - 1);
                const float* e = a.rope + ((size_t)pos * half + jj) * 2;
                t[j][0] = *reinterpret_cast<const f32x4*>(e);
                t[j][1] = *reinterpret_cast<const f32x4*>(e + 4);
            }
        };
        if (rope && da < a.rot) table(ta, da);
        if (rope && a.rot != HD && db < a.rot) table(tb, db);
        const float* bias = is_v ? a.vb : a.kb;
        const float* gain = is_v ? nullptr : a.kn_w;
        const bool norm = is_v ? a.v_norm != 0 : a.kn_w != nullptr;
        f32x4 wa = {}, wb = {};
        if (gain) {
            wa = *reinterpret_cast<const f32x4*>(gain + da);
            wb = *reinterpret_cast<const f32x4*>(gain + db);
        }
        if (bias) {  // (only where given: adding a zero would turn -0.0 into +0.0)
            const f32x4 ba = *reinterpret_cast<const f32x4*>(bias + (size_t)g * HD + da);
            const f32x4 bb = *reinterpret_cast<const f32x4*>(bias + (size_t)g * HD + db);
#pragma unroll
            for (int j = 0; j < RPG; ++j) {
                xa[j] += ba;
                xb[j] += bb;
            }
        }
        if (norm) {  // rms_norm_inplace (ops.rs:106-114) / rms_norm_noscale
            __shared__ double s_ss[NWV][VT_KEYS];
#pragma unroll
            for (int j = 0; j < RPG; ++j) {
                double t = 0.0;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float v = e < 4 ? xa[j][e & 3] : xb[j][e & 3];
                    const float sq = v * v;
                    t += (double)sq;
                }
#pragma unroll
                for (int off = NRG; off < 64; off <<= 1) t += __shfl_xor(t, off);
                if ((tid & 63) < NRG) s_ss[tid >> 6][rg * RPG + j] = t;
            }
            __syncthreads();
#pragma unroll
            for (int j = 0; j < RPG; ++j) {
                double t = s_ss[0][rg * RPG + j];
#pragma unroll
                for (int w = 1; w < NWV; ++w) t += s_ss[w][rg * RPG + j];
                const float sc = 1.0f / (float)sqrt(t / (double)HD + (double)a.kn_eps);
                if (gain) {
                    xa[j] = xa[j] * sc * wa;
                    xb[j] = xb[j] * sc * wb;
                } else {
                    xa[j] *= sc;
                    xb[j] *= sc;
                }
            }
        }
        if (rope && a.rot == HD) {
#pragma unroll
            for (int j = 0; j < RPG; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float sn = ta[j][e >> 1][2 * (e & 1)], cs = ta[j][e >> 1][2 * (e & 1) + 1];
                    const float lo = xa[j][e], hi = xb[j][e];
                    xa[j][e] = rope_lo(lo, hi, sn, cs);
                    xb[j][e] = rope_hi(lo, hi, sn, cs);
                }
        } else if (rope) {
            if constexpr (HD <= 256) {  // (host: a partial rotary at 512 takes kv_store_kernel)
                __shared__ __align__(16) float s_k[VT_KEYS][HD + 4];
#pragma unroll
                for (int j = 0; j < RPG; ++j) {
                    *reinterpret_cast<f32x4*>(&s_k[rg * RPG + j][da]) = xa[j];
                    *reinterpret_cast<f32x4*>(&s_k[rg * RPG + j][db]) = xb[j];
                }
                __syncthreads();
                auto rotate = [&](f32x4 (&y)[RPG], const f32x4 (&t)[RPG][2], int d0) __attribute__((always_inline)) {
                    const int pd = d0 < half ? d0 + half : d0 - half;
#pragma unroll
                    for (int j = 0; j < RPG; ++j) {
                        const f32x4 yp = *reinterpret_cast<const f32x4*>(&s_k[rg * RPG + j][pd]);
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const float sn = t[j][e >> 1][2 * (e & 1)], cs = t[j][e >> 1][2 * (e & 1) + 1];
                            y[j][e] = d0 < half ? rope_lo(y[j][e], yp[e], sn, cs) : rope_hi(yp[e], y[j][e], sn, cs);
                        }
                    }
                };
                if (da < a.rot) rotate(xa, ta, da);
                if (db < a.rot) rotate(xb, tb, db);
            }
        }
    }
    // the bf16 halves: hi, and lo = bf16 of what that rounding dropped (one
    // turning buffer for both: declared in the lambda, each conversion had its
    // own, and a hi/lo list workgroup twice the LDS)
    __shared__ __align__(8) uint16_t s_v[LIST ? HD : 1][VT_KEYS + 4];
    auto put = [&](uint16_t* plane, auto conv) __attribute__((always_inline)) {
        if (!is_v) {
            uint16_t* head = plane + (size_t)g * a.cap * HD + 4 * dc;
#pragma unroll
            for (int j = 0; j < RPG; ++j) {
                if (r0 + j < 0 || r0 + j >= a.n) continue;
                uint16_t* dst = head + (size_t)(LIST ? lp[j] : p0 + j) * HD;
                *reinterpret_cast<uint2*>(dst) =
                    make_uint2((uint32_t)conv(xa[j][0]) | ((uint32_t)conv(xa[j][1]) << 16),
                               (uint32_t)conv(xa[j][2]) | ((uint32_t)conv(xa[j][3]) << 16));
                *reinterpret_cast<uint2*>(dst + HD / 2) =
                    make_uint2((uint32_t)conv(xb[j][0]) | ((uint32_t)conv(xb[j][1]) << 16),
                               (uint32_t)conv(xb[j][2]) | ((uint32_t)conv(xb[j][3]) << 16));
            }
            return;
        }
        if constexpr (LIST) {
            __syncthreads();  // (the lo plane's turn: the hi values are read)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                uint16_t h[RPG];
#pragma unroll
                for (int j = 0; j < RPG; ++j) h[j] = conv(e < 4 ? xa[j][e & 3] : xb[j][e & 3]);
                *reinterpret_cast<uint2*>(&s_v[(e < 4 ? 0 : HD / 2) + 4 * dc + (e & 3)][rg * RPG]) =
                    make_uint2((uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16));
            }
            __syncthreads();
            const int row = tid % VT_KEYS, r = (rest >> 1) * VT_KEYS + row;
            if (r < a.n) {
                const int pos = a.pos[r];
                uint16_t* dst = plane + (size_t)g * HD * a.cap + (size_t)(pos / VT_KEYS) * (HD * VT_KEYS) + pos % VT_KEYS;
#pragma unroll 8
                for (int d = tid / VT_KEYS; d < HD; d += HD / VT_KEYS) dst[(size_t)d * VT_KEYS] = s_v[d][row];
            }
            return;
        }
        uint16_t* dst = plane + (size_t)g * HD * a.cap + (size_t)kt * (HD * VT_KEYS) + rg * RPG;
        const bool whole = r0 >= 0 && r0 + RPG <= a.n;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            uint16_t* row = dst + (size_t)((e < 4 ? 0 : HD / 2) + 4 * dc + (e & 3)) * VT_KEYS;
            uint16_t h[RPG];
#pragma unroll
            for (int j = 0; j < RPG; ++j) h[j] = conv(e < 4 ? xa[j][e & 3] : xb[j][e & 3]);
            if (whole) {
                *reinterpret_cast<uint2*>(row) =
                    make_uint2((uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16));
            } else {
#pragma unroll
                for (int j = 0; j < RPG; ++j)
                    if (r0 + j >= 0 && r0 + j < a.n) row[j] = h[j];
            }
        }
    };
    put(is_v ? a.vtc : a.kc, [](float v) { return f2bf(v); });
    if constexpr (HILO) put(is_v ? a.vlo : a.klo, [](float v) { return f2bf(v - bf2f(f2bf(v))); });
}

// One thread per (row, kv head, d).
template <int HD>
__global__ __launch_bounds__(256) void kv_gather_kernel(const GatherArgs a) {
    const size_t total = (size_t)a.n * a.n_head_kv * a.hd;
    for (size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x; idx < total;
         idx += (size_t)gridDim.x * 256) {
        const int d = (int)(idx % a.hd);
        const size_t rg = idx / a.hd;
        const int g = (int)(rg % a.n_head_kv);
        const int r = (int)(rg / a.n_head_kv);
        const int pos = a.pos[r];
        const size_t ki = ((size_t)g * a.cap + pos) * HD + d;
        a.out_k[idx] = a.klo ? bf2f(a.kc[ki]) + bf2f(a.klo[ki]) : bf2f(a.kc[ki]);
        const size_t vi = ((size_t)g * a.cap + (size_t)(pos / VT_KEYS) * VT_KEYS) * HD + (size_t)d * VT_KEYS +
                          pos % VT_KEYS;
        a.out_v[idx] = a.vlo ? bf2f(a.vtc[vi]) + bf2f(a.vlo[vi]) : bf2f(a.vtc[vi]);
    }
}

template <int HD, bool LIST>
void launch_run(const StoreArgs& a, bool epi, dim3 grid, hipStream_t st) {
    if (a.klo) {
        if (epi)
            hipLaunchKernelGGL((kv_store_run_kernel<HD, true, true, LIST>), grid, dim3(HD), 0, st, a);
        else
            hipLaunchKernelGGL((kv_store_run_kernel<HD, false, true, LIST>), grid, dim3(HD), 0, st, a);
    } else {
        if (epi)
            hipLaunchKernelGGL((kv_store_run_kernel<HD, true, false, LIST>), grid, dim3(HD), 0, st, a);
        else
            hipLaunchKernelGGL((kv_store_run_kernel<HD, false, false, LIST>), grid, dim3(HD), 0, st, a);
    }
}

enum StoreKernel { STORE_GENERAL, STORE_RUN, STORE_TILES };

// The kernel of a store.  The run kernel takes every call whose head dim fills
// its tile, the tile kernel whole 32-key tiles of bf16 layers up to head dim
// 256; the general kernel takes all.  g: (kv head, 32 rows) pairs, as many as
// the tile kernel has workgroups, per 256 CUs (a batch slot's store has only
// its XCDs); the run kernel has twice as many, of half the work each.  So up
// to 128 it fills CUs that the others leave idle, and past that its second
// load of the epilogue's operands and its half-rows of DRAM traffic count.
// us, heads x head dim:
// - with RoPE, not whole bf16 tiles: run (general / run: 16 x 128, 512 rows
//   from position 517, norm + RoPE 12.6 / 5.7; hi/lo 8 x 256, 4352 rows 97 / 35;
//   2 x 512, 256 rows 12.8 / 8.7; 32 x 128, 145 listed rows 10.3 / 5.3).
// - norms or biases alone, the same: run, but for hi/lo layers and lists at
//   head dim 512 with up to 64 pairs, where the general kernel's 64-wide
//   pieces fill more CUs (K norm, hi/lo, 256 rows of 2 x 512 7.8 / 9.3, 1536
//   17.4 / 11.0; rows past whole 64s cost it a second pass: 145 14.6 / 9.2).
// - nothing to compute: contiguous rows, run (32 x 128, 256 rows 7.1 / 5.1),
//   but for a few rows of a hi/lo layer (8 x 256, 32 rows 5.4 / 5.8, 64 6.2 /
//   5.8).  Lists and hi/lo tiles: at head dims 64 and 128 run up to the pairs
//   where the chip is full (list: 32 x 128, 128 rows 4.2 / 3.8, 512 7.1 / 8.5,
//   1024 14.3 / 13.5; hi/lo 512 10.5 / 12.6, 1024 18.8 / 19.1; 12 x 64, 512
//   4.0 / 3.5, 2560 6.8 / 8.0), at 256 and 512 the general kernel's pieces
//   until they fill it (list: 8 x 256, 145 4.1 / 4.7, 1536 12.3 / 11.8; hi/lo
//   tiles: 2 x 512, 256 4.3 / 6.4, 8 x 512, 512 9.1 / 8.9).
// - whole bf16 tiles with an epilogue, tile / run: partial rotaries turn
//   through LDS on both, tile (16 x 128, 256 rows 4.2 / 4.5, 1024 6.7 / 8.8; 8
//   x 256 6.4 / 5.9 at 512, 7.3 / 8.7 at 1024; with a norm at 256 9.9 / 7.5);
//   head dim 64 (a wave's 8 rows in run are 2 KB): tile (8 x 64, K norm, 256
//   3.5 / 4.2), but for a full rotary without a lone K norm (RoPE 3.4 / 3.3 at
//   256, 3.6 / 3.8 at 768, 4.7 / 4.5 at 1536); head dim 128: run while it
//   fills idle CUs (16 x 128, K norm 5.1 / 4.7 at 256, 7.0 / 7.3 at 1024; bias +
//   RoPE 5.3 / 4.2, 17.1 / 17.7 at 2560; norm + RoPE 6.5 / 5.2, 18.5 / 19.0),
//   always with the V norm (two norms in one thread: 14.0 / 11.9 at 1536); head
//   dim 256: run (8 x 256, norm + RoPE 10.9 / 6.3 at 256, 35.9 / 29.4 at 4352),
//   but for biases alone past 128 pairs (16 x 256, 1024 10.5 / 12.9).
StoreKernel pick_store(int hd_tile, const StoreArgs& a, int p0, bool epi) {
    const bool partial = a.rope && a.rot != a.hd;
    const bool run = a.vec && a.hd == hd_tile && !a.klo == !a.vlo &&
                     (!partial || (hd_tile <= 256 && a.rot % 8 == 0 && a.rot <= a.hd)) &&
                     (((uintptr_t)a.kn_w | (uintptr_t)a.kb | (uintptr_t)a.vb | (uintptr_t)a.rope) & 15) == 0;
    if (!run) return STORE_GENERAL;
    const bool hilo = a.klo != nullptr, list = p0 < 0, kn = a.kn_w != nullptr, vn = a.v_norm != 0;
    const bool whole = !list && p0 % VT_KEYS == 0 && a.n % VT_KEYS == 0;
    const long g = (long)a.n_head_kv * ((a.n + VT_KEYS - 1) / VT_KEYS) * 8 / a.xcd_n;
    if (whole && !hilo && hd_tile <= 256) {
        bool tiles;
        if (!epi)
            tiles = true;
        else if (hd_tile == 64)
            tiles = !a.rope || partial || (kn && !vn) || (g > 128 && g <= 256) || g >= 1024;
        else if (partial)
            tiles = hd_tile == 128 || (!kn && !vn && g > 128);
        else if (!a.rope && !vn && !(kn && hd_tile == 256))
            tiles = g > 128;
        else
            tiles = hd_tile == 128 && !vn && g >= (kn || a.n_head_kv < 16 ? 1024 : 512);
        return tiles ? STORE_TILES : STORE_RUN;
    }
    bool general;
    if (epi)
        general = hd_tile == 512 && !a.rope && !vn && g <= 64 && (hilo ? list || whole : list && !kn) &&
                  (!kn || a.n % SR == 0);
    else if (!list && !whole)
        general = hilo && a.n <= (hd_tile >= 256 ? hd_tile / 8 : 4);
    else if (hd_tile == 64)
        general = g > (hilo ? 320 : 640);
    else if (hd_tile == 128)
        general = g > 128 && (hilo || g < 1024);
    else
        general = g <= (hd_tile == 256 ? (list ? 320 : 128) : (list ? 192 : 64)) && (hilo || whole || a.n >= VT_KEYS);
    return general ? STORE_GENERAL : STORE_RUN;
}

}  // namespace

hipError_t launch_store(int hd_tile, const StoreArgs& args, hipStream_t st) {
    if (args.n <= 0) return hipSuccess;
    if (hd_tile != 64 && hd_tile != 128 && hd_tile != 256 && hd_tile != 512) return hipErrorInvalidValue;
    StoreArgs a = args;
    if (a.rstride == 0) a.rstride = a.n_head_kv * a.hd;  // (packed rows)
    if (a.rstride < a.n_head_kv * a.hd) return hipErrorInvalidValue;
    // Batch slot b of nb: the attention launch puts the slot's kv heads on
    // XCDs [8b/nb, 8(b+1)/nb).
    const int nb = a.n_batch > 0 ? a.n_batch : 1;
    a.xcd_lo = 8 * a.batch / nb;
    a.xcd_n = std::max(1, 8 * (a.batch + 1) / nb - a.xcd_lo);
    const int p0 = a.pos0 >= 0 ? a.pos0 : (a.pos == nullptr ? 0 : -1);
    const bool epi = a.kn_w || a.kb || a.vb || a.v_norm || a.rope;
    const StoreKernel kernel = pick_store(hd_tile, a, p0, epi);
    if (kernel == STORE_TILES) {
        a.pos0 = p0;
        const int work = a.n_head_kv * (a.n / VT_KEYS);
        a.per_xcd = (work + a.xcd_n - 1) / a.xcd_n;
        const dim3 grid((unsigned)(8 * a.per_xcd));
        switch (hd_tile * 2 + (epi ? 1 : 0)) {
            case 128: hipLaunchKernelGGL((kv_store_tiles_kernel<64, false>), grid, dim3(256), 0, st, a); break;
            case 129: hipLaunchKernelGGL((kv_store_tiles_kernel<64, true>), grid, dim3(256), 0, st, a); break;
            case 256: hipLaunchKernelGGL((kv_store_tiles_kernel<128, false>), grid, dim3(256), 0, st, a); break;
            case 257: hipLaunchKernelGGL((kv_store_tiles_kernel<128, true>), grid, dim3(256), 0, st, a); break;
            case 512: hipLaunchKernelGGL((kv_store_tiles_kernel<256, false>), grid, dim3(256), 0, st, a); break;
            default: hipLaunchKernelGGL((kv_store_tiles_kernel<256, true>), grid, dim3(256), 0, st, a); break;
        }
        return hipGetLastError();
    }
    if (kernel == STORE_RUN) {
        const bool list = p0 < 0;
        a.pos0 = p0;
        a.n_rb = list ? (a.n + VT_KEYS - 1) / VT_KEYS : (p0 + a.n - 1) / VT_KEYS - p0 / VT_KEYS + 1;
        const int work = a.n_head_kv * a.n_rb * 2;
        a.per_xcd = (work + a.xcd_n - 1) / a.xcd_n;
        const dim3 grid((unsigned)(8 * a.per_xcd));
        switch (hd_tile * 2 + (list ? 1 : 0)) {
            case 128: launch_run<64, false>(a, epi, grid, st); break;
            case 129: launch_run<64, true>(a, epi, grid, st); break;
            case 256: launch_run<128, false>(a, epi, grid, st); break;
            case 257: launch_run<128, true>(a, epi, grid, st); break;
            case 512: launch_run<256, false>(a, epi, grid, st); break;
            case 513: launch_run<256, true>(a, epi, grid, st); break;
            case 1024: launch_run<512, false>(a, epi, grid, st); break;
            default: launch_run<512, true>(a, epi, grid, st); break;
        }
        return hipGetLastError();
    }
    a.n_rb = (a.n + SR - 1) / SR;
    const int work = a.n_head_kv * (hd_tile / SD) * a.n_rb;
    a.per_xcd = (work + a.xcd_n - 1) / a.xcd_n;
    const dim3 grid((unsigned)(8 * a.per_xcd));
    switch (hd_tile) {
        case 64: hipLaunchKernelGGL(kv_store_kernel<64>, grid, dim3(256), 0, st, a); break;
        case 128: hipLaunchKernelGGL(kv_store_kernel<128>, grid, dim3(256), 0, st, a); break;
        case 256: hipLaunchKernelGGL(kv_store_kernel<256>, grid, dim3(256), 0, st, a); break;
        default: hipLaunchKernelGGL(kv_store_kernel<512>, grid, dim3(256), 0, st, a); break;
    }
    return hipGetLastError();
}

hipError_t launch_gather(int hd_tile, const GatherArgs& a, hipStream_t st) {
    const size_t total = (size_t)a.n * a.n_head_kv * a.hd;
    if (total == 0) return hipSuccess;
    size_t blocks = (total + 255) / 256;
    if (blocks > 65535) blocks = 65535;
    switch (hd_tile) {
        case 64: hipLaunchKernelGGL(kv_gather_kernel<64>, dim3((unsigned)blocks), dim3(256), 0, st, a); break;
        case 128: hipLaunchKernelGGL(kv_gather_kernel<128>, dim3((unsigned)blocks), dim3(256), 0, st, a); break;
        case 256: hipLaunchKernelGGL(kv_gather_kernel<256>, dim3((unsigned)blocks), dim3(256), 0, st, a); break;
        case 512: hipLaunchKernelGGL(kv_gather_kernel<512>, dim3((unsigned)blocks), dim3(256), 0, st, a); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace dr
