// attn_hilo32.hip -- the hi/lo attention (f32-accurate scores and values from
// bf16 halves, see attn_hilo.hip for the arithmetic) at head dims 256 and 512
// under position masks (no mask, window, causal prefix, query sequence ids):
// the layers DiffusionGemma runs at kq_scale 1.0 (forward.rs:338-341).  Short
// key loops without a bias or a rotary stay on the 16-row kernel (plan_hilo).
//
// What bounds it.  A hi/lo tile costs 2.5 times the matrix work of a bf16
// one (three products for the scores, two for the values), and the operands
// of K and V^T come from LDS.  With 16-row waves every operand read from LDS
// feeds 16 query rows, and LDS, not the matrix cores, sets the pace (4096
// against 2560 cycles per 128 rows and 32 keys).  Here a wave holds 32 query
// rows (v_mfma_f32_32x32x16_bf16) and 256 head dims, so each LDS byte feeds
// twice the rows: 4 waves, one per SIMD, up to 512 registers each (Q hi and
// lo 128, O^T 128).
//   head dim 256: four row blocks of 32, a wave each (128 rows per workgroup);
//   head dim 512: two row blocks, each of two waves that hold half the head
//   dims (64 rows per workgroup); the halves of every score meet in LDS.
//
// One wave per SIMD has nothing else to run while it waits, so the loop is
// software-pipelined: the scores of tile t + 1 are multiplied while the
// softmax of tile t runs on the VALU between the MFMAs, then tile t's values.
// Every LDS operand is read two steps ahead of its MFMA and the DMA of the
// next tiles is spread over the steps.
//   head dim 256: K and V^T tiles are double-buffered (128 KB), one barrier
//   per tile;
//   head dim 512: a tile is 128 KB, so K(t + 2) streams in while tile t's
//   values are multiplied and V^T(t) while the next tile's scores are.
//
// Measured against the 16-row kernel (and, with RoPE, the copy of Q and the
// epilogue pass it needs first), 16 query heads, one layer with its store:
//   8 KV heads, hd 256, window 1024, 256 rows x 4352 keys    59.0 ->  50.9 us
//   2 KV heads, hd 512, 256 rows x 4352 keys                168.2 -> 133.6 us
//   8 KV heads, hd 256, window 1024, causal prompt of 4096
//   and 256 canvas rows (every row asks)                    535.6 -> 324.9 us
// and, with the run store, by reading Q and writing the rows through LDS
//   47.3 -> 44.2, 125.4 -> 122.7 and 254.9 -> 243.0 us.
// A tile of 128 rows and 32 keys takes 2.35 us per CU at head dim 256 (1140
// TFLOP/s over the chip, where a 8192^3 bf16 matrix product reaches 1280),
// 2.4-3.2 us per 64 rows at 512.  The first pass above is bound beyond that by
// the memory past the L2s: its K and V^T planes hit there in 17 % of the
// requests, so that 1.13 GB are fetched and 71 MB written, at 4.95 TB/s (a
// large copy: 5.0); matrix cores busy 44 %, no LDS bank conflicts.  Splitting the accumulator in two, reading
// LDS four steps ahead, and grouping the MFMAs with VALU instructions
// changed none of these by 1 %.
//
// Masks.  Under a window and a causal prefix the keys that a row sees are an
// interval of positions.  A workgroup walks the union of its rows' intervals
// (a causal prompt's rows end at their own position: half the tiles of a
// first pass), and only tiles that some row of a wave sees in part are masked
// per element.
#include "attn_common.hpp"

#include <limits.h>
#include <math.h>

namespace dr {
namespace {

template <int HD>
struct Hilo32Geom {
    static constexpr int NW = 4;                    // waves per workgroup, one per SIMD
    static constexpr int NT = NW * 64;
    static constexpr int DSPLIT = HD / 256;         // waves per 32-row block
    static constexpr int RBW = NW / DSPLIT;         // 32-row blocks per workgroup
    static constexpr int QROWS = RBW * 32;
    static constexpr int KCH = HD / 8;              // 16-byte chunks per K row
    static constexpr int TILE = BN * HD;            // bf16 elements of a K or V^T tile (hi or lo)
    static constexpr int TILE_B = TILE * 2;         // its bytes
    static constexpr int NST = 16;                  // score steps of 16 head dims per wave
    static constexpr int NDB = 8;                   // 32-dim blocks of a wave's O^T
    static constexpr int NBUF = DSPLIT == 1 ? 2 : 1;
    static constexpr int DMAW = 2 * TILE_B / 1024 / NW;  // DMA instructions per wave: K hi + lo (and as many V^T)
    static constexpr int XCH_F = DSPLIT > 1 ? NW * 16 * 64 : 0;  // floats of the score exchange
    static constexpr size_t LDS_BYTES = (size_t)NBUF * 4 * TILE_B + (size_t)XCH_F * 4;
    static_assert(DMAW == NST / 2 * DSPLIT, "one DMA of K and of V^T per step (two at hd 512)");
    static_assert(NW * 32 * 1024 <= LDS_BYTES, "the output turns in the tiles' LDS");
    static_assert(LDS_BYTES <= 159 * 1024, "LDS budget");
};

// a + (16 lanes away) in the even rows of 16 lanes, b + the same in the odd
// ones
__device__ __forceinline__ double swap_add16(double a, double b) {
#if defined(__HIP_DEVICE_COMPILE__)
    const uint64_t ua = __builtin_bit_cast(uint64_t, a), ub = __builtin_bit_cast(uint64_t, b);
    const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)ua, (uint32_t)ub, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((uint32_t)(ua >> 32), (uint32_t)(ub >> 32), false, false);
    return __builtin_bit_cast(double, (uint64_t)lo[0] | ((uint64_t)hi[0] << 32)) +
           __builtin_bit_cast(double, (uint64_t)lo[1] | ((uint64_t)hi[1] << 32));
#else
    return a + b;
#endif
}

__device__ __forceinline__ float xor32_max(float x) { return __builtin_fmaxf(x, __shfl_xor(x, 32)); }

template <int HD>
__global__ __launch_bounds__(Hilo32Geom<HD>::NT) void attn_hilo32_kernel(const AttnArgs a) {
    using G = Hilo32Geom<HD>;
    constexpr int NW = G::NW, RBW = G::RBW, DSPLIT = G::DSPLIT, KCH = G::KCH, TILE_B = G::TILE_B;
    constexpr int NST = G::NST, NDB = G::NDB, NBUF = G::NBUF, DMAW = G::DMAW, QROWS = G::QROWS;
    extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
    __shared__ int s_red[2][NW];
    // LDS: K [NBUF][hi, lo] tiles (rows in sigma order, chunks swizzled), V^T
    // [NBUF][hi, lo] tiles, then the score exchange
    char* const lds = reinterpret_cast<char*>(smem);
    constexpr int K_OFF = 0, V_OFF = NBUF * 2 * TILE_B, X_OFF = 2 * NBUF * 2 * TILE_B;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rbw = wave % RBW, dh = wave / RBW;  // row block, head-dim half
    const int col = lane & 31, hf = lane >> 5;    // query column, lane half

    // ---- workgroup -> (batch, kv head, split, row group): XCD-grouped, row
    // group fastest (an XCD's L2 then holds a few heads' key ranges).  Row
    // groups run from the last one down: under a causal prefix the later rows
    // see more keys, and the long workgroups should not start last.
    const int nwg = a.n_wg, hw = blockIdx.x;
    const int lid = (nwg & 7) == 0 ? (hw & 7) * (nwg >> 3) + (hw >> 3) : hw;
    const int q1 = udiv(lid, a.rowgroups, a.mg_rowgroups);
    const int rg = a.rowgroups - 1 - (lid - q1 * a.rowgroups);
    const int q2 = udiv(q1, a.n_split, a.mg_split);
    const int split = q1 - q2 * a.n_split;
    const int b = udiv(q2, a.n_head_kv, a.mg_hkv);
    const int g = q2 - b * a.n_head_kv;
    const AttnSlot S = a.slot[b];
    const int rows_total = a.group * S.nq;
    const int wg_row0 = rg * QROWS;
    if (wg_row0 >= rows_total) return;  // uniform over the workgroup and all its splits
    const int r = wg_row0 + rbw * 32 + col;
    const bool rvalid = r < rows_total;
    int hg = 0, qi = 0;
    if (rvalid) row_split(r, S.nq, __builtin_amdgcn_rcpf((float)S.nq), a.group, hg, qi);

    // ---- the interval [klo, khi) of keys that this lane's row sees, the
    // workgroup's tile range, and the keys that every row of the wave sees
    int my_qpos = 0;
    if (rvalid && (a.window >= 0 || a.prefix >= 0 || S.qprefix || a.rope))
        my_qpos = S.qpos0 >= 0 ? S.qpos0 + qi : gload<int>(S.qpos + qi);  // (contiguous: no load)
    int klo = 0, khi = S.nk;
    if (rvalid) {
        const int pref = S.qprefix ? gload<int>(S.qprefix + qi) : a.prefix;
        if (a.window >= 0) {
            klo = (int)max(0L, (long)my_qpos - a.window + 1);
            khi = (int)min((long)S.nk, (long)my_qpos + a.window);
        }
        if (pref >= 0 && my_qpos < pref) khi = min(khi, my_qpos + 1);
        if (S.qseq && gload<int>(S.qseq + qi) != 0) khi = klo;  // (the keys are all of sequence 0)
        if (khi < klo) khi = klo;
    }
    const bool sees = rvalid && khi > klo;
    int wmin = sees ? klo : INT_MAX, wmax = sees ? khi : 0;      // union
    int fmin = rvalid ? klo : 0, fmax = rvalid ? khi : INT_MAX;  // seen by every row: [fmin, fmax)
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) {
        wmin = min(wmin, __shfl_xor(wmin, off));
        wmax = max(wmax, __shfl_xor(wmax, off));
        fmin = max(fmin, __shfl_xor(fmin, off));
        fmax = min(fmax, __shfl_xor(fmax, off));
    }
    fmin = __builtin_amdgcn_readfirstlane(fmin);
    fmax = __builtin_amdgcn_readfirstlane(fmax);
    if (lane == 0) {
        s_red[0][wave] = wmin;
        s_red[1][wave] = wmax;
    }
    __syncthreads();
    int kmin = INT_MAX, kmax = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        kmin = min(kmin, s_red[0][w]);
        kmax = max(kmax, s_red[1][w]);
    }
    kmin = __builtin_amdgcn_readfirstlane(kmin);
    kmax = __builtin_amdgcn_readfirstlane(kmax);
    const int kt_lo = kmax > kmin ? kmin / BN : 0;
    const int kt_hi = kmax > kmin ? (kmax + BN - 1) / BN : 0;
    const int ntiles = kt_hi - kt_lo;
    const int per = (ntiles + a.n_split - 1) / a.n_split;
    const int t0 = kt_lo + min(split * per, ntiles);
    const int t1 = kt_lo + min((split + 1) * per, ntiles);

    // ---- DMA: instruction j of this wave moves 64 chunks (1 KB) of K hi, K
    // lo (or V^T hi, V^T lo).  The first half of a tile pair's instructions
    // is the hi tile's: with 4 waves, waves 0 and 1 move the hi tile.
    const uint32_t plane_bytes = (uint32_t)a.cap * HD * 2;
    const bool lo_wave = wave >= NW / 2;
    const __amdgpu_buffer_rsrc_t rk = make_rsrc((lo_wave ? S.klo : S.k) + (size_t)g * a.cap * HD, plane_bytes);
    const __amdgpu_buffer_rsrc_t rv = make_rsrc((lo_wave ? S.vlo : S.vt) + (size_t)g * HD * a.cap, plane_bytes);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
    const int dma_lds = (lo_wave ? TILE_B : 0) + (wave % (NW / 2)) * DMAW * 1024;  // within a hi + lo pair
    const int dma_first = (wave % (NW / 2)) * DMAW * 64;                            // first chunk of the tile
    // K: LDS chunk (R, pc) holds chunk pc ^ swz(R) of key sigma(R).  A row is
    // KCH chunks (32 or 64): an instruction covers 2 rows (1 at hd 512).
    auto koff = [&](int j) __attribute__((always_inline)) {
        const int idx = dma_first + j * 64 + lane;
        const int R = idx / KCH, pc = idx % KCH;
        return (sigma(R) * HD + ((pc ^ swz<KCH>(R)) << 3)) * 2;
    };
    // V^T: LDS chunk (d, pv) holds chunk pv ^ swz<4>(d) of row d
    auto voff = [&](int j) __attribute__((always_inline)) {
        const int idx = dma_first + j * 64 + lane;
        const int d = idx / (BN / 8), pv = idx % (BN / 8);
        return (d * (BN / 8) + (pv ^ swz<4>(d))) * 16;
    };
    // (V^T's swizzle repeats every 16 rows, so its offsets advance by 1 KB per
    // instruction; K's do not, and stay in registers)
    int kvo[DMAW];
#pragma unroll
    for (int j = 0; j < DMAW; ++j) kvo[j] = koff(j);
    const int vvo = voff(0);
    auto dma_k = [&](int j, int t, int buf) __attribute__((always_inline)) {
        dma16_asm(rk, lds0 + K_OFF + buf * 2 * TILE_B + dma_lds + j * 1024, kvo[j], t * TILE_B);
    };
    auto dma_v = [&](int j, int t, int buf) __attribute__((always_inline)) {
        dma16_asm(rv, lds0 + V_OFF + buf * 2 * TILE_B + dma_lds + j * 1024, vvo, t * TILE_B + j * 1024);
    };
    // the first K tiles are requested before Q is read (Q passes through
    // V^T's part of LDS, so V^T follows it)
    if (t0 < t1) {
#pragma unroll
        for (int j = 0; j < DMAW; ++j) dma_k(j, t0, 0);
        if constexpr (NBUF == 2) {
            const int t = min(t0 + 1, t1 - 1);
#pragma unroll
            for (int j = 0; j < DMAW; ++j) dma_k(j, t, 1);
        }
    }

    // ---- Q: bias, QK-norm and RoPE (forward.rs:291-310), then the hi and lo
    // bf16 halves of q * scale * log2 e as MFMA operands: lane (col, hf) holds
    // row col at head dims dim(st) + 8 hf + (0..7).  Loaded in that layout
    // each instruction touches 32 rows, and Q took 8 of the 34 us of C5's
    // sliding layer.  So 32 lanes read a row (two rows per instruction, lane
    // l32 the dims 4 l32 .. + 3 of each 128, a dim's rotary partner d + HD / 2
    // among them), finish it there and pass the halves through LDS, 16 rows
    // of a row block at a time.  The waves of a split row block finish half
    // of its rows each.  (16-byte chunk c of a row's half sits at chunk c ^
    // (row & 15): the operand reads are conflict-free.)
    auto dim = [&](int st) __attribute__((always_inline)) { return (st / 8) * (HD / 2) + dh * 128 + 16 * (st % 8); };
    bf16x8 qh[NST], ql[NST];
    {
        constexpr int NP = 8 / DSPLIT, NPC = HD / 128;  // row pairs per wave and pass, 128-dim pieces
        const int l32 = lane & 31;
        char* const qlds = lds + V_OFF + rbw * 16 * (HD * 4);  // [16 rows][hi, lo][HD] bf16
        f32x4 w[NPC];  // the QK-norm's gains, loaded with the rows
#pragma unroll
        for (int c = 0; c < NPC; ++c) w[c] = a.qn_w ? gload<f32x4>(a.qn_w + 128 * c + 4 * l32) : f32x4{};
#pragma unroll
        for (int st = 0; st < NST; ++st) qh[st] = ql[st] = bf16x8{};
#pragma unroll 1  // (half the code: the prologue is straight-line and runs once)
        for (int pass = 0; pass < 2; ++pass) {
            const int i0 = 16 * pass + dh * 2 * NP;  // first row of this wave
            f32x4 x[NP][NPC], tab[NP][NPC];          // (pieces c and c + NPC / 2 share tab[.][2 c], [2 c + 1])
            int head[NP];
#pragma unroll
            for (int k = 0; k < NP; ++k) {  // this lane's row of pair k: i0 + 2 k + hf
                const int ri = __shfl(qi, i0 + 2 * k + hf);
                head[k] = (g * a.group + __shfl(hg, i0 + 2 * k + hf)) * HD;
                const float* row = static_cast<const float*>(S.q) + (size_t)ri * a.q_rstride + head[k] + 4 * l32;
#pragma unroll
                for (int c = 0; c < NPC; ++c) x[k][c] = gload<f32x4>(row + 128 * c);
            }
            if (a.rope) {  // full rotary: rot == HD (the host checks); pairs 128 c + 4 l32 .. + 3
#pragma unroll
                for (int k = 0; k < NP; ++k) {
                    const float* t = a.rope + (size_t)__shfl(my_qpos, i0 + 2 * k + hf) * HD + 8 * l32;
#pragma unroll
                    for (int c = 0; c < NPC; ++c) tab[k][c] = gload<f32x4>(t + 256 * (c / 2) + 4 * (c & 1));
                }
            }
            if (a.qb) {
#pragma unroll
                for (int k = 0; k < NP; ++k)
#pragma unroll
                    for (int c = 0; c < NPC; ++c) x[k][c] += gload<f32x4>(a.qb + head[k] + 128 * c + 4 * l32);
            }
            // rms_norm_inplace (ops.rs:106-114): f32 squares summed in f64.
            // The rows' sums meet across their 32 lanes together: at each step
            // a lane gives away half of its rows' sums and keeps the rest, so
            // lane (hf, l32) ends up with the sum of pair l32 / (32 / NP).
            if (a.qn_w) {
                double ss[NP];
#pragma unroll
                for (int k = 0; k < NP; ++k) {
                    ss[k] = 0.0;
#pragma unroll
                    for (int e = 0; e < 4 * NPC; ++e) {
                        const float v = x[k][e >> 2][e & 3];
                        const float sq = v * v;
                        ss[k] += (double)sq;
                    }
                }
#pragma unroll
                for (int k = 0; k < NP / 2; ++k) ss[k] = swap_add16(ss[k], ss[k + NP / 2]);
#pragma unroll
                for (int k = 0; k < NP / 4; ++k) {
                    const bool up = (lane & 8) != 0;
                    const double give = up ? ss[k] : ss[k + NP / 4], keep = up ? ss[k + NP / 4] : ss[k];
                    ss[k] = keep + __shfl_xor(give, 8);
                }
                if constexpr (NP == 8) {
                    const bool up = (lane & 4) != 0;
                    const double give = up ? ss[0] : ss[1], keep = up ? ss[1] : ss[0];
                    ss[0] = keep + __shfl_xor(give, 4);
                } else {
                    ss[0] += __shfl_xor(ss[0], 4);
                }
                ss[0] += __shfl_xor(ss[0], 2);
                ss[0] += __shfl_xor(ss[0], 1);
                const float sc = 1.0f / (float)sqrt(ss[0] / (double)HD + (double)a.qn_eps);
#pragma unroll
                for (int k = 0; k < NP; ++k) {
#pragma clang fp contract(off)
                    const float rs = __shfl(sc, (lane & 32) + k * (32 / NP));
#pragma unroll
                    for (int c = 0; c < NPC; ++c) x[k][c] = x[k][c] * rs * w[c];
                }
            }
            if (a.rope) {
#pragma unroll
                for (int k = 0; k < NP; ++k)
#pragma unroll
                    for (int c = 0; c < NPC / 2; ++c)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const float sn = tab[k][2 * c + (e >> 1)][2 * (e & 1)];
                            const float cs = tab[k][2 * c + (e >> 1)][2 * (e & 1) + 1];
                            const float lo = x[k][c][e], hi = x[k][c + NPC / 2][e];
                            x[k][c][e] = rope_lo(lo, hi, sn, cs);
                            x[k][c + NPC / 2][e] = rope_hi(lo, hi, sn, cs);
                        }
            }
            if (pass > 0 && DSPLIT > 1) lds_barrier();  // the first pass's operands are read
            asm volatile("" ::: "memory");
            __builtin_amdgcn_wave_barrier();  // (a wave's own accesses run in order)
#pragma unroll
            for (int k = 0; k < NP; ++k) {
                const int row = dh * 2 * NP + 2 * k + hf;
                // (rows past the last: finite garbage, never stored)
                char* const dst = qlds + row * (HD * 4) + (((l32 >> 1) ^ (row & 15)) << 4) + 8 * (l32 & 1);
#pragma unroll
                for (int c = 0; c < NPC; ++c) {
                    bf16x4 h, lo;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float xs = x[k][c][e] * a.c;
                        h[e] = (__bf16)xs;
                        lo[e] = (__bf16)(xs - (float)h[e]);
                    }
                    *reinterpret_cast<bf16x4*>(dst + 256 * c) = h;
                    *reinterpret_cast<bf16x4*>(dst + 256 * c + HD * 2) = lo;
                }
            }
            if constexpr (DSPLIT > 1) lds_barrier();
            asm volatile("" ::: "memory");
            __builtin_amdgcn_wave_barrier();
            if ((col >> 4) == pass) {
                const char* src = qlds + (col & 15) * (HD * 4);
#pragma unroll
                for (int st = 0; st < NST; ++st) {
                    const int off = ((dim(st) / 8 + hf) ^ (col & 15)) << 4;
                    qh[st] = *reinterpret_cast<const bf16x8*>(src + off);
                    ql[st] = *reinterpret_cast<const bf16x8*>(src + HD * 2 + off);
                }
            }
        }
    }

    f32x16 o[NDB];
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[db][i] = 0.0f;
    float m = -INFINITY, l = 0.0f;
    const bf16x2 ones = {(__bf16)1.0f, (__bf16)1.0f};

    // LDS read addresses: K chunk c(st) = dim(st) / 8 + hf of row col, swizzled
    // in its low four bits; V^T chunk 2 hf + s of row 32 db + col
    const int k_rd = K_OFF + col * (HD * 2) + dh * 256 + ((hf ^ (col & 15)) << 4);
    int v_rd[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) v_rd[s] = V_OFF + dh * (256 * 64) + col * 64 + (((2 * hf + s) ^ swz<4>(col)) << 4);
    auto rd_k = [&](int st, int base, bf16x8& h, bf16x8& lo) __attribute__((always_inline)) {
        const char* p = lds + (base ^ ((st % 8) << 5)) + (st / 8) * HD;
        h = *reinterpret_cast<const bf16x8*>(p);
        lo = *reinterpret_cast<const bf16x8*>(p + TILE_B);
    };
    // PV step v: d-block v / 2, contraction half v % 2
    auto rd_v = [&](int v, int boff, bf16x8& h, bf16x8& lo) __attribute__((always_inline)) {
        const char* p = lds + v_rd[v & 1] + boff + (v >> 1) * 2048;
        h = *reinterpret_cast<const bf16x8*>(p);
        lo = *reinterpret_cast<const bf16x8*>(p + TILE_B);
    };

    constexpr int AHEAD = 2;  // steps an LDS operand is read ahead of its MFMA
    f32x16 s, sn;             // scores of the current and of the next tile

    // One score step of the next tile.
    auto qk_step = [&](int st, int kb, bf16x8 (&fh)[AHEAD + 1], bf16x8 (&fl)[AHEAD + 1])
        __attribute__((always_inline)) {
        if (st + AHEAD < NST) rd_k(st + AHEAD, kb, fh[(st + AHEAD) % (AHEAD + 1)], fl[(st + AHEAD) % (AHEAD + 1)]);
        const bf16x8 kh = fh[st % (AHEAD + 1)], kl = fl[st % (AHEAD + 1)];
        sn = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kh, qh[st], sn, 0, 0, 0);
        sn = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kh, ql[st], sn, 0, 0, 0);
        sn = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kl, qh[st], sn, 0, 0, 0);
    };
    // hd 512: this wave's half of the scores to LDS, and the partner's added
    float* const xch = reinterpret_cast<float*>(lds + X_OFF);
    auto put_half = [&]() __attribute__((always_inline)) {
        f32x4* mine = reinterpret_cast<f32x4*>(xch) + wave * 256 + lane;
#pragma unroll
        for (int i = 0; i < 4; ++i) mine[i * 64] = f32x4{sn[4 * i], sn[4 * i + 1], sn[4 * i + 2], sn[4 * i + 3]};
    };
    auto add_half = [&]() __attribute__((always_inline)) {
        const f32x4* theirs = reinterpret_cast<const f32x4*>(xch) + (wave ^ RBW) * 256 + lane;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const f32x4 u = theirs[i * 64];
#pragma unroll
            for (int e = 0; e < 4; ++e) sn[4 * i + e] = sn[4 * i + e] + u[e];  // (commutes: same bits on both waves)
        }
    };

    // ---- one tile: NEXT says that tile t + 1 exists
    auto step = [&](int t, int kp, auto next) __attribute__((always_inline)) {
        constexpr bool NEXT = decltype(next)::value;
        // K(t + 1) (and V^T(t) where it is double-buffered) has landed; every
        // wave is done with the buffers that the DMA below overwrites
        wait_vmcnt<0>();
        lds_barrier();
        const int cur = NBUF == 2 ? kp : 0, nxt = NBUF == 2 ? kp ^ 1 : 0;
        const int t2 = min(t + 2, t1 - 1), tv = min(t + 1, t1 - 1);
        const int kb = k_rd + nxt * 2 * TILE_B, vb = cur * 2 * TILE_B;
        bf16x8 fh[AHEAD + 1], fl[AHEAD + 1];
        if constexpr (NEXT) {
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) rd_k(i, kb, fh[i], fl[i]);
        }
        // tiles that some row of the wave sees in part: per-element mask
        if (t * BN < fmin || t * BN + BN > fmax) {
            const int k0 = t * BN + 16 * hf - klo;
            const uint32_t n = (uint32_t)(khi - klo);
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = (uint32_t)(k0 + i) < n ? s[i] : -INFINITY;
        }
        if constexpr (NEXT) {
#pragma unroll
            for (int i = 0; i < 16; ++i) sn[i] = 0.0f;
        }
        __builtin_amdgcn_sched_barrier(0);
        // first half of the score steps: the row's maximum
        float mt[8];
#pragma unroll
        for (int st = 0; st < NST / 2; ++st) {
            if constexpr (NEXT) {
                if constexpr (NBUF == 2) {
                    dma_k(st, t2, cur);
                    dma_v(st, tv, nxt);
                }
            }
            if constexpr (NBUF == 1) {  // (V^T of tile t - 1 is consumed since the barrier)
                dma_v(2 * st, t, 0);
                dma_v(2 * st + 1, t, 0);
            }
            if constexpr (NEXT) qk_step(st, kb, fh, fl);
            if (st < 5) mt[st] = max3(s[3 * st], s[3 * st + 1], s[3 * st + 2]);
            if (st == 5) mt[5] = max3(mt[0], mt[1], s[15]);
            if (st == 6) mt[6] = max3(mt[2], mt[3], mt[4]);
            if (st == 7) mt[7] = xor32_max(__builtin_fmaxf(mt[5], mt[6]));
            __builtin_amdgcn_sched_barrier(0);
        }
        // The maximum moves with every larger score: the weight of a row's
        // largest score so far is then exactly 1, and at scale 1.0 that key is
        // most of the row.  Moved only past a threshold, as in the other
        // kernels, it is rounded to bf16 like the rest, and the outputs of C5's
        // sliding layer lie 2.0 % further from 64 bits than the 16-row
        // kernel's (its workgroups' ranges are longer); so they lie 19 %
        // closer.  The rescale is hidden under the MFMAs: 45.8 / 45.5 us with a
        // threshold of 8 / without, first pass over 4352 rows 249.4 / 249.1.
        const bool need = mt[7] > m;
        if (__builtin_amdgcn_ballot_w64(need) != 0) {
            const float f = need ? (m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - mt[7])) : 1.0f;
#pragma unroll
            for (int db = 0; db < NDB; ++db) o[db] *= f;
            l *= f;
            m = need ? mt[7] : m;
        }
        const float me = m == -INFINITY ? 0.0f : m;
        // second half: p = 2^(s - m) as bf16 and its sum
        bf16x8 pb[2];
#pragma unroll
        for (int st = 0; st < NST / 2; ++st) {
            if constexpr (NEXT) qk_step(NST / 2 + st, kb, fh, fl);
            const float p0 = __builtin_amdgcn_exp2f(s[2 * st] - me), p1 = __builtin_amdgcn_exp2f(s[2 * st + 1] - me);
            const bf16x2 pr = {(__bf16)p0, (__bf16)p1};
            pb[st >> 2][(2 * st) & 7] = pr[0];
            pb[st >> 2][(2 * st + 1) & 7] = pr[1];
            l = __builtin_amdgcn_fdot2_f32_bf16(pr, ones, l, false);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (DSPLIT > 1 && NEXT) put_half();
        // ---- O^T += V^T P^T
        bf16x8 vh[AHEAD + 1], vl[AHEAD + 1];
        if constexpr (DSPLIT == 1) {
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) rd_v(i, vb, vh[i], vl[i]);
        } else {
            // V^T(t) has landed, every wave is done with K(t + 1), the halves
            // are in LDS
            wait_vmcnt<0>();
            lds_barrier();
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) rd_v(i, vb, vh[i], vl[i]);
            if constexpr (NEXT) add_half();
        }
#pragma unroll
        for (int v = 0; v < 2 * NDB; ++v) {
            if constexpr (DSPLIT > 1 && NEXT) {
                if (v < DMAW / 2) {
                    dma_k(2 * v, t2, 0);
                    dma_k(2 * v + 1, t2, 0);
                }
            }
            if (v + AHEAD < 2 * NDB) rd_v(v + AHEAD, vb, vh[(v + AHEAD) % (AHEAD + 1)], vl[(v + AHEAD) % (AHEAD + 1)]);
            o[v >> 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vh[v % (AHEAD + 1)], pb[v & 1], o[v >> 1], 0, 0, 0);
            o[v >> 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vl[v % (AHEAD + 1)], pb[v & 1], o[v >> 1], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        s = sn;
    };

    if (t0 < t1) {
        // ---- scores of the first tile
        wait_vmcnt<0>();
        lds_barrier();  // (and every wave has its Q: V^T may take that part of LDS)
        if constexpr (NBUF == 2) {
#pragma unroll
            for (int j = 0; j < DMAW; ++j) dma_v(j, t0, 0);
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) sn[i] = 0.0f;
        {
            bf16x8 fh[AHEAD + 1], fl[AHEAD + 1];
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) rd_k(i, k_rd, fh[i], fl[i]);
#pragma unroll
            for (int st = 0; st < NST; ++st) qk_step(st, k_rd, fh, fl);
        }
        if constexpr (DSPLIT > 1) {
            put_half();
            lds_barrier();  // every wave is done with K(t0); the halves are in LDS
            const int t = min(t0 + 1, t1 - 1);
#pragma unroll
            for (int j = 0; j < DMAW; ++j) dma_k(j, t, 0);
            add_half();
        }
        s = sn;
        int t = t0, kp = 0;
        for (; t + 1 < t1; ++t, kp ^= 1) step(t, kp, std::true_type{});
        step(t, kp, std::false_type{});
        wait_vmcnt<0>();  // (no DMA may outlive the workgroup's LDS)
    }

    // ---- the row's sum over its lane halves; out or the split partial.
    // o[db][i] is O^T[d = 256 dh + 32 db + 8 (i / 4) + 4 hf + i % 4][col]: 16
    // bytes of 32 rows per register quad, so the wave turns its 32 rows x 256
    // dims in LDS (chunk c of row q at chunk c ^ q) and stores whole rows
    // (in the register layout the stores of C5's sliding layer, 33 MB of
    // partials, took 6 of its 34 us).
    l += __shfl_xor(l, 32);
    lds_barrier();  // every wave is done with the tiles
    char* const rows = lds + wave * 32 * 1024;
    const float f = a.n_split <= 1 ? __builtin_amdgcn_rcpf(l) : 1.0f;  // no visible key: 0 * inf = NaN (attention.rs:181-185)
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = o[db][4 * j + e] * f;
            *reinterpret_cast<f32x4*>(rows + col * 1024 + (((8 * db + 2 * j + hf) ^ col) << 4)) = v;
        }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    const size_t plane = (size_t)a.n_batch * a.n_head_kv * a.part_rows;
    const size_t prow0 = (size_t)(b * a.n_head_kv + g) * a.part_rows + wg_row0 + rbw * 32;
    const int nrow = min(32, rows_total - wg_row0 - rbw * 32);
#pragma unroll 1
    for (int i0 = 0; i0 < nrow; i0 += 8) {
        f32x4 v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k)
            v[k] = *reinterpret_cast<const f32x4*>(rows + (i0 + k) * 1024 + ((lane ^ (i0 + k)) << 4));
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            float* dst;
            if (a.n_split <= 1) {
                const int ri = __builtin_amdgcn_readlane(qi, i0 + k), rh = __builtin_amdgcn_readlane(hg, i0 + k);
                dst = S.out + (size_t)ri * a.o_rstride + (size_t)(g * a.group + rh) * HD;
            } else {
                dst = a.part_o + ((size_t)split * plane + prow0 + i0 + k) * HD;
            }
            if (i0 + k < nrow) gstore(dst + dh * 256 + 4 * lane, v[k]);
        }
    }
    if (a.n_split > 1 && rvalid && dh == 0 && hf == 0)
        gstore(a.part_ml + ((size_t)split * plane + prow0 + col) * 2, make_float2(m, l));
}

template <int HD>
hipError_t launch_hd(const LaunchPlan& p, const AttnArgs& a, hipStream_t st) {
    using G = Hilo32Geom<HD>;
    auto k = attn_hilo32_kernel<HD>;
    hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)G::LDS_BYTES);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k, dim3(p.n_workgroups), dim3(G::NT), G::LDS_BYTES, st, a);
    return hipGetLastError();
}

}  // namespace

int hilo32_rows(int hd_tile) {
    return hd_tile == 256 ? Hilo32Geom<256>::QROWS : (hd_tile == 512 ? Hilo32Geom<512>::QROWS : 0);
}

hipError_t launch_hilo32(const LaunchPlan& p, const AttnArgs& a, hipStream_t st) {
    if (a.hd != p.hd_tile || p.mask == MASK_KEYS) return hipErrorInvalidValue;
    if (a.rope && a.rot != a.hd) return hipErrorInvalidValue;
    for (int i = 0; i < a.n_batch; ++i)
        if (!a.slot[i].klo || !a.slot[i].vlo) return hipErrorInvalidValue;  // no lo planes
    switch (p.hd_tile) {
        case 256: return launch_hd<256>(p, a, st);
        case 512: return launch_hd<512>(p, a, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace dr
