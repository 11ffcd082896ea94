// attn_rows.hip -- the attention over the cache (attention.rs:101-186) for
// calls with many query rows: first passes, where every position asks, and
// batches of long canvases.  Head dims 64 and 128, bf16 operands, no mask or
// MASK_POS (window, causal prefix, query sequence ids), with the whole Q
// epilogue.
//
// What bounds it.  With rows to fill the chip several times over (32 heads,
// 2560 rows), the matrix cores: a copy of this kernel without softmax, LDS
// reads and DMA still takes 60 % of its time, at 1095 TFLOP/s (a 8192^3 bf16
// product reaches 1280 on the card); DMA and the return of its lines cost
// 15 %, the VALU 8 %.  At 28/4 heads, 2 x 1280 rows (1120 workgroups, little
// over two rounds) the matrix cores are busy 30 % of the CUs' busy time and
// the texture data path, which returns the DMA's lines, 72 % of the call; no
// LDS bank conflicts, 91 % of the lines from L2.  The
// staged kernel's 64-row workgroups of 8 waves (4 key groups of one tile
// each) pass a workgroup barrier per super-tile with a tile's scores, softmax
// and values in sequence.  Here a workgroup is 4 waves, two row blocks of 32
// x two key groups, and two workgroups share a CU, so the waves of a SIMD are
// never in step.  Each also overlaps within itself: per step the softmax of
// tile u runs on the VALU between the MFMAs of tile u - 1's values and tile
// u + 1's scores.  K and V^T tiles are double-buffered in LDS by DMA, one
// barrier per tile.  (Without that second overlap, values in their own
// tile's step, the calls took the same time within 1 %; separate
// accumulators for dependent MFMAs changed nothing.)
// Measured: 28/4 heads, 2 x 1280 rows, all asking: 107 -> 92 us per call (47
// GFLOP); 32 heads, 2560 rows: 193 -> 163 us (107 GFLOP).
//
// Why 64 rows x 2 key groups.  128 rows would halve the K/V stream, but a
// call is few rounds of workgroups: half as long workgroups leave half the
// tail (see plan_attention).  The two key groups meet in LDS at the end.
//
// The running maximum m enters the score product as its accumulator's
// initial value (16 registers holding -m of the lane's row), so p = exp2(S);
// it moves only when a score exceeds it by more than 8 (log2 units), before
// the next tile's scores begin, and O is rescaled once the values of the tile
// before are in it.  (A row's largest weight is exact in bf16 only if m is its
// score.  With half the staged kernel's key groups, so half its maxima, the
// outputs lie 0.1-0.8 % further from 64 bits than that kernel's: 2 x 1280 rows
// of 28/4 heads 3.554e-3 -> 3.565e-3.  A threshold of 2 brings them 0.2-1 %
// closer than its own for 5 % more time, 92.5 -> 98.0 us; of 4, 0.2 % closer to
// 0.5 % further for up to 4 % at head dim 64.)
#include "attn_common.hpp"

#include <limits.h>
#include <math.h>

namespace dr {
namespace {

template <int HD>
struct RowsGeom {
    static constexpr int RB = 2, KQ = 2, NW = RB * KQ, NT = NW * 64;
    static constexpr int QROWS = RB * 32;
    static constexpr int KCH = HD / 8;       // 16-byte chunks per K row
    static constexpr int TILE_B = BN * HD * 2;  // bytes of a K or V^T tile
    static constexpr int NST = HD / 16;      // score steps
    static constexpr int NDB = HD / 32;      // 32-dim blocks of O^T
    static constexpr int DMAW = TILE_B / 1024 / RB;  // DMA instructions per wave: K tile (and as many V^T)
    static constexpr size_t LDS_BYTES = (size_t)KQ * 2 * 2 * TILE_B;  // [key group][K, V^T][buffer]
    static constexpr size_t MERGE_BYTES = (size_t)RB * (HD / 2 + 2) * 64 * 4;  // key group 1's states
    static_assert(MERGE_BYTES <= LDS_BYTES, "the merge reuses the tile buffers");
    static_assert(DMAW >= 1, "DMA split");
};

// maximum of a lane and its partner lane ^ 32
__device__ __forceinline__ float max_xor32(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __builtin_fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
#else
    return x;
#endif
}

template <int HD>
__global__ __launch_bounds__(RowsGeom<HD>::NT, 2) void attn_rows_kernel(const AttnArgs a) {
    using G = RowsGeom<HD>;
    constexpr int RB = G::RB, KQ = G::KQ, NW = G::NW, KCH = G::KCH, TILE_B = G::TILE_B;
    constexpr int NST = G::NST, NDB = G::NDB, DMAW = G::DMAW, QROWS = G::QROWS;
    extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
    __shared__ int s_red[2][NW];
    char* const lds = reinterpret_cast<char*>(smem);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rb = wave % RB, kq = wave / RB;
    const int col = lane & 31, hf = lane >> 5;

    // workgroup -> (batch, kv head, row group), XCD-grouped; later rows first
    // (under a causal prefix they see more keys)
    const int nwg = a.n_wg, hw = blockIdx.x;
    const int lid = (nwg & 7) == 0 ? (hw & 7) * (nwg >> 3) + (hw >> 3) : hw;
    const int q2 = udiv(lid, a.rowgroups, a.mg_rowgroups);
    const int rg = a.rowgroups - 1 - (lid - q2 * a.rowgroups);
    const int b = udiv(q2, a.n_head_kv, a.mg_hkv);
    const int g = q2 - b * a.n_head_kv;
    const AttnSlot S = a.slot[b];
    const int rows_total = a.group * S.nq;
    const int wg_row0 = rg * QROWS;
    if (wg_row0 >= rows_total) return;  // uniform over the workgroup
    const int r = wg_row0 + rb * 32 + col;
    const bool rvalid = r < rows_total;
    int hg = 0, qi = 0;
    if (rvalid) row_split(r, S.nq, __builtin_amdgcn_rcpf((float)S.nq), a.group, hg, qi);

    // ---- the interval [klo, khi) of keys that this lane's row sees, the
    // workgroup's tile range, and the keys that every row of the wave sees
    int my_qpos = 0;
    if (rvalid && (a.window >= 0 || a.prefix >= 0 || S.qprefix || a.rope))
        my_qpos = S.qpos0 >= 0 ? S.qpos0 + qi : gload<int>(S.qpos + qi);
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
    int wmin = sees ? klo : INT_MAX, wmax = sees ? khi : 0;
    int fmin = rvalid ? klo : 0, fmax = rvalid ? khi : INT_MAX;
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
    const int t0 = kmax > kmin ? kmin / BN : 0;
    const int t1 = kmax > kmin ? (kmax + BN - 1) / BN : 0;
    const int nsteps = (t1 - t0 + KQ - 1) / KQ;  // tiles of key group kq: t0 + kq, t0 + kq + KQ, ..
    // (a key group without a tile in the last step multiplies a repeat of
    // the last tile, all of it masked)
    auto tile_of = [&](int u) __attribute__((always_inline)) { return t0 + u * KQ + kq; };

    // ---- DMA: instruction j of this wave moves 64 chunks (1 KB) of its key
    // group's tile, the two row blocks' waves half a tile each
    const uint32_t plane_bytes = (uint32_t)a.cap * HD * 2;
    const __amdgpu_buffer_rsrc_t rk = make_rsrc(S.k + (size_t)g * a.cap * HD, plane_bytes);
    const __amdgpu_buffer_rsrc_t rv = make_rsrc(S.vt + (size_t)g * HD * a.cap, plane_bytes);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
    const int k_base = kq * 4 * TILE_B, v_base = k_base + 2 * TILE_B;  // buffers side by side
    const int dma_first = rb * DMAW * 64;
    int kvo[DMAW];
#pragma unroll
    for (int j = 0; j < DMAW; ++j) {
        const int idx = dma_first + j * 64 + lane;
        const int R = idx / KCH, pc = idx % KCH;
        kvo[j] = (sigma(R) * HD + ((pc ^ swz<KCH>(R)) << 3)) * 2;
    }
    const int vd = (dma_first + lane) / (BN / 8), vp = (dma_first + lane) % (BN / 8);
    const int vvo = (vd * (BN / 8) + (vp ^ swz<4>(vd))) * 16;  // (+ 1 KB per instruction)
    auto dma_k = [&](int j, int t, int buf) __attribute__((always_inline)) {
        dma16_asm(rk, lds0 + k_base + buf * TILE_B + dma_first * 16 + j * 1024, kvo[j], t * TILE_B);
    };
    auto dma_v = [&](int j, int t, int buf) __attribute__((always_inline)) {
        dma16_asm(rv, lds0 + v_base + buf * TILE_B + dma_first * 16 + j * 1024, vvo, t * TILE_B + j * 1024);
    };
    if (nsteps > 0) {
        const int ta = min(tile_of(0), t1 - 1), tb = min(tile_of(1), t1 - 1);
#pragma unroll
        for (int j = 0; j < DMAW; ++j) dma_k(j, ta, 0);
#pragma unroll
        for (int j = 0; j < DMAW; ++j) dma_k(j, tb, 1);
    }

    // ---- Q of this lane's row at head dims 16 st + 8 hf + (0..7): bias,
    // QK-norm and RoPE (forward.rs:291-310), then bf16 of q * scale * log2 e.
    // A dim and its rotary partner d + HD / 2 are steps st and st + NST / 2
    // of one lane.
    bf16x8 qf[NST];
    {
        const size_t head = (size_t)(g * a.group + hg) * HD;
        const float* qrow = static_cast<const float*>(S.q) + (size_t)qi * a.q_rstride + head;
        f32x4 x[NST][2];
#pragma unroll
        for (int st = 0; st < NST; ++st)
#pragma unroll
            for (int p = 0; p < 2; ++p) x[st][p] = gload<f32x4>(qrow + 16 * st + 8 * hf + 4 * p);
        if (a.qb) {
#pragma unroll
            for (int st = 0; st < NST; ++st)
#pragma unroll
                for (int p = 0; p < 2; ++p) x[st][p] += gload<f32x4>(a.qb + head + 16 * st + 8 * hf + 4 * p);
        }
        if (a.qn_w) {  // rms_norm_inplace (ops.rs:106-114): f32 squares summed in f64
            double ss = 0.0;
#pragma unroll
            for (int st = 0; st < NST; ++st)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float v = x[st][e >> 2][e & 3];
                    const float sq = v * v;
                    ss += (double)sq;
                }
            ss += __shfl_xor(ss, 32);
            const float sc = 1.0f / (float)sqrt(ss / (double)HD + (double)a.qn_eps);
#pragma unroll
            for (int st = 0; st < NST; ++st)
#pragma unroll
                for (int p = 0; p < 2; ++p) {
#pragma clang fp contract(off)
                    x[st][p] = x[st][p] * sc * gload<f32x4>(a.qn_w + 16 * st + 8 * hf + 4 * p);
                }
        }
        if (a.rope) {  // full rotary: rot == HD (the planner checks)
            const float* tab = a.rope + (size_t)my_qpos * HD;  // [HD / 2] (sin, cos)
#pragma unroll
            for (int st = 0; st < NST / 2; ++st)
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    const int d0 = 16 * st + 8 * hf + 4 * p;
                    const f32x4 ta = gload<f32x4>(tab + 2 * d0), tb = gload<f32x4>(tab + 2 * d0 + 4);
                    const float sn[4] = {ta[0], ta[2], tb[0], tb[2]}, cs[4] = {ta[1], ta[3], tb[1], tb[3]};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float lo = x[st][p][e], hi = x[st + NST / 2][p][e];
                        x[st][p][e] = rope_lo(lo, hi, sn[e], cs[e]);
                        x[st + NST / 2][p][e] = rope_hi(lo, hi, sn[e], cs[e]);
                    }
                }
        }
        const float c = rvalid ? a.c : 0.0f;
#pragma unroll
        for (int st = 0; st < NST; ++st)
#pragma unroll
            for (int e = 0; e < 8; ++e) qf[st][e] = (__bf16)(x[st][e >> 2][e & 3] * c);
    }

    f32x16 o[NDB];
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[db][i] = 0.0f;
    f32x16 negm;  // -m of the lane's row, the scores' initial value
#pragma unroll
    for (int i = 0; i < 16; ++i) negm[i] = 0.0f;
    float mu = 0.0f, thr = -INFINITY, l = 0.0f;  // thr: -inf until m is set
    const bf16x2 ones = {(__bf16)1.0f, (__bf16)1.0f};

    const int k_rd = k_base + col * (HD * 2) + ((hf ^ swz<KCH>(col)) << 4);
    int v_rd[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) v_rd[s] = v_base + col * 64 + (((2 * hf + s) ^ swz<4>(col)) << 4);
    auto rd_k = [&](int st, int base) __attribute__((always_inline)) {
        return *reinterpret_cast<const bf16x8*>(lds + (base ^ (st << 5)));
    };
    auto rd_v = [&](int v, int boff) __attribute__((always_inline)) {  // d-block v / 2, contraction half v % 2
        return *reinterpret_cast<const bf16x8*>(lds + v_rd[v & 1] + boff + (v >> 1) * 2048);
    };
    constexpr int AHEAD = 4;  // MFMAs that an LDS operand is read ahead of its own
    constexpr int RING = AHEAD + 1;
    f32x16 s, sn;      // scores of this step's tile and of the next one
    bf16x8 pp[2];      // p of the tile before

    // One step: the softmax of tile u on the VALU, the values of tile u - 1
    // (PREV) and the scores of tile u + 1 (NEXT) on the matrix cores.
    auto step = [&](int u, int kp, auto prev, auto next) __attribute__((always_inline)) {
        constexpr bool PREV = decltype(prev)::value, NEXT = decltype(next)::value;
        constexpr int NPV = 2 * NDB, PV0 = NPV / 2;  // value MFMAs; those before the maximum is known
        // K(u + 1) and V^T(u - 1) have landed; every wave is done with K(u)
        // and V^T(u - 2), whose buffers the DMA below overwrites
        wait_vmcnt<0>();
        lds_barrier();
        const int t = tile_of(u);
        const int kb = k_rd + (kp ^ 1) * TILE_B, vb = (kp ^ 1) * TILE_B;
        const int t2 = min(tile_of(u + 2), t1 - 1), tv = min(t, t1 - 1);
        bf16x8 kf[RING], vf[RING];
        if constexpr (PREV) {
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) vf[i] = rd_v(i, vb);
        }
#pragma unroll
        for (int j = 0; j < DMAW; ++j) dma_v(j, tv, kp);
        // tiles that some row of the wave sees in part (or past the range)
        if (t * BN < fmin || t * BN + BN > fmax || t >= t1) {
            const int k0 = t * BN + 16 * hf - klo;
            const uint32_t n = t < t1 ? (uint32_t)(khi - klo) : 0u;
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = (uint32_t)(k0 + i) < n ? s[i] : -INFINITY;
        }
        __builtin_amdgcn_sched_barrier(0);
        auto pv = [&](int v) __attribute__((always_inline)) {
            if (v + AHEAD < NPV) vf[(v + AHEAD) % RING] = rd_v(v + AHEAD, vb);
            o[v >> 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[v % RING], pp[v & 1], o[v >> 1], 0, 0, 0);
        };
        auto qk = [&](int st) __attribute__((always_inline)) {
            if (st + AHEAD < NST) kf[(st + AHEAD) % RING] = rd_k(st + AHEAD, kb);
            sn = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[st % RING], qf[st], st == 0 ? negm : sn, 0, 0, 0);
        };
        // ---- the row's maximum under half of the value MFMAs
        float mt[5];
#pragma unroll
        for (int v = 0; v < PV0; ++v) {
            if constexpr (PREV) pv(v);
#pragma unroll
            for (int i = 0; i < 5; ++i)
                if (i * PV0 / 5 == v) mt[i] = max3(s[3 * i], s[3 * i + 1], s[3 * i + 2]);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (NEXT) {
#pragma unroll
            for (int i = 0; i < (AHEAD < NST ? AHEAD : NST); ++i) kf[i] = rd_k(i, kb);
        }
        const float mx = max_xor32(max3(max3(mt[0], mt[1], s[15]), max3(mt[2], mt[3], mt[4]), -INFINITY));
        const bool need = mx > thr;
        const bool moved = __builtin_amdgcn_ballot_w64(need) != 0;
        float alpha = 1.0f;
        if (moved) {
            const float delta = need ? mx : 0.0f;
            alpha = need ? (thr > 0.0f ? __builtin_amdgcn_exp2f(-delta) : 0.0f) : 1.0f;
            mu += delta;
            thr = need ? RESCALE_THRESHOLD : thr;
            l *= alpha;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                s[i] -= delta;
                negm[i] -= delta;
            }
        }
        // ---- p = 2^s as bf16 and its sum, under the next scores and the rest
        // of the values: a pair per MFMA or two
        bf16x8 pb[2];
        constexpr int NM = NST + NPV - PV0;  // MFMAs here
#pragma unroll
        for (int k = 0; k < NM; ++k) {
            // (alternating while both last)
            const bool do_pv = k % 3 == 2 && k / 3 < NPV - PV0;
            const int npv = (k + 1) / 3 < NPV - PV0 ? (k + 1) / 3 : NPV - PV0;  // value MFMAs before this one
            if (do_pv) {
                if constexpr (PREV) pv(PV0 + k / 3);
            } else if (k - npv < NST) {
                if constexpr (NEXT) qk(k - npv);
            } else {
                if constexpr (PREV) pv(PV0 + npv + (k - npv - NST));
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                if (j * NM / 8 == k) {
                    const bf16x2 pr = {(__bf16)__builtin_amdgcn_exp2f(s[2 * j]),
                                       (__bf16)__builtin_amdgcn_exp2f(s[2 * j + 1])};
                    pb[j >> 2][(2 * j) & 7] = pr[0];
                    pb[j >> 2][(2 * j + 1) & 7] = pr[1];
                    l = __builtin_amdgcn_fdot2_f32_bf16(pr, ones, l, false);
                }
            }
            if constexpr (NEXT) {
                if (k < DMAW) dma_k(k, t2, kp);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        // (O has the values of tile u - 1, relative to the m before)
        if (moved) {
#pragma unroll
            for (int db = 0; db < NDB; ++db) o[db] *= alpha;
        }
        pp[0] = pb[0];
        pp[1] = pb[1];
        s = sn;
    };

    if (nsteps > 0) {
        wait_vmcnt<0>();
        lds_barrier();
        sn = negm;
#pragma unroll
        for (int st = 0; st < NST; ++st)
            sn = __builtin_amdgcn_mfma_f32_32x32x16_bf16(rd_k(st, k_rd), qf[st], sn, 0, 0, 0);
        s = sn;
        int kp = 0;
        if (nsteps == 1) {
            step(0, kp, std::false_type{}, std::false_type{});
        } else {
            step(0, kp, std::false_type{}, std::true_type{});
            kp ^= 1;
            for (int u = 1; u + 1 < nsteps; ++u, kp ^= 1) step(u, kp, std::true_type{}, std::true_type{});
            step(nsteps - 1, kp, std::true_type{}, std::false_type{});
        }
        // the values of the last tile
        wait_vmcnt<0>();
        lds_barrier();
#pragma unroll
        for (int v = 0; v < 2 * NDB; ++v)
            o[v >> 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(rd_v(v, kp * TILE_B), pp[v & 1], o[v >> 1], 0, 0, 0);
    }

    // ---- key group 1's states to LDS, lane for lane; key group 0 merges
    l += __shfl_xor(l, 32);
    const float m = thr > 0.0f ? mu : -INFINITY;
    f32x4* const mo = reinterpret_cast<f32x4*>(lds) + rb * (NDB * 4 * 64) + lane;
    float* const ml = reinterpret_cast<float*>(lds + RB * NDB * 4 * 64 * 16) + rb * 128 + lane;
    lds_barrier();  // every wave is done with its tiles
    if (kq == 1) {
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                mo[(db * 4 + j) * 64] = f32x4{o[db][4 * j], o[db][4 * j + 1], o[db][4 * j + 2], o[db][4 * j + 3]};
        ml[0] = m;
        ml[64] = l;
    }
    lds_barrier();
    if (kq == 1 || !rvalid) return;
    const float m1 = ml[0], l1 = ml[64];
    const float M = __builtin_fmaxf(m, m1);
    const float w0 = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - M);
    const float w1 = m1 == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m1 - M);
    const float il = __builtin_amdgcn_rcpf(w0 * l + w1 * l1);  // no visible key: 0 * inf = NaN (attention.rs:181-185)
    const float f0 = w0 * il, f1 = w1 * il;
    float* orow = S.out + (size_t)qi * a.o_rstride + (size_t)(g * a.group + hg) * HD + 4 * hf;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const f32x4 y = mo[(db * 4 + j) * 64];
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = o[db][4 * j + e] * f0 + y[e] * f1;
            gstore(orow + 32 * db + 8 * j, v);
        }
}

template <int HD>
hipError_t launch_hd(const LaunchPlan& p, const AttnArgs& a, hipStream_t st) {
    using G = RowsGeom<HD>;
    auto k = attn_rows_kernel<HD>;
    hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)G::LDS_BYTES);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k, dim3(p.n_workgroups), dim3(G::NT), G::LDS_BYTES, st, a);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_rows(const LaunchPlan& p, const AttnArgs& a, hipStream_t st) {
    if (a.hd != p.hd_tile || p.mask == MASK_KEYS || p.n_split != 1) return hipErrorInvalidValue;
    if (a.rope && a.rot != a.hd) return hipErrorInvalidValue;
    if (a.q_bf16 || a.o_bf16) return hipErrorInvalidValue;
    switch (p.hd_tile) {
        case 64: return launch_hd<64>(p, a, st);
        case 128: return launch_hd<128>(p, a, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace dr
