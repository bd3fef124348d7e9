// fh3_attn.hip -- the DiT block's attention branch on gfx950: q/k rmsnorm,
// rope3 and dense online-softmax attention (src/core/fh3_ops.c:410-456,
// 458-505, 587-695; the sequence of src/model/fh3_dit.c:390-411).
//
// Two launches per call:
//   k_attn_prep  fp32 q, k, v rows (any token stride, so q/k/v can be read in
//                place from the qkv projection's output) -> fp16 operands in
//                the layouts the matrix cores read: Qp[h][slot][d] and
//                Kp[h][slot][d] row-major, Vt[h][d][slot] transposed.  Optional
//                per-head rmsnorm of q and k (weights [hd]) and rope3 on their
//                first rot_dim channels are applied on the way; q is scaled by
//                log2(e)/sqrt(hd) so that the softmax runs on exp2.
//   k_attn_fwd   flash-style attention: a workgroup owns 32 queries per
//                wavefront of one head (8 wavefronts for hd 128, 4 for hd 64
//                and for the sparse form), streams 64-key tiles of K and V^T
//                through double-buffered LDS, S^T = K.Q^T and O^T = V^T.P^T on
//                v_mfma_f32_32x32x16_f16 with fp32 accumulation, and keeps the
//                running max / sum in fp32 registers.
//
// Slots beyond n are zero in the prepared operands and masked as keys, so
// any n >= 1 works; the prepared buffers hold n_pad = round_up(n, 32 x wavefronts) slots.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fh3_kernels.h"

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));

constexpr int ATT_KT = 64;   // keys per tile
constexpr int ATT_QW = 32;   // queries per wavefront
constexpr int ATT_NW = 4;    // wavefronts per workgroup of the sparse kernel (two query tiles)
constexpr int ATT_QB = ATT_QW * ATT_NW;
// Dense kernel: with hd = 128, 8 wavefronts (256 queries, 2 per SIMD) share
// each K/V tile in LDS, halving the tile loads and LDS writes per query (+5 %);
// with hd = 64 the 4-wavefront form keeps 3 wavefronts per SIMD and is faster.
constexpr int dense_nw(int hd) { return hd == 128 ? 8 : 4; }
constexpr int ATT_PREP_T = 64;  // slots per prep workgroup
// The softmax offset m of a query is only raised when a tile's maximum
// exceeds it by more than ATT_TAU (log2 units), so p = exp2(s - m) <= 2^8 and
// the rescale of the accumulators is skipped on almost every tile.  Any offset
// gives the same o = sum(p v) / sum(p); fp16 holds p up to 65504.
constexpr float ATT_TAU = 8.0f;

// Order of the keys inside each 16-key block of Vt.  The P^T operand of the
// PV product is taken straight from the S^T accumulator, where lane half hf
// holds keys {4hf..4hf+3, 8+4hf..8+4hf+3} of each 16-key block; storing V^T
// in that order lets one 16-byte LDS read feed the matching A operand:
// position b of a block holds key (b & 3) | (b & 4) << 1 | (b & 8) >> 1.

// Tile pooling (video sparse attention): with a gather map each prep
// workgroup holds exactly one 64-slot tile, so it also writes the tile's
// mean-pooled q, k (and v when vpool is set), pool[h][tile][d] = sum over the
// tile's tokens in order of x * inv[tile], from the final fp32 rows (after
// norm and rope, before the softmax scale) -- the reference's accumulation
// order and roundings (src/core/fh3_vsa.c:224-250).
struct Pool {
    const float *inv;
    const int *cnt;
    float *q, *k, *v;
    int T;
};

// LDS row of the 64 staged rows: eight segments of HD/8 floats, one per thread
// of a row, each padded by four and the row padded again, so that the eight
// lanes of a 16-byte access (a row's segments, or eight neighbours) and the 16
// columns x 4 rows of V's transposed reads spread over the banks.
template <int HD> constexpr int prep_pitch() { return HD + 8 * 4 + 4; }
template <int HD> __device__ __forceinline__ int prep_at(int r, int d) {
    constexpr int DPT = HD / 8;
    return r * prep_pitch<HD>() + (d / DPT) * (DPT + 4) + d % DPT;
}

// sum over the first cnt rows of sx, in row order, times w (thread d < HD):
// sixteen rows' reads at a time ahead of the chain of additions
template <int HD>
__device__ __forceinline__ void pool_rows(const float *sx, int cnt, float w, float *dst) {
    const int d = threadIdx.x;
    if (d < HD) {
        float a = 0.f;
        int r = 0;
        for (; r + 16 <= cnt; r += 16) {
            float b[16];
#pragma unroll
            for (int i = 0; i < 16; i++) b[i] = sx[prep_at<HD>(r + i, d)];
#pragma unroll
            for (int i = 0; i < 16; i++) a = a + b[i] * w;
        }
        for (; r < cnt; r++) a = a + sx[prep_at<HD>(r, d)] * w;
        dst[d] = a;
    }
}

// Lane c of each eight holds chunks 2c and 2c + 1 (half8 o[0], o[1]) of its
// row's 16; afterwards o[0] of the eight lanes are chunks 0..7 and o[1] chunks
// 8..15, so that each store covers 128 consecutive bytes: lane c and lane 7 - c
// exchange one.  at: which chunks the lane then holds.
__device__ __forceinline__ void pair_chunks(half8 (&o)[2], int c, int (&at)[2]) {
    const bool up = c >= 4;
    u32x4 a = __builtin_bit_cast(u32x4, o[0]), b = __builtin_bit_cast(u32x4, o[1]);
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const uint32_t send = up ? a[e] : b[e];
        const uint32_t got = (uint32_t)__builtin_amdgcn_mov_dpp((int)send, 0x141, 0xF, 0xF, true);  // row_half_mirror
        a[e] = up ? got : a[e];
        b[e] = up ? b[e] : got;
    }
    o[0] = __builtin_bit_cast(half8, a), o[1] = __builtin_bit_cast(half8, b);
    at[0] = up ? 15 - 2 * c : 2 * c, at[1] = up ? 2 * c + 1 : 14 - 2 * c;
}

// The work is bound by memory: 12 bytes read and 6 written per element, and the
// rope tables, which for one head are larger than q.  One workgroup takes a tile of
// 64 slots of G consecutive heads: rows are loaded 16 bytes per lane in order, one
// operand ahead of the one in work, and reach the threads (eight to a row,
// HD/8 channels each) through LDS; each thread keeps its channels' table values
// for all q and k of its heads; a rope partner is normalised again from the raw
// row, which takes the place of another pass through LDS.  n = 16384 x 40 heads:
// 570 -> 292 us (5.2 TB/s); with tile pooling, n = 12922 x 56 heads: 746 -> 361 us
// (before: 128-byte runs per lane, one operand at a time, tables for each head).
// ANYROT: rope with rot % 8 != 0, channel by channel with the tables read in place.
template <int HD, bool ANYROT>
__global__ __launch_bounds__(512, 4) void k_attn_prep(const float *__restrict__ q, const float *__restrict__ k,
                                                   const float *__restrict__ v, int64_t ld, int64_t ldv, int n,
                                                   int heads, int G, const int *__restrict__ gather,
                                                   const float *__restrict__ qn_w, const float *__restrict__ kn_w,
                                                   float eps, const float *__restrict__ cosb,
                                                   const float *__restrict__ sinb, int rot, float qscale,
                                                   int n_pad, _Float16 *__restrict__ Qp, _Float16 *__restrict__ Kp,
                                                   _Float16 *__restrict__ Vt, Pool pl) {
    constexpr int DPT = HD / 8, C4 = DPT / 4;
    constexpr int LPR = HD / 4, RPP = 512 / LPR, PASS = ATT_PREP_T / RPP;  // lanes per row, rows per pass, passes
    __shared__ __align__(16) float sx[ATT_PREP_T * prep_pitch<HD>()];
    __shared__ __align__(16) float snw[2][HD];
    const int t = threadIdx.x, c = t & 7, d0 = c * DPT;
    const int tile = blockIdx.x;
    const int h0 = blockIdx.y * G, hn = heads - h0 < G ? heads - h0 : G;
    auto token = [&](int sl) { return gather ? gather[sl] : (sl < n ? sl : -1); };
    const int tok = token(tile * ATT_PREP_T + (t >> 3));
    const int lr = t / LPR, ld0 = (t % LPR) * 4;  // the row and channels this thread loads
    int ltok[PASS];
#pragma unroll
    for (int i = 0; i < PASS; i++) ltok[i] = token(tile * ATT_PREP_T + lr + RPP * i);

    f32x4 nx[PASS];  // the next operand's rows
    auto load = [&](int which, int h) {
        const float *src = (which == 2 ? v : which ? k : q) + (size_t)h * HD + ld0;
        const int64_t l = which == 2 ? ldv : ld;
#pragma unroll
        for (int i = 0; i < PASS; i++) {
            int tk = ltok[i];
            asm volatile("" : "+v"(tk));  // addresses made here, not kept for each operand through the loops
            nx[i] = tk >= 0 ? *(const f32x4 *)(src + tk * l) : f32x4{};
        }
    };
    load(0, h0);
    if (t < HD) {
        snw[0][t] = qn_w ? qn_w[t] : 1.f;
        snw[1][t] = kn_w ? kn_w[t] : 1.f;
    }
    const bool rope4 = !ANYROT && cosb;  // rot % 8 == 0: 4-channel chunks never straddle half or rot
    f32x4 ct[C4], st[C4];
#pragma unroll
    for (int i = 0; i < C4; i++) {
        ct[i] = st[i] = f32x4{};
        if (rope4 && tok >= 0 && d0 + 4 * i < rot) {
            ct[i] = *(const f32x4 *)(cosb + (size_t)tok * rot + d0 + 4 * i);
            st[i] = *(const f32x4 *)(sinb + (size_t)tok * rot + d0 + 4 * i);
        }
    }

    for (int hi = 0; hi < hn; hi++) {
        const int h = h0 + hi;
#pragma unroll 1
        for (int which = 0; which < 3; which++) {
            __syncthreads();  // the last operand's readers are done
#pragma unroll
            for (int i = 0; i < PASS; i++) *(f32x4 *)&sx[prep_at<HD>(lr + RPP * i, ld0)] = nx[i];
            if (which < 2)
                load(which + 1, h);
            else if (hi + 1 < hn)
                load(0, h + 1);
            __syncthreads();
            if (which == 2) break;
            int r = t >> 3, half = rot >> 1;
            asm volatile("" : "+v"(r), "+s"(half));  // as in load()
            const bool norm = (which ? kn_w : qn_w) != nullptr;
            const float *nw = snw[which];
            float x[DPT];
#pragma unroll
            for (int i = 0; i < C4; i++) {
                const f32x4 u = *(const f32x4 *)&sx[prep_at<HD>(r, d0) + 4 * i];
                x[4 * i] = u[0], x[4 * i + 1] = u[1], x[4 * i + 2] = u[2], x[4 * i + 3] = u[3];
            }
            float inv = 1.f;
            if (norm) {
                // four chains of HD/4 channels: the odd thread of a pair goes on from the even one's sum
                float ss = 0.f;
#pragma unroll
                for (int i = 0; i < DPT; i++) ss = fmaf(x[i], x[i], ss);
                ss = __shfl_xor(ss, 1);
#pragma unroll
                for (int i = 0; i < DPT; i++) ss = fmaf(x[i], x[i], ss);
                ss = __shfl(ss, (t & 63) | 1);
                ss += __shfl_xor(ss, 2);
                ss += __shfl_xor(ss, 4);
                inv = tok >= 0 ? 1.0f / sqrtf(ss / (float)HD + eps) : 0.f;
#pragma unroll
                for (int i = 0; i < C4; i++) {
                    const f32x4 w = *(const f32x4 *)&nw[d0 + 4 * i];
#pragma unroll
                    for (int e = 0; e < 4; e++) x[4 * i + e] = x[4 * i + e] * inv * w[e];
                }
            }
            if (rope4) {
                if (tok >= 0) {
#pragma unroll
                    for (int i = 0; i < C4; i++) {
                        const int d = d0 + 4 * i;
                        if (d < rot) {
                            const bool lo = d < half;
                            const int pd = lo ? d + half : d - half;
                            f32x4 pv = *(const f32x4 *)&sx[prep_at<HD>(r, pd)];
                            if (norm) {
                                const f32x4 w = *(const f32x4 *)&nw[pd];
#pragma unroll
                                for (int e = 0; e < 4; e++) pv[e] = pv[e] * inv * w[e];
                            }
#pragma unroll
                            for (int e = 0; e < 4; e++) {
                                const float a = x[4 * i + e] * ct[i][e], b = pv[e] * st[i][e];
                                x[4 * i + e] = lo ? a - b : a + b;
                            }
                        }
                    }
                }
            } else if (ANYROT && tok >= 0) {
                const float *cr = cosb + (size_t)tok * rot, *sr = sinb + (size_t)tok * rot;
                // rot through an empty asm: otherwise the per-element region
                // tests are hoisted out of the loops and their 64-bit lane
                // masks, two per element, overflow the scalar registers
                int rv = rot;
                asm volatile("" : "+s"(rv));
                const int hv = rv >> 1;
#pragma unroll
                for (int i = 0; i < DPT; i++) {
                    const int d = d0 + i;
                    if (d < rv) {
                        const bool lo = d < hv;
                        const int pd = lo ? d + hv : d - hv;
                        float pv = sx[prep_at<HD>(r, pd)];
                        if (norm) pv = pv * inv * nw[pd];
                        const float a = x[i] * cr[d], b = pv * sr[d];
                        x[i] = lo ? a - b : a + b;
                    }
                }
            }
            if (pl.q && tile < pl.T) {  // uniform over the workgroup
                __syncthreads();
#pragma unroll
                for (int i = 0; i < C4; i++)
                    *(f32x4 *)&sx[prep_at<HD>(r, d0) + 4 * i] =
                        f32x4{x[4 * i], x[4 * i + 1], x[4 * i + 2], x[4 * i + 3]};
                __syncthreads();
                pool_rows<HD>(sx, pl.cnt[tile], pl.inv[tile], (which ? pl.k : pl.q) + ((size_t)h * pl.T + tile) * HD);
            }
            const float sc = which ? 1.f : qscale;
            half8 o[DPT / 8];
#pragma unroll
            for (int i = 0; i < DPT; i++) o[i / 8][i % 8] = (_Float16)(x[i] * sc);
            half8 *dst = (half8 *)((which ? Kp : Qp) + ((size_t)h * n_pad + tile * ATT_PREP_T + r) * HD);
            if constexpr (HD == 128) {
                int at[2];
                pair_chunks(o, c, at);
                dst[at[0]] = o[0], dst[at[1]] = o[1];
            } else {
                dst[c] = o[0];
            }
        }
        // v: written transposed in the order above, four lanes to 64 bytes of a channel's row
        if (pl.v && tile < pl.T)
            pool_rows<HD>(sx, pl.cnt[tile], pl.inv[tile], pl.v + ((size_t)h * pl.T + tile) * HD);
        int tv = t;
        asm volatile("" : "+v"(tv));  // as in load()
#pragma unroll
        for (int i = 0; i < HD / 64; i++) {
            const int id = tv + 512 * i, d = (id >> 2) % HD, j = id & 3, half_tile = id / (4 * HD);
            // slots 32 half_tile + 8 j + e hold the keys that order names: row + (e % 4) + 2 (e & 4)
            const int row = 32 * half_tile + 16 * (j >> 1) + 4 * (j & 1);
            half8 o;
#pragma unroll
            for (int e = 0; e < 8; e++) o[e] = (_Float16)sx[prep_at<HD>(row + (e & 3) + 2 * (e & 4), d)];
            *(half8 *)(Vt + ((size_t)h * HD + d) * n_pad + (size_t)tile * ATT_PREP_T + 32 * half_tile + 8 * j) = o;
        }
    }
}

// Heads per workgroup: up to four share a tile's table values while 2048
// workgroups remain (eight to a CU).  n = 16384 x 40 heads: one 370, four 297,
// eight 305 us; n = 1500 x 40, where it is one: 26.9, no faster with more.
int prep_heads(int tiles, int heads) {
    const int64_t g = (int64_t)tiles * heads / 2048;
    return g < 1 ? 1 : g > 4 ? 4 : (int)g;
}

__device__ __forceinline__ float wave_swap_max(float x) { return fmaxf(x, __shfl_xor(x, 32)); }

// Block-sparse mode (video sparse attention).  Slots are tile-ordered: tile i
// owns slots 64 i .. 64 i + cnt[i] - 1 and gather[slot] names the token there
// (-1 for the empty rest of the tile).  The workgroup of query block qb holds
// query tiles 2 qb (wavefronts 0, 1) and 2 qb + 1 (wavefronts 2, 3); it walks
// the union of their selected key tiles, lists[(h * nqb + qb) * T + e] =
// key tile | (bit 14: tile 2 qb selects it) | (bit 15: tile 2 qb + 1 does),
// e < list_len[h * nqb + qb], and each pair of wavefronts skips the tiles its
// query tile did not select.  The output row of a slot goes to its token,
// plus coarse[h][tile][d] * gate[token][h][d] when a gate is given.
struct Sparse {
    const uint16_t *lists;
    const int *list_len;
    const int *cnt;
    const int *gather;
    const float *coarse;
    const float *gate;
    int T;
};

// (the second launch bound is the minimum number of wavefronts per SIMD: two)
template <int HD, bool SPARSE, int NW>
__global__ __launch_bounds__(64 * NW, 2) void k_attn_fwd(const _Float16 *__restrict__ Qp,
                                                     const _Float16 *__restrict__ Kp,
                                                     const _Float16 *__restrict__ Vt, int n, int n_pad,
                                                     int heads, float *__restrict__ O, int64_t o_ld, Sparse sp) {
    constexpr int KS = HD / 16;            // 16-wide steps of the S product
    constexpr int DB = HD / 32;            // 32-row blocks of O^T
    constexpr int KROW = HD + 8;           // LDS row of K (halfs), padded against bank conflicts
    constexpr int VROW = ATT_KT + 8;       // LDS row of V^T (halfs)
    constexpr int NT = 64 * NW;
    constexpr int QB = ATT_QW * NW;
    constexpr int KCH = ATT_KT * HD / 8 / NT;  // 16-byte chunks per thread per tile, K and V each
    __shared__ _Float16 sk[2][ATT_KT][KROW];
    __shared__ _Float16 sv[2][HD][VROW];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, hf = lane >> 5;

    // XCD-aware order: consecutive workgroup ids land on different XCDs, so
    // give each XCD a contiguous run of (head, query block) pairs
    const int nqb = n_pad / QB;
    const int total = heads * nqb;
    const int id = blockIdx.x;
    const int per = total >> 3;
    const int L = (id < per * 8) ? (id & 7) * per + (id >> 3) : id;
    const int h = L / nqb, qb = L - h * nqb;
    const int q0 = qb * QB + wave * ATT_QW;

    const _Float16 *kh = Kp + (size_t)h * n_pad * HD;
    const _Float16 *vh = Vt + (size_t)h * HD * n_pad;

    // Q^T fragments (B operand): lane holds query q0 + l32, d = 16 kk + 8 hf ..
    half8 qf[KS];
    {
        const half8 *qp = (const half8 *)(Qp + ((size_t)h * n_pad + q0 + l32) * HD + 8 * hf);
#pragma unroll
        for (int kk = 0; kk < KS; kk++) qf[kk] = qp[2 * kk];
        // Wait for them here: left to the loop, their waits stand among each
        // tile's products and drain the next tile's loads as well.
#pragma unroll
        for (int kk = 0; kk < KS; kk++) asm volatile("" : "+v"(qf[kk]));
    }

    // key tiles to visit: 0 .. nkt-1 (dense) or the block's list (sparse)
    const uint16_t *lst = nullptr;
    int nkt = (n + ATT_KT - 1) / ATT_KT;
    if (SPARSE) {
        lst = sp.lists + (size_t)L * sp.T;
        nkt = sp.list_len[L];
    }
    // Sparse: 64 list entries at a time and their tiles' token counts, one per
    // lane, read from there as scalars (loaded when used, an entry and a count
    // cost each tile two memory latencies, and their waits drained the tile loads)
    uint32_t ents = 0;
    int cnts = 0;
    auto load_entries = [&](int e) {
        const int i = e + lane < nkt ? e + lane : nkt - 1;
        ents = lst[i];
        cnts = sp.cnt[ents & 0x3FFF];
    };
    // entry e: a sparse list's entry or the key tile, and its number of keys
    auto entry = [&](int e, int &ent, int &keys) {
        if (SPARSE) {
            if ((e & 63) == 0) load_entries(e);
            ent = __builtin_amdgcn_readlane((int)ents, e & 63);
            keys = __builtin_amdgcn_readlane(cnts, e & 63);
        } else {
            ent = e;
            keys = n - e * ATT_KT;
        }
    };

    half8 rk[KCH], rv[KCH];
    auto load_tile = [&](int j) {
#pragma unroll
        for (int i = 0; i < KCH; i++) {
            const int c = tid + i * NT;
            const int kr = c / (HD / 8), kc = c % (HD / 8);
            rk[i] = *(const half8 *)(kh + (size_t)(j * ATT_KT + kr) * HD + kc * 8);
            const int vr = c / (ATT_KT / 8), vc = c % (ATT_KT / 8);
            rv[i] = *(const half8 *)(vh + (size_t)vr * n_pad + j * ATT_KT + vc * 8);
        }
    };
    auto store_tile = [&](int b) {
#pragma unroll
        for (int i = 0; i < KCH; i++) {
            const int c = tid + i * NT;
            const int kr = c / (HD / 8), kc = c % (HD / 8);
            *(half8 *)&sk[b][kr][kc * 8] = rk[i];
            const int vr = c / (ATT_KT / 8), vc = c % (ATT_KT / 8);
            *(half8 *)&sv[b][vr][vc * 8] = rv[i];
        }
    };

    f32x16 o[DB];
#pragma unroll
    for (int i = 0; i < DB; i++) o[i] = f32x16{};
    f32x16 nm = {};     // minus the query's softmax offset, as an accumulator to start from
    float lsum = 0.f;
    float thr = -INFINITY;  // before the first tile: its maximum becomes the offset, whatever it is

    int ent = 0, kv = 0;  // kv: keys in the tile (>= 1)
    if (nkt > 0) {
        entry(0, ent, kv);
        load_tile(SPARSE ? ent & 0x3FFF : ent);
        store_tile(0);
    }
    __syncthreads();
    for (int e = 0; e < nkt; e++) {
        const int b = e & 1;
        int ent_n = 0, kv_n = 0;
        if (e + 1 < nkt) {
            entry(e + 1, ent_n, kv_n);
            load_tile(SPARSE ? ent_n & 0x3FFF : ent_n);
        }
        // sparse: whether this pair of wavefronts' query tile selected it (wave-uniform)
        const bool active = SPARSE ? ((ent >> (14 + (wave >> 1))) & 1) != 0 : true;
        if (active) {
            // dense: raised wave priority through the tile's matrix and softmax
            // work (the other wavefront on the SIMD is then mostly loading or
            // waiting; +1-2 %; the sparse walk loses with it)
            if constexpr (!SPARSE) __builtin_amdgcn_s_setprio(2);
            // S^T[key][query] - m for the 64 keys: two 32-key accumulators that
            // start at -m, so that the softmax needs no subtraction
            f32x16 s[2] = {nm, nm};
#pragma unroll
            for (int kk = 0; kk < KS; kk++) {
#pragma unroll
                for (int st = 0; st < 2; st++) {
                    const half8 a = *(const half8 *)&sk[b][32 * st + l32][16 * kk + 8 * hf];
                    s[st] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qf[kk], s[st], 0, 0, 0);
                }
            }
            // lane holds keys 32 st + 8 (v/4) + 4 hf + v%4 of query q0 + l32
            if (kv < ATT_KT) {
                const int kh = kv - 4 * hf;
#pragma unroll
                for (int st = 0; st < 2; st++)
#pragma unroll
                    for (int v = 0; v < 16; v++) s[st][v] = kh > 32 * st + 8 * (v >> 2) + (v & 3) ? s[st][v] : -INFINITY;
            }
            float mt = s[0][0];
#pragma unroll
            for (int v = 1; v < 16; v++) mt = fmaxf(mt, s[0][v]);
#pragma unroll
            for (int v = 0; v < 16; v++) mt = fmaxf(mt, s[1][v]);
            // Only where some lane's own maximum asks for it do the two halves
            // of a query compare theirs (wave-uniform).
            if (__ballot(mt > thr)) {
                mt = wave_swap_max(mt);
                const float up = mt > thr ? mt : 0.f;
                const float alpha = thr < 0.f ? 0.f : __builtin_amdgcn_exp2f(-up);
#pragma unroll
                for (int v = 0; v < 16; v++) nm[v] -= up;
                thr = ATT_TAU;
                lsum *= alpha;
#pragma unroll
                for (int i = 0; i < DB; i++) o[i] *= alpha;
#pragma unroll
                for (int st = 0; st < 2; st++)
#pragma unroll
                    for (int v = 0; v < 16; v++) s[st][v] -= up;
            }
#pragma unroll
            for (int st = 0; st < 2; st++)
#pragma unroll
                for (int v = 0; v < 16; v++) s[st][v] = __builtin_amdgcn_exp2f(s[st][v]);

            // P^T fragments: 16-key step t = values 4g..4g+7 of accumulator
            // t/2, g = 2 (t % 2); they pair with V^T stored in the order
            // given above.  The row sum is taken over the same fp16 values the
            // product uses.
            half8 pf[4];
            float ps[2] = {0.f, 0.f};
#pragma unroll
            for (int tt = 0; tt < 4; tt++) {
                uint32_t w[4];
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    w[q] = __builtin_bit_cast(uint32_t, half2v{(_Float16)s[tt >> 1][8 * (tt & 1) + 2 * q],
                                                               (_Float16)s[tt >> 1][8 * (tt & 1) + 2 * q + 1]});
                    asm("" : "+v"(w[q]));  // one pair, not converted once for each use
                    ps[q & 1] = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2v, w[q]), half2v{1, 1}, ps[q & 1], false);
                }
                pf[tt] = __builtin_bit_cast(half8, u32x4{w[0], w[1], w[2], w[3]});
            }
            lsum += ps[0] + ps[1];
#pragma unroll
            for (int db = 0; db < DB; db++) {
#pragma unroll
                for (int tt = 0; tt < 4; tt++) {
                    const half8 a = *(const half8 *)&sv[b][32 * db + l32][16 * tt + 8 * hf];
                    o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, pf[tt], o[db], 0, 0, 0);
                }
            }
        }
        if constexpr (!SPARSE) __builtin_amdgcn_s_setprio(0);
        if (e + 1 < nkt) store_tile(b ^ 1);
        ent = ent_n;
        kv = kv_n;
        __syncthreads();
    }

    const float l = lsum + __shfl_xor(lsum, 32);
    const float inv = 1.0f / l;
    const int slot = q0 + l32;
    int row = slot < n ? slot : -1;
    int tile = 0;
    if (SPARSE) {
        tile = slot / ATT_KT;
        row = (tile < sp.T && slot - tile * ATT_KT < sp.cnt[tile]) ? sp.gather[slot] : -1;
    }
    if (row >= 0) {
        float *orow = O + (size_t)row * o_ld + (size_t)h * HD;
        const float *crow = SPARSE && sp.coarse ? sp.coarse + ((size_t)h * sp.T + tile) * HD : nullptr;
        const float *grow_ = crow ? sp.gate + (size_t)row * o_ld + (size_t)h * HD : nullptr;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int d = 32 * db + 8 * g + 4 * hf;
                f32x4 w;
#pragma unroll
                for (int q = 0; q < 4; q++) w[q] = o[db][4 * g + q] * inv;
                if (crow) {
                    const f32x4 cv = *(const f32x4 *)(crow + d), gv = *(const f32x4 *)(grow_ + d);
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const float t = cv[q] * gv[q];
                        w[q] = w[q] + t;
                    }
                }
                *(f32x4 *)(orow + d) = w;
            }
    }
}


// ---------------------------------------------------------------------------
// Video sparse attention (src/core/fh3_vsa.c:186-507).  The tile statistics
// are computed in the reference's exact order and roundings (one thread per
// output, products and sums rounded separately), so the tile scores -- and
// with them the top-k tile choice -- are bit-identical to the CPU's; the fine
// attention then runs on k_attn_fwd over each query tile's selected tiles.
// ---------------------------------------------------------------------------

// scores[h][i][j] = (sum_d qp[h][i][d] * kp[h][j][d], in order) * scale
// TS x TS tiles from LDS, TS/16 x TS/16 of them to a thread (rows and columns 16
// apart: the eight lanes of a 16-byte LDS read then start on different banks).
// TS = 64 is bound by the separate products and sums; 245 tiles x 56 heads: 194 ->
// 36 us (before: every dot product read its whole key row from memory).  With few
// tiles it takes as long as one such tile, 12 us: 16 x 16 ones then (1 tile x 16
// heads 3.3 us, 100 x 16 5.7 against 13.4; 245 x 56 38.6 against 35.8).
template <int HD, int TS>
__global__ __launch_bounds__(256) void k_vsa_scores(const float *__restrict__ qp, const float *__restrict__ kp,
                                                    int T, float scale, float *__restrict__ sc) {
    constexpr int X = TS / 16;
    __shared__ __align__(16) float sq[TS][HD + 4], sk[TS][HD + 4];
    const int i0 = blockIdx.y * TS, j0 = blockIdx.x * TS, h = blockIdx.z, t = threadIdx.x;
    for (int c = t; c < TS * HD / 4; c += 256) {
        const int r = c / (HD / 4), d = 4 * (c % (HD / 4));
        const int i = i0 + r < T ? i0 + r : T - 1, j = j0 + r < T ? j0 + r : T - 1;
        *(f32x4 *)&sq[r][d] = *(const f32x4 *)(qp + ((size_t)h * T + i) * HD + d);
        *(f32x4 *)&sk[r][d] = *(const f32x4 *)(kp + ((size_t)h * T + j) * HD + d);
    }
    __syncthreads();
    const int ti = t >> 4, tj = t & 15;
    float dot[X][X] = {};
#pragma unroll 4
    for (int d = 0; d < HD; d += 4) {
        f32x4 a[X], b[X];
#pragma unroll
        for (int x = 0; x < X; x++) {
            a[x] = *(const f32x4 *)&sq[ti + 16 * x][d];
            b[x] = *(const f32x4 *)&sk[tj + 16 * x][d];
        }
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int x = 0; x < X; x++)
#pragma unroll
                for (int y = 0; y < X; y++) dot[x][y] = dot[x][y] + a[x][e] * b[y][e];
    }
#pragma unroll
    for (int x = 0; x < X; x++)
#pragma unroll
        for (int y = 0; y < X; y++) {
            const int i = i0 + ti + 16 * x, j = j0 + tj + 16 * y;
            if (i < T && j < T) sc[((size_t)h * T + i) * T + j] = dot[x][y] * scale;
        }
}

// The selection of one query tile by one wavefront, as bits m[e] of the key
// tiles 64 e + lane: every tile for prefix query tiles or when all are kept;
// otherwise the prefix tiles and the kv video tiles of largest score, ties to
// the lower tile index (the order of the reference's qsort comparator,
// src/core/fh3_vsa.c:178-184).  The scores become order-preserving keys, held in
// registers; the kv-th largest is built bit by bit, each bit kept where at least
// kv keys reach it.
template <int R>
__device__ __forceinline__ void vsa_select_row(const float *__restrict__ srow, int T, int P, int kv, bool all,
                                               uint64_t (&m)[R]) {
    const int lane = threadIdx.x & 63;
    uint32_t key[R];
#pragma unroll
    for (int e = 0; e < R; e++) {
        const int j = 64 * e + lane;
        m[e] = __ballot(j < T && (all || j < P));
        key[e] = 0;  // below every threshold tried
        if (!all && j >= P && j < T) {
            float f = srow[j];
            f = f == 0.f ? 0.f : f;  // -0 ties with +0, as in the comparator
            const uint32_t u = __float_as_uint(f);
            key[e] = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
        }
    }
    if (all) return;
    uint32_t thr = 0;
    for (int bit = 31; bit >= 0; bit--) {
        const uint32_t cand = thr | (1u << bit);
        int cnt = 0;
#pragma unroll
        for (int e = 0; e < R; e++) cnt += (int)__popcll(__ballot(key[e] >= cand));
        if (cnt >= kv) thr = cand;
    }
    int want = kv;  // how many of the keys equal to the threshold are in
#pragma unroll
    for (int e = 0; e < R; e++) want -= (int)__popcll(__ballot(key[e] > thr));
#pragma unroll
    for (int e = 0; e < R; e++) {
        const int j = 64 * e + lane;
        const uint64_t eq = __ballot(j >= P && j < T && key[e] == thr);
        const bool in = key[e] > thr || (((eq >> lane) & 1) && (int)__popcll(eq & ((1ull << lane) - 1)) < want);
        m[e] |= __ballot(in);
        want -= (int)__popcll(eq);
    }
}

// Union tile lists of query-tile pairs (2 qb, 2 qb + 1) for k_attn_fwd: a
// wavefront selects for each of the two, the first writes the list in tile
// order.  T <= 64 R.  245 tiles x 56 heads: 229 -> 16 us (before: a radix select
// over LDS histograms that one thread scanned).
template <int R>
__global__ __launch_bounds__(128) void k_vsa_lists(const float *__restrict__ sc, int T, int P, int kv, int all,
                                                   int nqb, uint16_t *__restrict__ lists,
                                                   int *__restrict__ list_len) {
    __shared__ uint64_t sel1[R];
    const int qb = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = 2 * qb + wave;
    uint64_t m[R] = {};
    if (i < T) vsa_select_row<R>(sc + ((size_t)h * T + i) * T, T, P, kv, all != 0 || i < P, m);
    if (wave == 1 && lane == 0) {
#pragma unroll
        for (int e = 0; e < R; e++) sel1[e] = m[e];
    }
    __syncthreads();
    if (wave == 1) return;
    uint16_t *out = lists + ((size_t)h * nqb + qb) * T;
    int at = 0;
#pragma unroll
    for (int e = 0; e < R; e++) {
        const uint64_t b = sel1[e], u = m[e] | b;
        const int bits = (int)((m[e] >> lane) & 1) | (int)((b >> lane) & 1) << 1;
        if (bits) out[at + __popcll(u & ((1ull << lane) - 1))] = (uint16_t)((64 * e + lane) | (bits << 14));
        at += __popcll(u);
    }
    if (lane == 0) list_len[h * nqb + qb] = at;
}

// Gated coarse branch: per (query tile i, head h) a softmax over all tile
// scores mixes the pooled v: coarse[h][i][d] = sum_j expf(s_j - max) / sum * vp[h][j][d].
// A workgroup takes RB query tiles, so that each pooled v is read once for all of
// them; bound by the latency of those reads, hence the unrolling.  245 tiles x 56
// heads: one query tile (4 reads ahead) 84, eight 45, eight with 8 reads ahead 38
// us.  Few workgroups or more than 32 KB of weights are better off with one query
// tile and 16 reads ahead: 245 x 1 10.3 us (eight 29.5), 245 x 16 23.4 (31.0), 4096 x 4
// 1326 (two 2931).
template <int HD, int RB>
__global__ __launch_bounds__(HD) void k_vsa_coarse(const float *__restrict__ sc, const float *__restrict__ vp,
                                                   int T, float *__restrict__ coarse) {
    extern __shared__ __align__(16) float wsh[];  // [T][RB] softmax weights
    __shared__ float red[RB][HD / 64];
    const int i0 = blockIdx.x * RB, h = blockIdx.y, d = threadIdx.x, lane = d & 63, wave = d >> 6;
    const float *srow[RB];
    float mx[RB], sum[RB], acc[RB];
#pragma unroll
    for (int x = 0; x < RB; x++) {
        srow[x] = sc + ((size_t)h * T + (i0 + x < T ? i0 + x : T - 1)) * T;
        mx[x] = -1e30f;
        sum[x] = acc[x] = 0.f;
    }
    for (int j = d; j < T; j += HD)
#pragma unroll
        for (int x = 0; x < RB; x++) mx[x] = fmaxf(mx[x], srow[x][j]);
#pragma unroll
    for (int x = 0; x < RB; x++) {
        for (int o = 32; o > 0; o >>= 1) mx[x] = fmaxf(mx[x], __shfl_xor(mx[x], o));
        if (lane == 0) red[x][wave] = mx[x];
    }
    __syncthreads();
#pragma unroll
    for (int x = 0; x < RB; x++) {
        mx[x] = red[x][0];
        for (int w = 1; w < HD / 64; w++) mx[x] = fmaxf(mx[x], red[x][w]);
    }
    for (int j = d; j < T; j += HD)
#pragma unroll
        for (int x = 0; x < RB; x++) {
            const float w = expf(srow[x][j] - mx[x]);
            wsh[j * RB + x] = w;
            sum[x] += w;
        }
    __syncthreads();  // red is read
#pragma unroll
    for (int x = 0; x < RB; x++) {
        for (int o = 32; o > 0; o >>= 1) sum[x] += __shfl_xor(sum[x], o);
        if (lane == 0) red[x][wave] = sum[x];
    }
    __syncthreads();
#pragma unroll
    for (int x = 0; x < RB; x++) {
        sum[x] = 0.f;
        for (int w = 0; w < HD / 64; w++) sum[x] += red[x][w];
        sum[x] = 1.0f / sum[x];
    }
    for (int j = d; j < T; j += HD)
#pragma unroll
        for (int x = 0; x < RB; x++) wsh[j * RB + x] = wsh[j * RB + x] * sum[x];
    __syncthreads();
    const float *vcol = vp + (size_t)h * T * HD + d;
    constexpr int AHEAD = RB == 1 ? 16 : 8;
#pragma unroll AHEAD
    for (int j = 0; j < T; j++) {
        const float v = vcol[(size_t)j * HD];
#pragma unroll
        for (int x = 0; x < RB; x++) acc[x] += wsh[j * RB + x] * v;
    }
#pragma unroll
    for (int x = 0; x < RB; x++)
        if (i0 + x < T) coarse[((size_t)h * T + i0 + x) * HD + d] = acc[x];
}

int64_t attn_pad_dense(int n, int hd) {
    const int64_t qb = ATT_QW * dense_nw(hd);
    return ((int64_t)n + qb - 1) / qb * qb;
}

template <int HD>
hipError_t attn_launch(const float *q, const float *k, const float *v, int64_t ld, int n, int heads,
                       const float *qn_w, const float *kn_w, float eps, const float *cosb, const float *sinb,
                       int rot, void *ws, float *o, int64_t o_ld, hipStream_t st) {
    const int n_pad = (int)attn_pad_dense(n, HD);
    _Float16 *Qp = (_Float16 *)ws;
    _Float16 *Kp = Qp + (size_t)heads * n_pad * HD;
    _Float16 *Vt = Kp + (size_t)heads * n_pad * HD;
    const float qscale = 1.4426950408889634f / sqrtf((float)HD);
    const int G = prep_heads(n_pad / ATT_PREP_T, heads);
    hipLaunchKernelGGL((cosb && rot % 8 ? k_attn_prep<HD, true> : k_attn_prep<HD, false>),
                       dim3(n_pad / ATT_PREP_T, (heads + G - 1) / G), dim3(512), 0, st, q, k, v, ld, ld, n, heads, G, (const int *)nullptr, qn_w, kn_w, eps, cosb, sinb, rot, qscale, n_pad, Qp, Kp, Vt, Pool{});
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    constexpr int NW = dense_nw(HD);
    const int blocks = heads * (n_pad / (ATT_QW * NW));
    hipLaunchKernelGGL((k_attn_fwd<HD, false, NW>), dim3(blocks), dim3(64 * NW), 0, st, Qp, Kp, Vt, n, n_pad, heads, o,
                       o_ld, Sparse{});
    return hipGetLastError();
}

}  // namespace

extern "C" int64_t fh3k_attn_pad(int n) { return ((int64_t)n + ATT_QB - 1) / ATT_QB * ATT_QB; }

extern "C" size_t fh3k_attn_ws_bytes(int n, int heads, int hd) {
    return (size_t)3 * heads * attn_pad_dense(n, hd) * hd * sizeof(_Float16);
}

extern "C" int fh3k_attn_head_dim_ok(int hd) { return hd == 64 || hd == 128; }

extern "C" hipError_t fh3k_attention(const float *q, const float *k, const float *v, int64_t ld, int n, int heads,
                                     int hd, const float *qn_w, const float *kn_w, float eps, const float *cosb,
                                     const float *sinb, int rot, void *ws, float *o, int64_t o_ld, hipStream_t st) {
    if (hd == 128) return attn_launch<128>(q, k, v, ld, n, heads, qn_w, kn_w, eps, cosb, sinb, rot, ws, o, o_ld, st);
    if (hd == 64) return attn_launch<64>(q, k, v, ld, n, heads, qn_w, kn_w, eps, cosb, sinb, rot, ws, o, o_ld, st);
    return hipErrorInvalidValue;
}

// ---------------------------------------------------------------------------
// Video sparse attention launchers
// ---------------------------------------------------------------------------
namespace {

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

struct VsaWs {
    _Float16 *Qp, *Kp, *Vt;
    float *qp, *kp, *vp, *sc, *coarse;
    uint16_t *lists;
    int *list_len;
    size_t bytes;
};

VsaWs vsa_ws(void *base, int T, int heads, int hd) {
    const int64_t n_pad = fh3k_attn_pad(ATT_KT * T);
    const int64_t nqb = n_pad / ATT_QB;
    char *p = (char *)base;
    VsaWs w;
    size_t at = 0;
    auto take = [&](size_t b) {
        char *r = p ? p + at : nullptr;
        at += align256(b);
        return r;
    };
    const size_t op = (size_t)heads * n_pad * hd * sizeof(_Float16);
    w.Qp = (_Float16 *)take(op);
    w.Kp = (_Float16 *)take(op);
    w.Vt = (_Float16 *)take(op);
    const size_t pool = (size_t)heads * T * hd * sizeof(float);
    w.qp = (float *)take(pool);
    w.kp = (float *)take(pool);
    w.vp = (float *)take(pool);
    w.coarse = (float *)take(pool);
    w.sc = (float *)take((size_t)heads * T * T * sizeof(float));
    w.lists = (uint16_t *)take((size_t)heads * nqb * T * sizeof(uint16_t));
    w.list_len = (int *)take((size_t)heads * nqb * sizeof(int));
    w.bytes = at;
    return w;
}

template <int HD>
hipError_t vsa_launch(const float *q, const float *k, const float *v, int64_t ld, int64_t ldv, const float *qn_w,
                      const float *kn_w, float eps, const float *cosb, const float *sinb, int rot, const float *gate,
                      float *o, int64_t o_ld, int heads, const float *inv, const int *gather, const int *cnt, int T,
                      int P, int kv, int all, float scale, void *ws, hipStream_t st) {
    const int n_pad = (int)fh3k_attn_pad(ATT_KT * T);
    const int nqb = n_pad / ATT_QB;
    VsaWs w = vsa_ws(ws, T, heads, HD);
    const float qscale = 1.4426950408889634f / sqrtf((float)HD);
    Pool pl{inv, cnt, w.qp, w.kp, gate ? w.vp : nullptr, T};
    const int G = prep_heads(n_pad / ATT_PREP_T, heads);
    hipLaunchKernelGGL((cosb && rot % 8 ? k_attn_prep<HD, true> : k_attn_prep<HD, false>),
                       dim3(n_pad / ATT_PREP_T, (heads + G - 1) / G), dim3(512), 0, st, q, k, v, ld, ldv, ATT_KT * T,
                       heads, G, gather, qn_w, kn_w, eps, cosb, sinb, rot, qscale, n_pad, w.Qp, w.Kp, w.Vt, pl);
    // 16 x 16 score tiles while 64 x 64 ones would leave CUs without any
    const int t64 = (T + 63) / 64, t16 = (T + 15) / 16;
    if ((int64_t)t64 * t64 * heads < 256)
        hipLaunchKernelGGL((k_vsa_scores<HD, 16>), dim3(t16, t16, heads), dim3(256), 0, st, w.qp, w.kp, T, scale, w.sc);
    else
        hipLaunchKernelGGL((k_vsa_scores<HD, 64>), dim3(t64, t64, heads), dim3(256), 0, st, w.qp, w.kp, T, scale, w.sc);
    hipLaunchKernelGGL((T <= 256 ? k_vsa_lists<4> : T <= 1024 ? k_vsa_lists<16> : k_vsa_lists<64>), dim3(nqb, heads),
                       dim3(128), 0, st, w.sc, T, P, kv, all, nqb, w.lists, w.list_len);
    if (gate) {
        // eight query tiles to a workgroup while that leaves three of them to a CU and their weights take at
        // most 32 KB of LDS
        const int rb = T <= 1024 && (int64_t)((T + 7) / 8) * heads >= 768 ? 8 : 1;
        hipLaunchKernelGGL((rb == 8 ? k_vsa_coarse<HD, 8> : k_vsa_coarse<HD, 1>), dim3((T + rb - 1) / rb, heads),
                           dim3(HD), (size_t)T * rb * sizeof(float), st, w.sc, w.vp, T, w.coarse);
    }
    Sparse sp{w.lists, w.list_len, cnt, gather, gate ? w.coarse : nullptr, gate, T};
    hipLaunchKernelGGL((k_attn_fwd<HD, true, ATT_NW>), dim3(heads * nqb), dim3(64 * ATT_NW), 0, st, w.Qp, w.Kp, w.Vt,
                       ATT_KT * T, n_pad, heads, o, o_ld, sp);
    return hipGetLastError();
}

}  // namespace

extern "C" int fh3k_vsa_max_tiles(void) { return 4096; }

extern "C" size_t fh3k_vsa_ws_bytes(int T, int heads, int hd) { return vsa_ws(nullptr, T, heads, hd).bytes; }

extern "C" hipError_t fh3k_vsa_attention(const float *q, const float *k, const float *v, int64_t ld, int64_t ldv,
                                         const float *qn_w, const float *kn_w, float eps, const float *cosb,
                                         const float *sinb, int rot, const float *gate, float *o, int64_t o_ld,
                                         int heads, int hd, const float *inv, const int *gather, const int *cnt,
                                         int T, int P, int kv, int all, float scale, void *ws, hipStream_t st) {
    if (T <= 0 || T > fh3k_vsa_max_tiles()) return hipErrorInvalidValue;
    if (hd == 128)
        return vsa_launch<128>(q, k, v, ld, ldv, qn_w, kn_w, eps, cosb, sinb, rot, gate, o, o_ld, heads, inv, gather,
                               cnt, T, P, kv, all, scale, ws, st);
    if (hd == 64)
        return vsa_launch<64>(q, k, v, ld, ldv, qn_w, kn_w, eps, cosb, sinb, rot, gate, o, o_ld, heads, inv, gather,
                              cnt, T, P, kv, all, scale, ws, st);
    return hipErrorInvalidValue;
}
