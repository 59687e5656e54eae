// Causal GQA attention of a few query rows over a long context on the fp32
// MFMA (reference attention_batch, src/tensor.rs:1099-1139, used by
// forward_seq, src/model.rs:555-566): pieces of under kTiledMinTokens tokens,
// where the per-row kernel reads the whole context once per query row.  The
// products stay exact f32 products, as in that kernel, and K and V are read
// from the f32 cache as they are.
//
// A workgroup owns 32 query columns -- 32 / GROUP consecutive positions of
// the GROUP query heads that share KV head g -- and a run of 64-key blocks;
// wavefront w takes keys 16 w .. +15 of each block, straight from memory into
// MFMA operands (no other wavefront needs them), with an online softmax of
// its own.  The wavefronts are merged through LDS at the end, and the runs by
// attn_f32_combine_kernel.
//
// v_mfma_f32_16x16x4_f32: lane l supplies A row l & 15 and B column l & 15 at
// k = l >> 4 and receives D rows 4 (l >> 4) .. +3 of column l & 15.  Any k
// order serves as long as both operands agree:
// - scores S^T = K Q^T: lane (r, q) holds dims 16 c + 4 q .. +3 of key r and
//   of column r; MFMA j of chunk c takes the j-th of them;
// - O^T += V^T P^T: the lane's scores are keys 4 q + i of column r, so MFMA i
//   takes key 4 q + i; the lane loads dims 64 h + 4 r .. +3 of that key, and
//   row tile (h, e) is made of the dims 64 h + 4 r + e, so that D gives lane
//   (r, q) dims 64 h + 16 q + 4 i' + e of column r.
//
// Bound by the fp32 matrix rate and the cache's reads from L2 (once per 32
// columns).
#include <algorithm>

#include "common.cuh"
#include "kernels.hpp"

namespace tmg {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kFHD = 128;   // head dim
constexpr int kFCols = 32;  // query columns per workgroup, two MFMA column tiles
constexpr int kFKB = 64;    // keys per block, 16 per wavefront

// Workgroup (tile * nsp + sp) * nkv + g: run sp of column tile `tile`.
template <int GROUP>
__global__ __launch_bounds__(kBlock, 2) void attn_f32_kernel(const AttnArgs a, int nsp) {
    __shared__ __attribute__((aligned(16))) f32x4 s_o[4][2][8][64];
    __shared__ float2 s_ml[4][kFCols];
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const int r = lane & 15, q4 = lane >> 4;
    const int g = (int)blockIdx.x % a.nkv, rest = (int)blockIdx.x / a.nkv;
    const int sp = rest % nsp, tile = rest / nsp;
    const int kvd = a.nkv * kFHD, qd = a.nq * kFHD;
    const int first = tile * (kFCols / GROUP);                        // the tile's first query row
    const int last_row = min(a.T, first + kFCols / GROUP) - 1;        // and its last
    const int first_pos = a.start + first, last_pos = a.start + last_row;
    const int nb = last_pos / kFKB + 1;
    const int b0 = sp * nb / nsp, b1 = (sp + 1) * nb / nsp;

    int qpos[2];
    f32x4 q[2][8];
#pragma unroll
    for (int ct = 0; ct < 2; ct++) {
        const int c = ct * 16 + r, ti = min(first + c / GROUP, last_row);
        qpos[ct] = a.start + ti;
        // scores come out in log2 units
        const float sl2 = a.scale * 1.4426950408889634f;
        const float *src = a.q + (size_t)ti * qd + (g * GROUP + c % GROUP) * kFHD + 4 * q4;
#pragma unroll
        for (int d = 0; d < 8; d++) q[ct][d] = *reinterpret_cast<const f32x4 *>(src + 16 * d) * sl2;
    }
    float m[2] = {-INFINITY, -INFINITY}, l[2] = {0.f, 0.f};
    f32x4 o[2][8];
#pragma unroll
    for (int ct = 0; ct < 2; ct++)
#pragma unroll
        for (int d = 0; d < 8; d++) o[ct][d] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int b = b0; b < b1; b++) {
        const int k0 = b * kFKB + wave * 16;
        if (k0 > last_pos) break;
        // rows past the tile's last position repeat it (their scores are masked)
        const float *ksrc = a.k_cache + (size_t)min(k0 + r, last_pos) * kvd + g * kFHD + 4 * q4;
        f32x4 k[8], v[4][2];
#pragma unroll
        for (int d = 0; d < 8; d++) k[d] = *reinterpret_cast<const f32x4 *>(ksrc + 16 * d);
        f32x4 s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int d = 0; d < 8; d++)
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int ct = 0; ct < 2; ct++)
                    s[ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[d][j], q[ct][d][j], s[ct], 0, 0, 0);
        // V after the scores: both in flight at once spill registers
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float *vsrc = a.v_cache + (size_t)min(k0 + 4 * q4 + i, last_pos) * kvd + g * kFHD + 4 * r;
            v[i][0] = *reinterpret_cast<const f32x4 *>(vsrc);
            v[i][1] = *reinterpret_cast<const f32x4 *>(vsrc + 64);
        }
        const bool diag = k0 + 15 > first_pos;
#pragma unroll
        for (int ct = 0; ct < 2; ct++) {
            if (diag) {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (k0 + 4 * q4 + i > qpos[ct]) s[ct][i] = -INFINITY;
            }
            const float mx = max_xor16_32(fmaxf(fmaxf(s[ct][0], s[ct][1]), fmaxf(s[ct][2], s[ct][3])));
            // the maximum is raised in steps of at least 2^8 (see attn_prefill_kernel)
            const bool raise = mx > m[ct] + 8.0f;
            if (__builtin_amdgcn_ballot_w64(raise)) {
                const float corr = raise ? __builtin_amdgcn_exp2f(m[ct] - mx) : 1.0f;
                m[ct] = raise ? mx : m[ct];
                l[ct] *= corr;
#pragma unroll
                for (int d = 0; d < 8; d++) o[ct][d] *= corr;
            }
            const float ref = m[ct] == -INFINITY ? 0.0f : m[ct];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                s[ct][i] = __builtin_amdgcn_exp2f(s[ct][i] - ref);
                l[ct] += s[ct][i];
            }
        }
        // a masked key has weight zero, but zero times an infinite or NaN
        // value of a later row would not be: such a block goes key by key
        bool odd = false;
        if (diag) {
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int h = 0; h < 2; h++)
#pragma unroll
                    for (int e = 0; e < 4; e++) odd = odd || !(fabsf(v[i][h][e]) < INFINITY);
        }
        if (__builtin_amdgcn_ballot_w64(odd)) {
#pragma unroll 1
            for (int key = 0; key < 16 && k0 + key <= last_pos; key++) {
                const float *vrow = a.v_cache + (size_t)(k0 + key) * kvd + g * kFHD + 16 * q4;
#pragma unroll
                for (int ct = 0; ct < 2; ct++) {
                    float p = 0.0f;
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const float x = __shfl(s[ct][i], (key >> 2) * 16 + r);
                        p = (key & 3) == i ? x : p;
                    }
                    if (k0 + key > qpos[ct]) continue;
#pragma unroll
                    for (int h = 0; h < 2; h++)
#pragma unroll
                        for (int e = 0; e < 4; e++)
#pragma unroll
                            for (int i = 0; i < 4; i++) o[ct][h * 4 + e][i] += p * vrow[64 * h + 4 * i + e];
                }
            }
            continue;
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int ct = 0; ct < 2; ct++)
                        o[ct][h * 4 + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[i][h][e], s[ct][i], o[ct][h * 4 + e], 0, 0, 0);
    }
    // merge the wavefronts: thread (ct, h, lane) owns dims 64 h + 16 q .. +15
    // of column (ct, r)
#pragma unroll
    for (int ct = 0; ct < 2; ct++) {
        const float L = add_xor32(add_xor16(l[ct]));
        if (q4 == 0) s_ml[wave][ct * 16 + r] = make_float2(m[ct], L);
#pragma unroll
        for (int d = 0; d < 8; d++) s_o[wave][ct][d][lane] = o[ct][d];
    }
    __syncthreads();
    const int ct = wave & 1, h = wave >> 1, c = ct * 16 + r;
    float M = -INFINITY, L = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; w++) M = fmaxf(M, s_ml[w][c].x);
    f32x4 out[4];  // out[i][e]: dim 4 i + e of the thread's 16
#pragma unroll
    for (int i = 0; i < 4; i++) out[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; w++) {
        const float2 ml = s_ml[w][c];
        const float f = ml.x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ml.x - M);
        L += ml.y * f;
        if (f == 0.0f && ml.y == 0.0f) continue;  // no key of this wavefront's is visible
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const f32x4 x = s_o[w][ct][h * 4 + e][lane];
#pragma unroll
            for (int i = 0; i < 4; i++) out[i][e] += x[i] * f;
        }
    }
    if (nsp > 1) {
        f32x4 *part = reinterpret_cast<f32x4 *>(a.part) + (size_t)blockIdx.x * 1024 + t;
#pragma unroll
        for (int i = 0; i < 4; i++) part[i * kBlock] = out[i];
        if (h == 0 && q4 == 0) *reinterpret_cast<float2 *>(a.part_ml + ((size_t)blockIdx.x * kFCols + c) * 2) = make_float2(M, L);
        return;
    }
    const int ti = first + c / GROUP;
    if (ti >= a.T) return;
    const float inv = 1.0f / L;
    const size_t ob = (size_t)ti * qd + (g * GROUP + c % GROUP) * kFHD + 64 * h + 16 * q4;
#pragma unroll
    for (int i = 0; i < 4; i++) store_split4(out[i] * inv, a.out_hi + ob + 4 * i, a.out_lo + ob + 4 * i);
}

// Merges the runs of a column tile in key order: workgroup (tile * 4 + i) *
// nkv + g takes quad i of every thread's 16 dims.
template <int GROUP>
__global__ __launch_bounds__(kBlock) void attn_f32_combine_kernel(const AttnArgs a, int nsp) {
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const int g = (int)blockIdx.x % a.nkv, rest = (int)blockIdx.x / a.nkv;
    const int i = rest & 3, tile = rest >> 2;
    const int c = (wave & 1) * 16 + (lane & 15), h = wave >> 1, q4 = lane >> 4;
    const int ti = tile * (kFCols / GROUP) + c / GROUP;
    float M = -INFINITY, L = 0.0f;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    constexpr int NC = 8;  // runs in flight
#pragma unroll 1
    for (int s = 0; s < nsp; s += NC) {
        float2 ml[NC];
        f32x4 v[NC];
#pragma unroll
        for (int x = 0; x < NC; x++)
            if (s + x < nsp) {
                const size_t wg = ((size_t)tile * nsp + s + x) * a.nkv + g;
                ml[x] = *reinterpret_cast<const float2 *>(a.part_ml + (wg * kFCols + c) * 2);
                v[x] = reinterpret_cast<const f32x4 *>(a.part)[wg * 1024 + i * kBlock + t];
            }
#pragma unroll
        for (int x = 0; x < NC; x++)
            // a run without a visible key adds nothing; one whose scores are all
            // NaN has no maximum either, but a NaN sum, which has to go through
            if (s + x < nsp && !(ml[x].x == -INFINITY && ml[x].y == 0.0f)) {
                const float nm = fmaxf(M, ml[x].x);
                const float f0 = __builtin_amdgcn_exp2f(M - nm), f1 = __builtin_amdgcn_exp2f(ml[x].x - nm);
                M = nm;
                L = L * f0 + ml[x].y * f1;
                o = o * f0 + v[x] * f1;
            }
    }
    if (ti >= a.T) return;
    const size_t ob = (size_t)ti * (a.nq * kFHD) + (g * GROUP + c % GROUP) * kFHD + 64 * h + 16 * q4 + 4 * i;
    store_split4(o * (1.0f / L), a.out_hi + ob, a.out_lo + ob);
}

// Runs per column tile: two workgroups per CU, a run at least one block.
int f32_runs(const AttnArgs &a) {
    const int wgs = (a.T + kFCols / (a.nq / a.nkv) - 1) / (kFCols / (a.nq / a.nkv)) * a.nkv;
    if (!a.part || !a.part_ml) return 1;
    return std::max(1, std::min(std::min(kAttnF32Runs / wgs, (a.start + a.T + kFKB - 1) / kFKB), 64));
}

template <int GROUP>
void launch_group(const AttnArgs &a, hipStream_t s) {
    const int nsp = f32_runs(a), tiles = (a.T + kFCols / GROUP - 1) / (kFCols / GROUP);
    hipLaunchKernelGGL(attn_f32_kernel<GROUP>, dim3(tiles * nsp * a.nkv), dim3(kBlock), 0, s, a, nsp);
    if (nsp > 1)
        hipLaunchKernelGGL(attn_f32_combine_kernel<GROUP>, dim3(tiles * 4 * a.nkv), dim3(kBlock), 0, s, a, nsp);
}

}  // namespace

bool attn_f32_pays(const AttnArgs &a) {
    const int group = a.nkv > 0 ? a.nq / a.nkv : 0;
    if (a.hd != kFHD || !a.out_hi || !a.out_lo || a.pos_seq || a.nq != group * a.nkv ||
        !(group == 1 || group == 2 || group == 4 || group == 8))
        return false;
    // The per-row kernel: 1.66 us per 64 positions of one round of workgroups,
    // 200 such chunks per us (300 with one query head per KV head) once the chip
    // is full, each row those up to its own position (with the last row's count
    // for all, this kernel was taken where it was slower: the 1B shape at 145-180
    // tokens by 2% of the prefill, one query head per KV head by 8-10%).  With
    // four or more query heads its chunks are 16 positions and slower, and the
    // last row's count stands for that.  This one: 2.6 us per block of a run, 2 us
    // per block and 256 workgroups once it is full, 11 us for the launch, first
    // loads and merge, 6 us for merging runs.
    const double chunks = (a.start + a.T + 63) / 64;
    // chunks of rows 0 .. n - 1
    auto below = [](int64_t n) { return 32 * (n / 64) * (n / 64 - 1) + n / 64 * (n % 64) + n; };
    const double all = group < 4 ? (double)(below(a.start + a.T) - below(a.start)) : a.T * chunks;
    const double rows_us = 3.0 + std::max(1.66 * chunks, all * a.nkv / (group == 1 ? 300.0 : 200.0));
    const int nsp = f32_runs(a), tiles = (a.T + kFCols / group - 1) / (kFCols / group);
    const double run = std::max(1.0, chunks / nsp), wgs = (double)tiles * nsp * a.nkv;
    return 11.0 + std::max(2.6 * run, 2.0 * run * wgs / 256.0) + (nsp > 1 ? 6.0 : 0.0) < rows_us;
}

LaunchPlan attn_f32_plan(const AttnArgs &a) {
    const int cols = kFCols / (a.nq / a.nkv), tiles = (a.T + cols - 1) / cols * a.nkv;
    return LaunchPlan{kAttnF32, tiles, tiles * f32_runs(a)};
}

hipError_t launch_attn_f32(const AttnArgs &a, hipStream_t s) {
    if (a.T <= 0 || a.hd != kFHD || !a.out_hi || !a.out_lo || a.pos_seq) return hipErrorInvalidValue;
    switch (a.nq / a.nkv) {
        case 1: launch_group<1>(a, s); break;
        case 2: launch_group<2>(a, s); break;
        case 4: launch_group<4>(a, s); break;
        case 8: launch_group<8>(a, s); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace tmg
